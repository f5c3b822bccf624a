"""Slabs of 65 to 256 decoded tokens from the tiled kernel (kernels/linear.py, _mid_tile): against float32, the same rows in every step of a bucket, and
what stays with the other kernels."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(6144, 4096), (4096, 4096), (4096, 14336), (2048, 8192)])
@pytest.mark.parametrize("m", [65, 96, 97, 128, 129, 160, 161, 224, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_slabs(n, k, m, dtype):
    from swiftllm_amd.worker.kernels.linear import SplitKPartials, _mid_tile, linear_splitk
    g = torch.Generator(device="cuda").manual_seed(m + k)
    a, w = torch.randn(256, k, generator=g, device="cuda").to(dtype), torch.randn(n, k, generator=g, device="cuda").to(dtype)
    tile = _mid_tile(a[:m], w)
    assert (tile is None) == (k >= 2 * n and m > 160)
    if tile is None:
        return
    y = linear_splitk(a[:m], w)
    assert isinstance(y, SplitKPartials) and y.k_splits == tile[1] and y.shape == (m, n)
    slabs = y.slabs[:y.k_splits * m * n].view(y.k_splits, m, n)
    want = a[:m].double() @ w.double().t()
    # fp32 sums of k products: k roundings by 2^-24 at most of partial sums of 4 sqrt(k) at most, as likely up as down: sqrt(k) 4 sqrt(k) 2^-24 3^-0.5
    # and six times that for the largest of a million (0.014 at 14336; a product that is left out is about 1)
    assert (slabs.double().sum(0) - want).abs().max() < 14 * k * 2.0 ** -24
    again = linear_splitk(a[:-(-m // 32) * 32], w)
    full = again.slabs[:again.k_splits * again.shape[0] * n].view(again.k_splits, again.shape[0], n)[:, :m].clone()
    y = linear_splitk(a[:m], w)
    assert again.k_splits == y.k_splits and torch.equal(full, y.slabs[:y.k_splits * m * n].view(y.k_splits, m, n))


@pytest.mark.parametrize("n,k,first", [(5120, 5120, False), (2048, 8192, True), (1024, 16384, False), (4096, 5120, True), (8192, 8192, None)])
def test_the_measured_kernel_stays_where_it_is_faster(n, k, first, monkeypatch):
    """first: ahead of what was measured at load (False: only where the library serves the class, None: never)."""
    from swiftllm_amd.worker.kernels import route_tune
    from swiftllm_amd.worker.kernels.linear import _mid_tile
    a, w = torch.zeros(120, k, dtype=torch.float16, device="cuda"), torch.zeros(n, k, dtype=torch.float16, device="cuda")
    w._swl_packed = w
    for wide in (False, True):
        monkeypatch.setitem(route_tune._table, route_tune._key(n, k, torch.float16, 128, False), wide)
        assert (_mid_tile(a, w) is not None) == (False if first is None else first or not wide)


def test_others_stay():
    from swiftllm_amd.worker.kernels.linear import _mid_tile
    new = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device="cuda")      # noqa: E731
    for a, w in ((new(100, 4096), new(28672, 4096)), (new(100, 2048), new(4096, 2048)), (new(100, 4096), new(4096, 4096).t()), (new(100, 4100)[:, :4096], new(4096, 4096)),
                 (new(100, 4097)[:, 1:], new(4096, 4096)), (new(100, 5504), new(4096, 5504))):
        assert _mid_tile(a, w) is None
