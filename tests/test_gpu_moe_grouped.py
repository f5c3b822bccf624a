"""The expert products over assignments sorted on the device (csrc/moe_grouped.hip): the sort against torch's stable one, the two
products and their activations against float64, at edges of the 128-row tiles, 64-deep slices and 128-column tiles."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _assign(n, top, experts, kind, g):
    if kind == "one":       # every token to the same experts: all others are empty
        return torch.arange(top).repeat(n, 1).add(experts - top)
    if kind == "runs":      # counts of exactly one tile, one more, one less
        flat = torch.repeat_interleave(torch.arange(experts), torch.tensor(([128, 129, 127] * experts)[:experts]))
        flat = torch.cat((flat, torch.zeros(max(0, n * top - flat.numel()), dtype=torch.long)))[:n * top]
        return flat[torch.randperm(n * top, generator=g)].view(n, top)
    return torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(n)])


@pytest.mark.parametrize("n,top,experts,kind", [(1, 1, 1, "any"), (700, 2, 5, "any"), (4099, 3, 70, "any"), (64, 2, 8, "one"),
                                                (256, 3, 6, "runs")])
def test_sort_by_expert(n, top, experts, kind):
    from swiftllm_amd import _hip
    idx = _assign(n, top, experts, kind, torch.Generator().manual_seed(n)).to(torch.int32).cuda()
    order, where = torch.empty(n * top, dtype=torch.int32, device="cuda"), torch.empty(n * top, dtype=torch.int64, device="cuda")
    offsets = torch.empty(experts + 1, dtype=torch.int32, device="cuda")
    _hip.call("swl_moe_sort", _hip.ptr(order), _hip.ptr(where), _hip.ptr(offsets), _hip.ptr(idx), n * top, experts, _hip.stream())
    flat = idx.reshape(-1).long().cpu()
    want = torch.argsort(flat, stable=True)
    assert torch.equal(order.long().cpu(), want)
    assert torch.equal(where.cpu()[want], torch.arange(n * top))
    assert torch.equal(offsets.long().cpu(), torch.cat((torch.zeros(1, dtype=torch.long), torch.bincount(flat, minlength=experts).cumsum(0))))


@pytest.mark.parametrize("shift", [0, 1])       # ids on and off the 16-byte boundaries
@pytest.mark.parametrize("n,experts", [(3, 2), (4095, 9), (4096, 9), (4097, 9), (16384, 3), (16387, 3), (40001, 130)])
def test_sort_at_the_ends_of_pieces(n, experts, shift):
    """4096 ids in one piece of four a thread, pieces of 16384 beyond; ids that name no expert count as the nearest."""
    from swiftllm_amd import _hip
    ids = torch.randint(-1, experts + 1, (n + shift,), generator=torch.Generator().manual_seed(n)).to(torch.int32)
    idx, flat = ids.cuda()[shift:], ids[shift:].long().clamp(0, experts - 1)
    order, where = torch.full((n,), -1, dtype=torch.int32, device="cuda"), torch.full((n,), -1, dtype=torch.int64, device="cuda")
    offsets = torch.empty(experts + 1, dtype=torch.int32, device="cuda")
    _hip.call("swl_moe_sort", _hip.ptr(order), _hip.ptr(where), _hip.ptr(offsets), _hip.ptr(idx), n, experts, _hip.stream())
    want = torch.argsort(flat, stable=True)
    assert torch.equal(order.long().cpu(), want) and torch.equal(where.cpu()[want], torch.arange(n))
    assert torch.equal(offsets.long().cpu(), torch.cat((torch.zeros(1, dtype=torch.long), torch.bincount(flat, minlength=experts).cumsum(0))))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,top,experts,width,ff,kind,form", [
    (300, 2, 5, 128, 64, "any", "silu"), (129, 1, 3, 64, 72 * 8, "any", "clamped"), (256, 3, 6, 192, 128, "runs", "silu_in"),
    (200, 2, 8, 256, 192, "one", "relu2"), (77, 4, 70, 64, 64, "any", "relu2"), (1000, 2, 8, 1024, 320, "any", "silu"),
    (90, 2, 4, 72, 64, "any", "silu"), (90, 2, 4, 64, 100, "any", "relu2")])      # (the last two: sizes that stay with the library)
def test_sorted_experts(n, top, experts, width, ff, kind, form, dtype):
    from swiftllm_amd.worker.kernels import moe
    g = torch.Generator().manual_seed(n)
    h = torch.randn(n, width, generator=g).to(dtype)
    up = (torch.randn(experts, ff * (1 if form == "relu2" else 2), width, generator=g) / width ** 0.5).to(dtype)
    down = (torch.randn(experts, width, ff, generator=g) / ff ** 0.5).to(dtype)
    idx, wts = _assign(n, top, experts, kind, g), torch.rand(n, top, generator=g) + 0.1
    served = width % 64 == 0 and ff % 64 == 0
    assert moe._sorted_served(h.cuda(), up.cuda(), down.cuda(), ff) == served
    args = (h.cuda(), idx.to(torch.int32).cuda(), wts.cuda(), up.cuda(), down.cuda())
    if form == "relu2":
        got = moe.moe_experts_relu2(*args)
    else:
        got = moe.moe_experts(*args, 1.5, moe.ACT_CLAMPED if form == "clamped" else moe.ACT_SILU, weigh_inputs=form == "silu_in")
    want, size = torch.zeros(n, width, dtype=torch.float64), torch.zeros(n, width, dtype=torch.float64)
    for j in range(top):
        z = torch.einsum("tk,tfk->tf", h.double() * (wts[:, j:j + 1] if form == "silu_in" else 1.0), up.double()[idx[:, j]])
        if form == "relu2":
            y = torch.relu(z) ** 2
        else:
            a, u = z[:, :ff], z[:, ff:]
            if form == "clamped":
                a, u = a.clamp(max=1.5), u.clamp(-1.5, 1.5)
                y = a * torch.sigmoid(1.702 * a) * (u + 1)
            else:
                y = a * torch.sigmoid(a) * u
        w = 1.0 if form == "silu_in" else wts[:, j:j + 1].double()
        want += w * torch.einsum("tf,twf->tw", y, down.double()[idx[:, j]])
        size += w * (torch.einsum("tf,twf->tw", y ** 2, down.double()[idx[:, j]] ** 2).sqrt() + 1.0)
    # one rounding of the activations, which enter a sum of ff terms with random signs (4 of its standard deviations; the library form
    # rounds the first products too), and one of each result: 2^-9 relative in bf16, 2^-12 in fp16
    eps = 2.0 ** (-9 if dtype == torch.bfloat16 else -12)
    assert ((got.double().cpu() - want).abs() <= 8 * eps * (size + want.abs())).all()


@pytest.mark.parametrize("form", ["silu", "silu_in", "relu2"])
def test_assignments_of_other_strides(form):
    """Ids and weights stored choice by choice (columns of the [tokens, choices] view are contiguous) give what contiguous ones give."""
    from swiftllm_amd.worker.kernels import moe
    g = torch.Generator().manual_seed(3)
    n, top, experts, width, ff = 150, 2, 5, 128, 64
    h, down = torch.randn(n, width, generator=g).bfloat16().cuda(), (torch.randn(experts, width, ff, generator=g) / 8).bfloat16().cuda()
    up = (torch.randn(experts, ff * (1 if form == "relu2" else 2), width, generator=g) / 11).bfloat16().cuda()
    idx, wts = _assign(n, top, experts, "any", g).int().cuda(), (torch.rand(n, top, generator=g) + 0.1).cuda()
    assert moe._sorted_served(h, up, down, ff)

    def run(i, w):
        if form == "relu2":
            return moe.moe_experts_relu2(h, i, w, up, down)
        return moe.moe_experts(h, i, w, up, down, 0.0, moe.ACT_SILU, weigh_inputs=form == "silu_in")
    assert torch.equal(run(idx, wts), run(idx.t().contiguous().t(), wts.t().contiguous().t()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("n,top,experts,K,N,kind", [
    (1500, 2, 8, 64, 4096 + 8, "any"),          # one slice, a last column tile of 8
    (900, 2, 70, 128, 1600, "any"),             # more experts than lanes, tiles of a few rows, two slices
    (640, 1, 5, 192, 16384, "runs"),            # tiles filled to the row, one over, one short
    (300, 2, 3, 320, 16384, "one")])            # an empty expert
def test_many_tiles(n, top, experts, K, N, kind, mode, dtype):
    """More tiles than two a CU take the form with one staged slice: the bits of launches over parts of the columns, which stay below."""
    from swiftllm_amd import _hip
    g = torch.Generator().manual_seed(K)
    total = n * top
    idx = _assign(n, top, experts, kind, g).to(torch.int32).cuda()
    order, where = torch.empty(total, dtype=torch.int32, device="cuda"), torch.empty(total, dtype=torch.int64, device="cuda")
    offsets = torch.empty(experts + 1, dtype=torch.int32, device="cuda")
    _hip.call("swl_moe_sort", _hip.ptr(order), _hip.ptr(where), _hip.ptr(offsets), _hip.ptr(idx), total, experts, _hip.stream())
    x = torch.randn(n, K, generator=g).to(dtype).cuda()
    w = (torch.randn(experts, 2 if mode == 1 else 1, N, K, generator=g) / K ** 0.5).to(dtype).cuda()
    in_w = (torch.rand(total, generator=g) + 0.5).cuda() if mode == 1 else None

    def product(w):
        cols = w.shape[2]
        out = torch.zeros(total, cols, dtype=dtype, device="cuda")
        _hip.call("swl_moe_gemm", _hip.ptr(out), _hip.ptr(x), _hip.ptr(w), _hip.ptr(order), _hip.ptr(offsets), _hip.ptr(in_w), total, n,
                  top, experts, K, cols, mode, 0, 1.5, _hip.dtype_code(dtype), _hip.stream())
        return out
    row_tiles, width = (total + 64 * experts) // 128, 64 if mode == 1 else 128
    part = width * (512 // row_tiles)
    assert row_tiles * -(-N // width) > 512 and part > 0
    got = product(w)
    assert torch.equal(got, torch.cat([product(w[:, :, c:c + part].contiguous()) for c in range(0, N, part)], 1))
    assert got.abs().amax(1).min() > 0
