"""The gated units of the tiled products (csrc/gemm_tile.h: dense and of experts) where their arguments are anything: rows of x with a single one pick
single weights, so that every product is known exactly. Gates far below zero, the last ones with a result, infinities, NaN."""
import pytest
import torch

pytestmark = pytest.mark.gpu
K, N = 256, 2048
DTYPES = [torch.bfloat16, torch.float16]
ACTS = [0, 1, 2, 3]      # kernels/moe.py's units, TILE_SILU_ROUNDED of kernels/linear.py


def picked(gate, up, act, dtype, m=K):
    """Weights [2 N, K] whose product with row k of one-hot x is (gate[k], up[k]), in the unit's order of halves, and x."""
    first, second = (up, gate) if act >= 2 else (gate, up)
    x = torch.zeros((m, K), dtype=dtype, device="cuda")
    x[torch.arange(m), torch.arange(m) % K] = 1
    return x, torch.cat([first.T, second.T]).to(dtype).contiguous()


def unit64(g, u, act, dtype, limit):
    g, u = g.double(), u.double()
    if act == 0:
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        return g / (1 + torch.exp(-1.702 * g)) * (u + 1)
    s = g / (1 + torch.exp(-g))
    return (s.to(dtype).double() if act == 3 else s) * u


def dense(x, w, act, limit, extra=1):
    """More than 256 rows, the tiled kernel's launch."""
    from swiftllm_amd.worker.kernels.linear import TILE_GATED, linear_tile
    y = linear_tile(torch.cat([x, x[:extra]]), w, TILE_GATED + act, limit=limit)
    assert y is not None
    return y[:x.shape[0]]


def experts(x, w, act, limit):
    """All rows by the second of two experts, in order."""
    from swiftllm_amd import _hip
    m = x.shape[0]
    ww = torch.stack([torch.ones_like(w), w])
    order = torch.arange(m, dtype=torch.int32, device="cuda")
    offsets = torch.tensor([0, 0, m], dtype=torch.int32, device="cuda")
    out = torch.empty((m, w.shape[0] // 2), dtype=x.dtype, device="cuda")
    _hip.call("swl_moe_gemm", _hip.ptr(out), _hip.ptr(x), _hip.ptr(ww), _hip.ptr(order), _hip.ptr(offsets), 0, m, m, 1, 2, K, w.shape[0] // 2, 1, act, float(limit),
              _hip.dtype_code(x.dtype), _hip.stream())
    return out


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("act", ACTS)
@pytest.mark.parametrize("lo,hi", [(-88.5, -87.4), (-87, -20), (-20, -10), (-10, 10), (10, 80)])
def test_as_exact_as_the_units_of_decoded_tokens(lo, hi, act, dtype):
    """Results are the float64 unit's, rounded, but where that lies within the fp32 error of the middle between two numbers. The error is at most four units
    of 2^-24 for silu (an exponential, a sum, a quotient) and one of the product; -1.702 z is rounded: as many units more as it is
    large, and two for the product with z and the sum behind it. A number's
    neighbours are 2^-8 (2^-11) of it apart or more, so at most 2 e 2^8 (2^11) of the results are another number, and those are neighbours."""
    g = torch.Generator(device="cuda").manual_seed(int(1000 - lo) + act)
    # (results that are normal numbers: of float16 too, by large factors behind the unit; its argument is 1.702 z where act is 0)
    if dtype == torch.float16 and hi < -9 and (act == 3 or hi < -15):
        pytest.skip("zero in float16")
    scale = 1e4 if dtype == torch.float16 and hi < -9 else 1.0
    gate = ((torch.rand((K, N), generator=g, device="cuda") * (hi - lo) + lo) / (1.702 if act == 0 else 1.0)).to(dtype)
    up = ((torch.rand((K, N), generator=g, device="cuda") + 0.5) * scale).to(dtype)
    limit = 6e4
    want = unit64(gate, up, act, dtype, limit)
    exact = want.to(dtype)
    units = 5 + (2 + max(-lo, hi) if act == 0 else 0)
    share = 2 * units * 2.0 ** -24 * (2 ** 11 if dtype == torch.float16 else 2 ** 8) * (2 if act == 3 else 1)
    x, w = picked(gate, up, act, dtype)
    for name, run in (("dense", dense), ("experts", experts)):
        if name == "experts" and act > 1:
            continue
        y = run(x, w, act, limit)
        other = y != exact
        assert float(other.double().mean()) <= share + 4 / other.numel(), (name, float(other.double().mean()), share)
        ulp = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7
        floor = 2.0 ** -24 if dtype == torch.float16 else 2.0 ** -126 * ulp
        # (act 3: a neighbour of the rounded silu, times up, rounded again)
        assert bool(((y.double() - exact.double()).abs() <= (2 if act == 3 else 1) * ulp * exact.double().abs() + floor).all()), name


def same(y, want):
    """Equal or neighbours (both units have errors of their own), NaN where NaN is."""
    ulp = 2.0 ** -10 if y.dtype == torch.float16 else 2.0 ** -7
    a, b = y.double(), want.double()
    assert torch.equal(a.isnan(), b.isnan())
    assert bool((a.isnan() | (a == b) | ((a - b).abs() <= ulp * b.abs())).all())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("act", ACTS)
def test_what_the_units_make_of_infinities_and_nan(act, dtype):
    """The same as of the product and the unit in a launch of its own (swl_glu_clamp, swl_silu_mul): rows doubled beyond the largest number, rows of NaN."""
    from swiftllm_amd.worker.kernels.moe import gated_unit
    from swiftllm_amd.worker.kernels.silu_and_mul import silu_and_mul_inplace
    big = 60000.0 if dtype == torch.float16 else 3e38
    values = torch.tensor([big, -big, 0.0, 1.0, -1.0, 20.0, -20.0, -88.0, -89.0, -104.0, 300.0, -300.0, 1e-30, 6e-5, 0.5, -0.5], device="cuda")
    at = torch.arange(N, device="cuda")
    gate, up = values[at % 16].expand(K, N), values[at // 16 % 16].expand(K, N)
    x, w = picked(gate, up, act, dtype)
    x[1::3] *= 2
    x[2::3] *= float("nan")
    y = dense(x, w, act, 7.0, extra=3)
    z = torch.nn.functional.linear(x, w)        # (products that are exact, or infinite, or NaN)
    if act == 3:
        silu_and_mul_inplace(z)
        want = z[:, :N]
    else:
        want = gated_unit(z, N, act, 7.0)
    same(y, want)
    if act <= 1:
        want = gated_unit((x.float().nan_to_num(0.0) @ w.float().T).masked_fill(x.isnan().any(1, keepdim=True), float("nan")), N, act, 7.0).to(dtype)
        same(experts(x, w, act, 7.0), want)
