"""Gated norms over heads and over groups (csrc/delta_rule.hip, csrc/ssd.hip) against float64: rows in registers, at the edges of what a thread,
a wave and a workgroup hold, and rows that lie on no 16 bytes, which the column-by-column kernels serve."""
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}     # half a unit in the last place of a result below 1


def rows(n, c, shift, dtype, g):
    wide = torch.randn(n, c + 16, generator=g).to(dtype)
    return wide[:, shift:shift + c], wide.cuda()[:, shift:shift + c]


@pytest.mark.parametrize("n,H,dv,per_head,shift", [(1, 1, 32, False, 0), (3, 5, 64, True, 8), (257, 3, 128, True, 0), (33, 2, 128, False, 8), (5, 3, 128, True, 1),
                                                   (7, 2, 24, False, 0), (4, 1, 256, False, 0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_heads(n, H, dv, per_head, shift, dtype):
    from swiftllm_amd.worker.kernels.delta_rule import gated_head_rmsnorm
    g = torch.Generator().manual_seed(n + dv)
    o, w = torch.randn(n, H * dv, generator=g), torch.randn(H * dv if per_head else dv, generator=g)
    gate, gate_dev = rows(n, H * dv, shift, dtype, g)
    _, out = rows(n, H * dv, shift, dtype, g)
    gated_head_rmsnorm(out, o.cuda(), gate_dev, w.cuda(), H, dv, 1e-6, 0.7)
    x, z = o.double().view(n, H, dv), gate.double().reshape(n, H, dv)
    want = (0.7 * x / (x.pow(2).mean(-1, keepdim=True) + 1e-6).sqrt() * w.double().view(-1, dv) * (z * z.sigmoid())).reshape(n, -1)
    # a rounding of the result, and 16 of fp32 on the way
    assert ((out.cpu().double() - want).abs() <= want.abs() * (2 * EPS[dtype] + 16 * EPS[torch.float32]) + 1e-7).all()


@pytest.mark.parametrize("n,cols,groups,shift", [(1, 8, 1, 0), (3, 520, 1, 8), (9, 1024, 2, 0), (5, 2048, 1, 0), (4, 2056, 1, 8), (3, 4104, 1, 0), (2, 8192, 1, 0), (2, 8200, 1, 0),
                                                 (5, 1024, 1, 1), (6, 60, 3, 0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_groups(n, cols, groups, shift, dtype):
    from swiftllm_amd import _hip
    g = torch.Generator().manual_seed(n + cols)
    y, w = torch.randn(n, cols, generator=g), torch.randn(cols, generator=g)
    gate, gate_dev = rows(n, cols, shift, dtype, g)
    _, out = rows(n, cols, shift, dtype, g)
    y_dev, w_dev = y.cuda(), w.cuda()
    _hip.call("swl_gated_group_rmsnorm", _hip.ptr(out), out.stride(0), _hip.ptr(y_dev), _hip.ptr(gate_dev), gate_dev.stride(0), _hip.ptr(w_dev), 1e-6, n, cols, groups,
              _hip.dtype_code3(dtype), _hip.stream())
    z = gate.double()
    v = (y.double() * (z * z.sigmoid())).view(n, groups, -1)
    want = (v / (v.pow(2).mean(-1, keepdim=True) + 1e-6).sqrt()).reshape(n, cols) * w.double()
    assert ((out.cpu().double() - want).abs() <= want.abs() * (2 * EPS[dtype] + 16 * EPS[torch.float32]) + 1e-7).all()


def spoiled(n, c, dtype, g):
    """Rows of x (fp32) and of gates with infinities, NaN and gates far below zero among them, and which rows those are."""
    x, gate = torch.randn(n, c, generator=g), torch.randn(n, c, generator=g)
    x[3, 5], x[8, c - 1], x[13, 40] = float("nan"), float("inf"), float("-inf")
    gate[21, 0], gate[34, 33], gate[55, c - 1] = float("nan"), float("inf"), float("-inf")
    gate[60] = torch.linspace(-80, 80, c)
    return x, gate.to(dtype), [3, 8, 13, 21, 34, 55, 60]


def check(y, clean, want, at, dtype, floor):
    """Rows with such values are float64's, NaN for NaN; the others are what they are without them, bit for bit."""
    y, rest = y.cpu(), [i for i in range(len(y)) if i not in at]
    assert torch.equal(y[rest], clean.cpu()[rest])
    a, b = y[at].double(), want[at]
    assert torch.equal(a.isnan(), b.isnan())
    # a rounding of the result, and 64 of fp32 on the way (the exponential of 80 is 40 of them off)
    assert bool((a.isnan() | (a == b) | ((a - b).abs() <= (2 * EPS[dtype] + 64 * 2.0 ** -24) * b.abs() + floor)).all())


@pytest.mark.parametrize("H,dv", [(2, 32), (3, 64), (2, 128)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_heads_that_are_no_numbers(H, dv, dtype):
    from swiftllm_amd.worker.kernels.delta_rule import gated_head_rmsnorm
    g = torch.Generator().manual_seed(dv)
    n, w = 67, torch.randn(dv, generator=g)
    o, gate, at = spoiled(n, H * dv, dtype, g)
    results = []
    for a, b in ((o, gate), (torch.where(torch.isfinite(o), o, 1.0), torch.where(torch.isfinite(gate), gate, 1.0))):
        results.append(torch.empty(n, H * dv, dtype=dtype, device="cuda"))
        gated_head_rmsnorm(results[-1], a.cuda(), b.cuda(), w.cuda(), H, dv, 1e-6, 0.7)
    x, z = o.double().view(n, H, dv), gate.double().view(n, H, dv)
    want = (0.7 * x / (x.pow(2).mean(-1, keepdim=True) + 1e-6).sqrt() * w.double() * (z * z.sigmoid())).reshape(n, -1)
    check(results[0], results[1], want, at, dtype, 2.0 ** -24 if dtype == torch.float16 else 2.0 ** -126)


@pytest.mark.parametrize("cols,groups", [(64, 1), (2048, 2), (4096, 1), (8192, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_groups_that_are_no_numbers(cols, groups, dtype):
    from swiftllm_amd import _hip
    g = torch.Generator().manual_seed(cols)
    n, w = 67, torch.randn(cols, generator=g)
    o, gate, at = spoiled(n, cols, dtype, g)
    results = []
    for a, b in ((o, gate), (torch.where(torch.isfinite(o), o, 1.0), torch.where(torch.isfinite(gate), gate, 1.0))):
        out, a, b, dev = torch.empty(n, cols, dtype=dtype, device="cuda"), a.cuda(), b.cuda(), w.cuda()
        _hip.call("swl_gated_group_rmsnorm", _hip.ptr(out), cols, _hip.ptr(a), _hip.ptr(b), cols, _hip.ptr(dev), 1e-6, n, cols, groups, _hip.dtype_code3(dtype), _hip.stream())
        torch.cuda.synchronize()
        results.append(out)
    x, z = o.double(), gate.double()
    x = (x * (z * z.sigmoid())).view(n, groups, -1)
    want = (x / (x.pow(2).mean(-1, keepdim=True) + 1e-6).sqrt()).reshape(n, -1) * w.double()
    check(results[0], results[1], want, at, dtype, 2.0 ** -24 if dtype == torch.float16 else 2.0 ** -126)
