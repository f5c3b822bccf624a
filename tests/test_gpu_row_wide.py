"""Residual steps with rows in registers (csrc/row_wide.h: rms_stream.hip, layernorm.hip) against float64, at the edges of every split of a
row: one wave, two or four a row, the last columns of a row and the last rows of a launch, and rows that stay with the other kernels."""
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 1e-5
# (1024 rows: a wave a row up to 1024 columns, two up to 2048; 2050 and 8196 columns: column by column)
SHAPES = [(3, 4), (33, 260), (5, 1024), (1025, 1024), (1023, 1024), (1027, 60), (2, 1028), (1026, 1028), (1025, 2048), (7, 2048), (3, 2050),
          (1024, 3000), (2, 4096), (3, 4100), (2, 8188), (1, 8196)]


def _rms(x):
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS)


def _ln(x, wb):
    d = x - x.mean(1, keepdim=True)
    return d / torch.sqrt((d * d).mean(1, keepdim=True) + EPS) * wb[0].double() + wb[1].double()


def _close(x, out, want, out_want, dtype):
    # the stream: a few fp32 roundings of the row's values and of a sum of up to 8196 squares; the result: one rounding to its type on top
    scale = max(1.0, float(want.abs().max()))
    assert (x.double().cpu() - want).abs().max() <= 4e-6 * scale
    eps = {torch.float32: 4e-6, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -10}[dtype]
    assert ((out.double().cpu() - out_want).abs() <= eps * out_want.abs() + 4e-6 * float(out_want.abs().max())).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,width", SHAPES)
def test_rows(rows, width, dtype):
    from swiftllm_amd.worker.kernels.layernorm import add_layernorm
    from swiftllm_amd.worker.kernels.rms_stream import gated_add_rmsnorm, post_norm_add
    g = torch.Generator().manual_seed(rows + width)
    x, x0 = torch.randn(rows, width, generator=g) * 2, torch.randn(rows, width, generator=g)
    a, b, r, s = (torch.randn(rows, n, generator=g).to(dtype) for n in (width, width, width + 8, 3))
    w = [1 + 0.2 * torch.randn(width, generator=g) for _ in range(4)]
    bias = torch.randn(width, generator=g)
    xd, ad, bd, rd = x.double(), a.double(), b.double(), r.double()
    wd, wc = [v.double() for v in w], [v.cuda() for v in w]

    for shift in (4, 2):        # (2: a gate that is not aligned goes column by column)
        gpu = x.cuda()
        out = gated_add_rmsnorm(gpu, a.cuda(), wc[0], r.cuda()[:, shift:shift + width], bias.cuda(), b.cuda(), s.cuda()[:, 1:2], wc[1], EPS)
        y = (ad + torch.sigmoid(s.double()[:, 1:2]) * bd) * torch.sigmoid(rd[:, shift:shift + width] + bias.double())
        want = xd + _rms(y) * wd[0]
        _close(gpu, out, want, _rms(want) * wd[1], dtype)

    for norms in (True, False):
        if 2 * width + 4 > 16384:
            break
        gpu = x.cuda()
        out = post_norm_add(gpu, a.cuda(), wc[0], b.cuda(), wc[1] if norms else None, wc[2] if norms else None, 0.5, wc[3] if norms else None, EPS)
        y = 0.5 * (_rms(ad) * wd[1] + _rms(bd) * wd[2] if norms else ad + bd)
        want = xd + _rms(y) * wd[0]
        _close(gpu, out, want, _rms(want) * wd[3] if norms else want, dtype)

    gpu = x.cuda()
    out = add_layernorm(gpu, a.cuda(), 0.3, (wc[0], wc[1]), x0.cuda(), bias.cuda(), (wc[2], wc[3]), EPS)
    want = xd + 0.3 * _ln(ad, w[:2]) + x0.double() + bias.double()
    _close(gpu, out, want, _ln(want, w[2:]), dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,width,parts", [(1, 1024, 1), (5, 1028, 3), (33, 2048, 4), (7, 4096, 8), (3, 8192, 16), (200, 3000, 5), (1025, 64, 2)])
def test_slabs_of_a_split_product(rows, width, parts, dtype):
    """The sublayer's result as the fp32 slabs of a product whose K was split, added up here, or before where the gate is not aligned."""
    from swiftllm_amd.worker.kernels.linear import SplitKPartials
    from swiftllm_amd.worker.kernels.rms_stream import gated_add_rmsnorm
    g = torch.Generator().manual_seed(rows + width)
    slabs = torch.randn(parts, rows, width, generator=g) * parts ** -0.5
    x, b, r, s = (torch.randn(rows, n, generator=g) for n in (width, width, width + 8, 1))
    b, r, s = b.to(dtype), r.to(dtype), s.to(dtype)
    w, w2, bias = 1 + 0.2 * torch.randn(width, generator=g), 1 + 0.2 * torch.randn(width, generator=g), torch.randn(width, generator=g)
    for shift in (4, 2):
        gpu = x.cuda()
        out = gated_add_rmsnorm(gpu, SplitKPartials(slabs.cuda(), parts, rows, width, dtype), w.cuda(), r.cuda()[:, shift:shift + width],
                                bias.cuda(), b.cuda(), s.cuda(), w2.cuda(), EPS)
        m = slabs.double().sum(0)
        y = (m + torch.sigmoid(s.double()) * b.double()) * torch.sigmoid(r.double()[:, shift:shift + width] + bias.double())
        want = x.double() + _rms(y) * w.double()
        if shift == 4:
            _close(gpu, out, want, _rms(want) * w2.double(), dtype)
        else:       # one rounding of m to its type first
            eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
            assert (gpu.double().cpu() - want).abs().max() <= 4 * eps * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,width", [(3, 1028), (32, 2048), (6, 4096), (2, 8192), (1030, 1000), (1030, 1544)])
def test_one_slab(rows, width, dtype):
    """A product that was not split, for every number of columns that a thread holds."""
    test_slabs_of_a_split_product(rows, width, 1, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,width,taps,form", [(1, 4, 4, "m"), (3, 1024, 3, "gated"), (5, 1028, 2, "parts"), (4, 2048, 4, "none"), (7, 2052, 1, "m"),
                                                  (1100, 1020, 3, "gated"), (2, 4096, 4, "parts"), (3, 1022, 3, "m"), (3, 4096, 5, "none")])
def test_gated_add_rmsnorm_conv(rows, width, taps, form, dtype):
    """The convolution in the norm's launch: the stream and the normed rows as the norm alone leaves them, the sum and the carried inputs
    (bit by bit) as the convolution of these rows does. Rows and taps the kernel does not take are refused by `fits`."""
    from swiftllm_amd.worker.kernels.rms_stream import ConvInput, StateRef, causal_conv_state, gated_add_rmsnorm
    from swiftllm_amd.worker.kernels.linear import SplitKPartials
    g = torch.Generator().manual_seed(rows * width + taps)
    rand = lambda *shape, dt=torch.float32: torch.randn(*shape, generator=g).to(dt).cuda()
    off, slots = 12, rows + 2
    pool = rand(slots, off + 2 * (taps - 1) * width + 4)
    pos = torch.tensor([(0, 1, 2, 3, 9)[i % 5] for i in range(rows)], dtype=torch.int32).cuda()
    code = (2 * torch.randperm(slots, generator=g)[:rows] + torch.arange(rows) % 2).to(torch.int32).cuda()
    seq = torch.arange(rows, dtype=torch.int32).cuda()
    x, w, post, pre, bias = rand(rows, width), rand(taps, width), rand(width), rand(width), rand(width)
    kw = {"eps": EPS, "pre": pre, "out_dtype": dtype}
    if form == "parts":
        kw["m"] = SplitKPartials(rand(3, rows, width), 3, rows, width, dtype)
    elif form != "none":
        kw["m"] = rand(rows, width, dt=dtype)
    if form == "gated":
        kw |= {"gate": rand(rows, width, dt=dtype), "gate_bias": bias, "m2": rand(rows, width, dt=dtype), "m2_gate": rand(rows, 3, dt=dtype)[:, 1:2]}
    kw["post"] = post
    st = StateRef(pool.clone(), pos, pos, code, seq, seq, torch.ones_like(seq), longest=1)
    conv, x1 = ConvInput(w, st, off), x.clone()
    if width % 4 or taps > 4:
        assert not conv.fits(x1)
        return
    assert conv.fits(x1)
    h, total = gated_add_rmsnorm(x1, conv=conv, **kw)
    x2 = x.clone()
    gated_add_rmsnorm(x2, **kw)
    _close(x1, h, x2.double().cpu(), _rms(x2.double().cpu()) * pre.double().cpu(), dtype)
    ref = StateRef(pool.clone(), pos, pos, code, seq, seq, torch.ones_like(seq), longest=1)
    want = causal_conv_state(h, w, ref, off, add_input=True).double()
    assert torch.equal(st.pool, ref.pool)
    # up to five fp32 terms, whose products a compiler may or may not round before they are added, then one rounding to the type
    size = 5 * (w.double().abs().sum(0) + 1) * max(float(pool.abs().max()), float(h.abs().max()))
    eps = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dtype]
    assert ((total.double() - want).abs() <= eps * want.abs() + 2.0 ** -24 * size).all()
