"""The tiled products of prompt-sized steps (csrc/gemm_tile.hip) against products in 64 bits: every tile at the edges of its rows, columns and of the
turns that its workgroups take, every activation, several matrices x in one launch, rows with gaps, and what is left to the library."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(out, x, w, n, shape, act=0, act_cols=0, limit=0.0, x_cols=0, x_next=0):
    from swiftllm_amd import _hip
    m, k = out.shape[0], w.shape[1]
    _hip.call("swl_gemm_tile", _hip.ptr(out), _hip.ptr(x), _hip.ptr(w), m, n, k, x.stride(-2), out.stride(0), x_cols, x_next, act, act_cols,
              float(limit), shape, _hip.dtype_code(out.dtype), _hip.stream())
    torch.cuda.synchronize()


def _operands(m, n, k, dtype, groups=1):
    g = torch.Generator(device="cuda").manual_seed(m + 3 * n + k)
    x = torch.randn((groups * m, k + 8), generator=g, device="cuda").to(dtype)[:, :k]        # rows with gaps
    w = (torch.randn((n, k), generator=g, device="cuda") / k ** 0.5).to(dtype)
    return x, w


def _product_bound(z, x, w):
    """Largest difference of a product whose fp32 sums may run in any order (each addition rounds by 2^-24 of the magnitudes' sum, K of them at
    most), rounded once: half an ulp, or a whole one where the sums straddle."""
    ulp = 2.0 ** -10 if x.dtype == torch.float16 else 2.0 ** -7
    return ulp * z.abs() + 2.0 ** -24 * x.shape[1] * (x.double().abs() @ w.double().abs().T) + (2.0 ** -24 if x.dtype == torch.float16 else 0.0)


SIZES = [(1, 8, 256), (257, 136, 384), (300, 1032, 256), (129, 264, 640), (65, 1000, 1024), (1025, 520, 512), (2500, 3080, 256), (700, 72, 2048)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", range(12))
@pytest.mark.parametrize("m,n,k", SIZES + [(4500, 4352, 256)])
def test_products_are_rounded_once(m, n, k, shape, dtype):
    x, w = _operands(m, n, k, dtype)
    out = torch.full((m + 2, n + 16), 7.0, dtype=dtype, device="cuda")
    _run(out[:m, :n], x, w, n, shape)
    z = x.double() @ w.double().T
    assert bool(((out[:m, :n].double() - z).abs() <= _product_bound(z, x, w)).all())
    assert bool((out[m:] == 7).all()) and bool((out[:, n:] == 7).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [1, 2, 3, 4, 5, 6, 10, 11])
@pytest.mark.parametrize("m,n,k", SIZES)
def test_gated_units_and_squared_relu(m, n, k, shape, dtype):
    """A unit f(a, b) of two rounded products that may be an ulp off each: |df/da| |a| + |df/db| |b| ulps, and an ulp of the result (two where it is
    rounded in between). |d silu| <= 1.1 and |silu| <= |z|, |d (z sigmoid(1.702 z))| <= 1.2, relu(z)^2 has 2 z."""
    ulp = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7
    x, w = _operands(m, 2 * n, k, dtype)
    z = x.double() @ w.double().T
    slack = _product_bound(z, x, w)
    a, b, da, db = z[:, :n], z[:, n:], slack[:, :n], slack[:, n:]
    silu, limit = torch.nn.functional.silu, 0.7
    g, u = a.clamp(max=limit), b.clamp(-limit, limit)
    wants = {2: (g * torch.sigmoid(1.702 * g) * (u + 1), 1.2 * da * (u.abs() + 1) + db * g.abs()), 3: (silu(a) * b, 1.1 * da * b.abs() + db * a.abs()),
             4: (silu(b) * a, 1.1 * db * a.abs() + da * b.abs()), 5: (silu(b) * a, 1.1 * db * a.abs() + da * b.abs() + ulp * (silu(b) * a).abs())}
    floor = 2.0 ** -24 if dtype == torch.float16 else 0.0
    for act, (want, off) in wants.items():
        out = torch.full((m + 1, n + 8), 7.0, dtype=dtype, device="cuda")
        _run(out[:m, :n], x, w, n, shape, act, 0, limit)
        # (da db: both products off at once; 2^-20: expf and the unit's own fp32 roundings)
        assert bool(((out[:m, :n].double() - want).abs() <= off + da * db + (ulp + 2.0 ** -20) * want.abs() + floor).all()), act
        assert bool((out[m:] == 7).all()) and bool((out[:, n:] == 7).all())
    cols = max(4, n // 2 // 4 * 4)
    out = torch.empty((m, n), dtype=dtype, device="cuda")
    _run(out, x, w[:n], n, shape, 1, cols)
    want, off = a.clone(), da.clone()
    want[:, :cols] = torch.relu(a[:, :cols]) ** 2
    off[:, :cols] = (2 * a[:, :cols].abs() + da[:, :cols]) * da[:, :cols] + ulp * want[:, :cols] + floor
    assert bool(((out.double() - want).abs() <= off).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", range(12))
def test_columns_of_several_matrices(shape, dtype):
    from swiftllm_amd.worker.kernels.linear import linear_grouped
    m, groups, size, k = 333, 3, 768 if shape in (3, 6, 8, 9) else 512, 384      # (those are 192 columns wide)
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn((groups, m, k), generator=g, device="cuda").to(dtype)
    w = (torch.randn((groups * size, k), generator=g, device="cuda") / k ** 0.5).to(dtype)
    out = torch.empty((m, groups * size), dtype=dtype, device="cuda")
    _run(out, x, w, groups * size, shape, x_cols=size, x_next=m * k)
    for i in range(groups):
        cols = slice(i * size, (i + 1) * size)
        z = x[i].double() @ w[cols].double().T
        assert bool(((out[:, cols].double() - z).abs() <= _product_bound(z, x[i], w[cols])).all())
    if shape == 0:
        assert torch.equal(linear_grouped(x, w, True), out)


def test_ragged_rows_and_what_is_left_to_the_library():
    from swiftllm_amd.worker.kernels.linear import TILE_RELU2, linear, linear_gated, linear_tile
    x, w = _operands(400, 1025, 512, torch.bfloat16)
    y = linear_tile(x, w, TILE_RELU2, 1024)
    z = x.double() @ w.double().T
    assert y.shape == (400, 1025) and y.stride(0) == 1032
    assert bool(((y[:, 1024].double() - z[:, 1024]).abs() <= _product_bound(z, x, w)[:, 1024]).all())
    assert bool(((y.float()[:, :1024] - torch.relu(z.float()[:, :1024]) ** 2).norm() <= 1e-2 * (z[:, :1024] ** 2).norm()))
    assert linear_tile(x[:256], w) is None and linear_tile(x.float(), w.float()) is None and linear_tile(x[:, :456], w[:, :456]) is None
    assert linear_tile(x[:, 4:], w[:, :508].contiguous()) is None and linear_gated(x, w, 1) is None
    long_x, long_w = _operands(300, 512, 4096, torch.bfloat16)      # few tiles, long sums
    assert linear_tile(long_x, long_w) is None
    for a, b in ((long_x, long_w), (x[:, :456], w[:, :456].contiguous()), (x, w)):
        z = a.double() @ b.double().T
        assert bool(((linear(a, b, True).double() - z).abs() <= _product_bound(z, a, b)).all())


def test_replayed_from_a_graph_beside_other_launches():
    x, w = _operands(3000, 2048, 512, torch.bfloat16)
    out = torch.empty((3000, 2048), dtype=torch.bfloat16, device="cuda")
    _run(out, x, w, 2048, 0)
    want, graph = out.clone(), torch.cuda.CUDAGraph()
    from swiftllm_amd.worker.kernels.linear import linear
    with torch.cuda.graph(graph):
        got = linear(x, w, True)
    for _ in range(3):
        got.zero_()
        graph.replay()
        assert torch.equal(got, want)
        (x.float() @ w.float().T).sum().item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,top,experts,K,N", [
    (700, 2, 8, 256, 136),          # tiles of 128 x 128, a column tile of 8, experts that end anywhere in a tile
    (300, 1, 70, 384, 264),         # more experts than lanes, most of them a few rows
    (40, 3, 130, 512, 72),          # more experts than rows, no assignments for some
    (4000, 2, 5, 256, 2048),        # several tiles a workgroup
    (6000, 2, 3, 1024, 1024),       # tiles of 256 x 128 and 256 x 256
    (9000, 2, 8, 512, 4096)])
def test_products_of_experts(n, top, experts, K, N, dtype):
    """Rows gathered through the sorted assignments (weights on the products or none), and rows by position, against products in 64 bits."""
    from swiftllm_amd import _hip
    g = torch.Generator(device="cuda").manual_seed(n + K)
    total = n * top
    idx = (torch.rand((n, top), generator=g, device="cuda") ** 2 * experts).int().clamp(max=experts - 1)      # (some experts take most)
    idx[idx == 1] = 0
    order, where = torch.empty(total, dtype=torch.int32, device="cuda"), torch.empty(total, dtype=torch.int64, device="cuda")
    offsets = torch.empty(experts + 1, dtype=torch.int32, device="cuda")
    _hip.call("swl_moe_sort", _hip.ptr(order), _hip.ptr(where), _hip.ptr(offsets), _hip.ptr(idx), total, experts, _hip.stream())
    x = torch.randn((n, K), generator=g, device="cuda").to(dtype)
    w = (torch.randn((experts, 2 * N, K), generator=g, device="cuda") / K ** 0.5).to(dtype)
    in_w = torch.rand(total, generator=g, device="cuda") + 0.5
    ulp, floor = (2.0 ** -10, 2.0 ** -24) if dtype == torch.float16 else (2.0 ** -7, 0.0)
    flat, bounds = order.long(), offsets.tolist()
    z = torch.empty((total, 2 * N), dtype=torch.float64, device="cuda")
    size = torch.empty_like(z)
    xs = x[flat // top].double()
    for e in range(experts):
        a, b = bounds[e], bounds[e + 1]
        z[a:b], size[a:b] = xs[a:b] @ w[e].double().T, xs[a:b].abs() @ w[e].double().abs().T
    off = 2.0 ** -24 * K * size        # (fp32 sums in any order)
    limit = 0.7
    for mode, act, weigh, ordered in ((0, 0, False, True), (1, 0, True, True), (1, 1, True, True), (1, 1, False, True), (2, 0, False, True), (0, 0, False, False)):
        cols = 2 * N if mode == 1 else N
        ww = w if mode == 1 else w[:, :N].contiguous()
        rows = x if ordered else xs.to(dtype)
        out = torch.full((total + 1, N), 7.0, dtype=dtype, device="cuda")
        _hip.call("swl_moe_gemm", _hip.ptr(out), _hip.ptr(rows), _hip.ptr(ww), _hip.ptr(order) if ordered else 0, _hip.ptr(offsets),
                  _hip.ptr(in_w) if weigh else 0, total, rows.shape[0], top, experts, K, N, mode, act, limit, _hip.dtype_code(dtype), _hip.stream())
        torch.cuda.synchronize()
        scale = in_w[flat].double()[:, None] if weigh else 1.0
        p, d = z[:, :cols] * scale, off[:, :cols] * scale
        if mode == 1:
            f, s, df, ds = p[:, :N], p[:, N:], d[:, :N], d[:, N:]
            if act == 0:
                f, s = f.clamp(max=limit), s.clamp(-limit, limit)
                want, slack = f * torch.sigmoid(1.702 * f) * (s + 1), 1.2 * df * (s.abs() + 1) + ds * f.abs()
            else:
                want, slack = torch.nn.functional.silu(f) * s, 1.1 * df * s.abs() + ds * f.abs()
            slack = slack + df * ds + 2.0 ** -20 * want.abs()      # (the unit's own fp32 roundings)
        elif mode == 2:
            want, slack = torch.relu(p) ** 2, (2 * p.abs() + d) * d
        else:
            want, slack = p, d
        assert bool(((out[:total].double() - want).abs() <= slack + ulp * want.abs() + floor).all()), (mode, act, weigh, ordered)
        assert bool((out[total] == 7).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", range(12))
@pytest.mark.parametrize("m,n,k,splits", [(1, 8, 512, 2), (257, 136, 768, 3), (300, 1032, 2048, 8), (129, 264, 1280, 5), (1025, 520, 1024, 2), (2500, 3080, 512, 2), (700, 72, 256, 1)])
def test_slabs_of_k_shares(m, n, k, splits, shape, dtype):
    """Every slab is the fp32 sum over its share, whatever the order of the additions; nothing is written behind the last."""
    from swiftllm_amd import _hip
    x, w = _operands(m, n, k, dtype)
    slabs = torch.full((splits * m + 2, n), 7.0, device="cuda")
    _hip.call("swl_gemm_tile_partial", _hip.ptr(slabs), splits * m * n * 4, _hip.ptr(x), _hip.ptr(w), m, n, k, x.stride(0), splits, shape,
              _hip.dtype_code(dtype), _hip.stream())
    xs, ws = x.double().reshape(m, splits, -1).transpose(0, 1), w.double().reshape(n, splits, -1).permute(1, 2, 0).contiguous()
    bound = 2.0 ** -24 * (k // splits) * (xs.abs() @ ws.abs()).reshape(-1, n) + 2.0 ** -24 * (xs @ ws).reshape(-1, n).abs()
    assert bool(((slabs[:splits * m].double() - (xs @ ws).reshape(-1, n)).abs() <= bound).all())
    assert bool((slabs[splits * m:] == 7).all())


@pytest.mark.parametrize("m,n,k,want", [(300, 1024, 4096, True), (2029, 1024, 6144, True), (600, 2048, 8192, True), (300, 4096, 14336, True),
                                        (7691, 1024, 1024, False), (5112, 4096, 14336, False), (256, 1024, 4096, False), (300, 1026, 4096, False)])
def test_slabs_where_tiles_are_few(m, n, k, want):
    """What linear_tile_partial takes, and that its sums are those of the product's rows (whose one rounding is the difference)."""
    from swiftllm_amd.worker.kernels import rms_stream
    from swiftllm_amd.worker.kernels.linear import linear, linear_tile_partial
    x, w = _operands(m, n, k, torch.bfloat16)
    parts = linear_tile_partial(x, w)
    assert (parts is not None) == want
    if not want:
        return
    z = x.double() @ w.double().T
    assert bool(((parts.materialize().double() - z).abs() <= _product_bound(z, x, w)).all())
    # the fp32 stream's step on the slabs and on the rows: y / rms(y) of rows of about unit size, each rounded by half an ulp
    g = torch.Generator(device="cuda").manual_seed(1)
    stream, ones = torch.randn((m, n), generator=g, device="cuda"), torch.ones(n, device="cuda")
    a, b = stream.clone(), stream.clone()
    rms_stream.gated_add_rmsnorm(a, parts, post=ones, pre=ones)
    rms_stream.gated_add_rmsnorm(b, linear(x, w, skinny=True), post=ones, pre=ones)
    rms = z.pow(2).mean(-1, keepdim=True).sqrt()
    assert bool(((a - b).double().abs() <= 2 * _product_bound(z, x, w) / rms + 2.0 ** -7 * (z / rms).abs()).all())
