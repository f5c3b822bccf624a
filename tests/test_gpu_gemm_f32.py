"""Products of a few tokens in true fp32 (csrc/gemm_f32.hip) against float64: edges of the 256-column slices, of the four-row waves and of
the token counts that have a form of their own."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("N,K", [(1, 4), (3, 252), (17, 256), (1025, 1028), (64, 4096), (2048, 512), (4097, 260), (8200, 1024)])
def test_gemm_f32(M, N, K):
    from swiftllm_amd import _hip
    g = torch.Generator().manual_seed(M * N + K)
    x = torch.full((M, K + 8), float("nan"))
    x[:, :K] = torch.randn(M, K, generator=g)
    x, w = x.cuda(), torch.randn(N, K, generator=g).cuda()
    want = x[:, :K].double() @ w.double().t()
    size = x[:, :K].double().abs() @ w.double().abs().t()
    first = None
    for ks in (0, 1, 2, 4):
        out = torch.full((M + 1, N + 4), 7.0, device="cuda")
        _hip.call("swl_gemm_f32", _hip.ptr(out), _hip.ptr(x), _hip.ptr(w), M, N, K, x.stride(0), out.stride(0), ks, _hip.stream())
        # one rounding a term: K / 64 of a lane in a row and at most 24 additions of partial sums
        assert ((out[:M, :N].double() - want).abs() <= (K / 64 + 24) * 2.0 ** -24 * size + 1e-30).all(), ks
        assert (out[M] == 7.0).all() and (out[:, N:] == 7.0).all()
        if ks == 0:
            first = out
    # a token's bits do not hang on its company
    alone = torch.empty(1, N, device="cuda")
    _hip.call("swl_gemm_f32", _hip.ptr(alone), _hip.ptr(x[M - 1]), _hip.ptr(w), 1, N, K, K, N, 0, _hip.stream())
    assert torch.equal(alone[0], first[M - 1, :N])


@pytest.mark.parametrize("M,N,K,form", [(8, 64, 64, "own"), (9, 2049, 64, "library"), (17, 64, 64, "library"), (3, 64, 62, "library"),
                                        (3, 64, 64, "odd"), (3, 64, 64, "columns"), (0, 64, 64, "library")])
def test_linear_f32_routes(M, N, K, form, monkeypatch):
    """What the kernel does not take goes to the library as before: more tokens, odd rows, unaligned or strided columns, no tokens."""
    from swiftllm_amd import _hip
    from swiftllm_amd.worker.kernels.linear import linear_f32
    calls = []
    real = _hip.call
    monkeypatch.setattr(_hip, "call", lambda name, *a: (calls.append(name), real(name, *a))[1])
    g = torch.Generator().manual_seed(5)
    x, w = torch.randn(M, 2 * K + 1, generator=g).cuda(), torch.randn(N, K, generator=g).cuda()
    x = x[:, 1:K + 1] if form == "odd" else x[:, 0:2 * K:2] if form == "columns" else x[:, :K].contiguous()
    got = linear_f32(x, w)
    assert (calls == ["swl_gemm_f32"]) == (form == "own")
    assert torch.allclose(got.double(), x.double() @ w.double().t(), rtol=0, atol=1e-4) and got.shape == (M, N)


@pytest.mark.parametrize("columns", [60, 68, 128])
def test_linear_f32_refuses_rows_of_another_length(columns):
    """A product whose sides have different columns is the library's to refuse: contiguous rows and column slices of wider ones."""
    from swiftllm_amd.worker.kernels.linear import linear_f32
    x, w = torch.randn(3, 128, device="cuda"), torch.randn(64, 64, device="cuda")
    for a in (x[:, :columns], x[:, :columns].contiguous()):
        with pytest.raises(RuntimeError):
            linear_f32(a, w)


@pytest.mark.parametrize("M", [1, 2, 3, 4, 7, 16])
@pytest.mark.parametrize("N1,N2,K,form", [(1, 2, 4, "glu"), (64, 17, 252, ""), (1024, 3200, 1024, ""), (257, 513, 516, "relu2"), (255, 2 * 131, 1028, "glu"),
                                          (4096, 8194, 256, "glu"), (33, 4100, 260, "relu2"), (4097, 64, 64, "refused")])
def test_gemm_f32_pair(M, N1, N2, K, form):
    """Two products in one launch: the bits of the two launches, and of the activation's where the second has one."""
    from swiftllm_amd import _hip
    from swiftllm_amd.worker.kernels.linear import linear_f32_pair
    from swiftllm_amd.worker.kernels.moe import relu_squared
    g = torch.Generator().manual_seed(M + N1 * N2 + K)
    x1, x2, w1, w2 = (torch.randn(n, K, generator=g).cuda() for n in (M, M, N1, N2))

    def alone(x, w):
        out = torch.empty(M, w.shape[0], device="cuda")
        _hip.call("swl_gemm_f32", _hip.ptr(out), _hip.ptr(x), _hip.ptr(w), M, w.shape[0], K, K, w.shape[0], 0, _hip.stream())
        return out

    kw = {"glu": {"glu_limit": 0.75}, "relu2": {"relu2_columns": N2 - 1}}.get(form, {})
    got = linear_f32_pair(x1, w1, x2, w2, **kw)
    served = [_hip.load().swl_gemm_f32_supported(M, n, K) == 2 for n in (N1, N2)]
    if form == "refused" or not all(served):
        assert got is None
        return
    want = alone(x2, w2)
    if form == "glu":
        want, both = torch.empty(M, N2 // 2, device="cuda"), want
        _hip.call("swl_glu_clamp", _hip.ptr(want), _hip.ptr(both), 0, M, N2 // 2, 0.75, 0, _hip.dtype_code3(torch.float32), _hip.stream())
    elif form == "relu2":
        want = torch.cat((relu_squared(want, N2 - 1), want[:, N2 - 1:]), dim=1)
        assert got[1].stride(0) % 4 == 0
    assert torch.equal(got[0], alone(x1, w1)) and torch.equal(got[1], want)
