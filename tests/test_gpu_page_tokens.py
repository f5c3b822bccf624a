"""Stores into transposed pages whose workgroups take their tokens in groups of 128 (csrc/swl_common.h, page_token): a step around the
edges of a group leaves the rows and the pool that the same tokens leave in steps below 128, which keep the grid's order."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
H, G, D = 3, 2, 64


def _kernels():
    from swiftllm_amd.worker.kernels import rope_kv, window_attn as wa
    g = torch.Generator().manual_seed(5)
    w = {n: torch.randn(n, generator=g).cuda() for n in (H * D, G * D, D)}
    freq = (10000.0 ** (-torch.arange(0, D, 2, dtype=torch.float64) / D)).cuda()
    mixer = SimpleNamespace(num_q_heads=H, num_kv_heads=G, head_dim=D, value_dim=D, q_size=H * D, k_size=G * D, v_size=G * D,
                            q_temp_coef=0.1, q_temp_every=16)
    rot = SimpleNamespace(dims=D, half=True, multiplier=1.0)
    latent = SimpleNamespace(num_q_heads=1, head_dim=D, rot_dim=D, kv_rank=2 * D, rot=rot)

    def from_latent(x, *to):
        qa = torch.zeros(x.shape[0], 3 * D, dtype=x.dtype, device="cuda")
        rope_kv.latent_rope_and_store_kv(x, qa, freq, w[G * D], *to, latent, 2 * D, 1e-6)
        return qa

    return {"qknorm": lambda x, *to: wa.qknorm_and_store_kv(x, w[D], w[D], *to, mixer, 1e-6),
            "qknorm_full": lambda x, *to: wa.qknorm_full_and_store_kv(x, w[H * D], w[G * D], *to, mixer, 1e-6, True),
            "bias_norm": lambda x, *to: wa.qkv_bias_norm_store(x, w[H * D], w[G * D], w[G * D], w[D], None, *to, mixer, 1e-6),
            "rope": lambda x, *to: rope_kv.rope_and_store_kv(x, freq, D, *to, H, G, G, D, D),
            "qk_norm_rope": lambda x, *to: rope_kv.qk_norm_rope_and_store_kv(x, None, None, w[D], w[D], None, freq, rot, *to, H, G, G, D, D, 1e-6),
            "latent": from_latent}


@pytest.mark.parametrize("tokens", [127, 128, 129, 255, 256, 300])
@pytest.mark.parametrize("name", ["qknorm", "qknorm_full", "bias_norm", "rope", "qk_norm_rope", "latent"])
def test_same_pool(name, tokens):
    from swiftllm_amd.worker.kernels.window_attn import PoolSlice
    run, g = _kernels()[name], torch.Generator().manual_seed(tokens)
    rows = torch.randn(tokens, (H + 2 * G) * D, generator=g).to(torch.bfloat16).cuda()
    first = tokens // 3                 # two sequences, the second from the middle of a page on
    seq = torch.tensor([0] * first + [1] * (tokens - first), dtype=torch.int32, device="cuda")
    pos = torch.cat([torch.arange(first), 7 + torch.arange(tokens - first)]).int().cuda()
    table = torch.randperm(64, generator=g)[:2 * 21].view(2, 21).int().cuda()
    results = []
    for step in (tokens, 100):
        x, pool, made = rows.clone(), torch.zeros(64, 2 * G * D * 16 + D * 16, dtype=torch.bfloat16, device="cuda"), []
        for a in range(0, tokens, step):
            part = x[a:a + step]
            made.append(run(part, pool, PoolSlice(0, 3 * D * 16 if name == "latent" else G * D * 16), table, seq[a:a + step], pos[a:a + step]))
        results.append([x, pool] + ([torch.cat(made)] if made[0] is not None else []))
    assert results[0][1].any()
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.parametrize("tokens", [128, 129, 300])
@pytest.mark.parametrize("taps", [2, 4, 5])
def test_same_pool_and_carried_inputs(taps, tokens):
    """The kernel whose tokens also read their neighbours' rows and write the sequence's carried convolution inputs: what a whole step stores
    and carries on to the next tokens is what steps below 128 do."""
    from test_gpu_lorulix import Slots
    from swiftllm_amd.worker.kernels.rope_kv import qkv_conv_rope_and_store_kv
    from swiftllm_amd.worker.kernels.window_attn import PoolSlice
    g = torch.Generator().manual_seed(tokens + taps)
    C = (H + 2 * G) * D
    rand = lambda *shape: torch.randn(*shape, generator=g)      # noqa: E731
    bias, conv, norm = rand(C).cuda(), (rand(taps, C) / taps ** 0.5).cuda(), (1 + 0.3 * rand(D)).cuda()
    freq = (10000.0 ** (-torch.arange(0, D, 2, dtype=torch.float64) / D)).cuda()
    rot = SimpleNamespace(dims=D, half=True, multiplier=1.0)
    rows = rand(7 + tokens + 10, C).to(torch.bfloat16).cuda()
    table = torch.randperm(64, generator=g)[:2 * 21].view(2, 21).int().cuda()
    first = tokens // 3         # of sequence 0; the rest goes on with sequence 1, which has 7 tokens already
    order = [(0, i) for i in range(first)] + [(1, 7 + i) for i in range(tokens - first)]
    results = []
    for most in (tokens, 100):
        slots, pool, made = Slots([2 * (taps - 1) * C], num_slots=2), torch.zeros(64, 2 * G * D * 16, dtype=torch.bfloat16, device="cuda"), []
        at = 0
        steps = [[(1, 0, 7)]]
        for a in range(0, tokens, most):
            part = order[a:a + most]
            steps.append([(s, min(p for x, p in part if x == s), sum(x == s for x, _ in part)) for s in sorted({x for x, _ in part})])
        steps.append([(0, first, 5), (1, 7 + tokens - first, 5)])       # (reads what was carried)
        for portions in steps:
            n = sum(c for _, _, c in portions)
            made.append(qkv_conv_rope_and_store_kv(rows[at:at + n], bias, conv, norm, norm, freq, rot, pool, PoolSlice(0, G * D * 16), table,
                                                   slots.ref(portions), slots.off[0], H, G, D, D, D, D, 1e-6))
            at += n
        results.append((torch.cat(made), pool))
    assert bool(torch.isfinite(results[0][0].float()).all()) and results[0][1].any()
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("taps,dim,vdim,rot_dims,half", [(4, 128, 64, 64, True), (1, 64, 128, 64, False), (3, 16, 24, 16, True), (2, 32, 32, 8, False),
                                                         (0, 128, 128, 0, True)])
def test_four_tokens_a_workgroup(taps, dim, vdim, rot_dims, half, dtype):
    """From 4096 tokens of any width a workgroup takes four in a row, whose portions may begin and end between them: the rows, pages and carried
    inputs of steps of fewer (below 1536: one)."""
    from test_gpu_lorulix import Slots
    from swiftllm_amd.worker.kernels.rope_kv import qkv_conv_rope_and_store_kv
    from swiftllm_amd.worker.kernels.window_attn import PoolSlice
    g = torch.Generator().manual_seed(dim + taps)
    heads, kv, kd, vd = 3, 2, dim + 8, vdim + 8
    C = (heads + kv) * dim + kv * vdim
    rand = lambda *shape: torch.randn(*shape, generator=g)      # noqa: E731
    bias, conv, norm = rand(C).cuda(), (rand(taps, C) / taps ** 0.5).cuda() if taps else None, (1 + 0.3 * rand(dim)).cuda()
    freq = (777.0 ** (-torch.arange(0, rot_dims, 2, dtype=torch.float64) / rot_dims)).cuda() if rot_dims else None
    rot = SimpleNamespace(dims=rot_dims, half=half, multiplier=1.0)
    lens, cuts = [1, 2, 1, 5, 3, 1000, 1, 1, 520, 3, 1400, 2, 1161, 1], [0, 6, 10, 12, 14]
    assert sum(lens) >= 4096 and sum(lens) % 4 and max(sum(lens[a:b]) for a, b in zip(cuts, cuts[1:])) < 1536
    ahead = [(s, 0, 3) for s in range(0, len(lens), 2)]         # (half of the sequences have tokens already)
    begin = [3 if s % 2 == 0 else 0 for s in range(len(lens))]
    total = sum(c for _, _, c in ahead) + sum(lens) + len(lens)
    rows = rand(total, C).to(dtype).cuda()
    table = torch.randperm(90 * len(lens), generator=g).view(len(lens), 90).int().cuda()
    results = []
    for whole in (True, False):
        slots, made, at = Slots([2 * max(taps - 1, 0) * C], num_slots=len(lens)), [], 0
        pool = torch.zeros(table.numel(), kv * (kd + vd) * 16, dtype=dtype, device="cuda")
        main = [(s, begin[s], c) for s, c in enumerate(lens)]
        steps = [ahead] + ([main] if whole else [main[a:b] for a, b in zip(cuts, cuts[1:])]) + [[(s, begin[s] + c, 1) for s, c in enumerate(lens)]]
        for portions in steps:
            n = sum(c for _, _, c in portions)
            made.append(qkv_conv_rope_and_store_kv(rows[at:at + n], bias, conv, norm, norm, freq, rot, pool, PoolSlice(0, kv * kd * 16), table,
                                                   slots.ref(portions), slots.off[0], heads, kv, dim, vdim, kd, vd, 1e-6))
            at += n
        assert at == total
        results.append((torch.cat(made), pool))
    assert bool(torch.isfinite(results[0][0].float()).all()) and results[0][1].any()
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("heads,kv,dim,vdim,n", [(3, 1, 128, 64, 33), (5, 2, 64, 8, 5), (1, 1, 16, 128, 17), (33, 3, 128, 128, 3), (4, 4, 32, 40, 150),
                                                  (4, 2, 64, 36, 33), (3, 1, 128, 20, 5), (3, 3, 64, 33, 150)])
@pytest.mark.parametrize("kind", ["bias_norm", "bias", "mix", "mix_slice", "full", "norm"])
def test_rows_of_aligned_eights(kind, heads, kv, dim, vdim, n, dtype):
    """Rows in registers against the kernel for any rows, which takes them where their stride is not a multiple of 16 bytes: one rounding of the
    type apart, sums of up to 4224 squares in another order; values in whole pieces of eight over all heads or not, or beside another layer's that
    start anywhere; with and without a pool."""
    from swiftllm_amd.worker.kernels import window_attn as wa
    g = torch.Generator().manual_seed(heads * dim + vdim)
    rand = lambda *shape: torch.randn(*shape, generator=g)      # noqa: E731
    nq, nk, nv = heads * dim, kv * dim, kv * vdim
    C = nq + nk + nv
    rows, other = rand(n, C).to(dtype), rand(n, nv + 3).to(dtype).cuda()
    other = other[:, 3:] if kind == "mix_slice" else other[:, :nv].contiguous()
    w = {size: (1 + 0.3 * rand(size)).cuda() for size in {nq, nk, nv, dim}}
    mixer = SimpleNamespace(num_q_heads=heads, num_kv_heads=kv, head_dim=dim, value_dim=vdim, q_size=nq, k_size=nk, v_size=nv, q_temp_coef=0.1,
                            q_temp_every=3)
    pos, seq = torch.arange(n, dtype=torch.int32).cuda(), torch.zeros(n, dtype=torch.int32).cuda()
    table = torch.randperm(12, generator=g).view(1, 12).int().cuda()
    for with_pool in (True, False):
        results = []
        for extra in (8 + -C % 8, 1 + C % 2):
            wide = torch.zeros(n, C + extra, dtype=dtype)
            wide[:, :C] = rows
            wide = wide.cuda()
            x = wide[:, :C]
            pool = torch.zeros(12, 16 * (nk + nv), dtype=dtype, device="cuda") if with_pool else None
            to = (pool, wa.PoolSlice(0, 16 * nk), table, seq, pos, mixer, 1e-6)
            if kind == "norm":
                wa.qknorm_and_store_kv(x, w[dim], w[dim], *to)
            elif kind == "full":
                wa.qknorm_full_and_store_kv(x, w[nq], w[nk], *to, True)
            elif kind == "bias":
                wa.qkv_bias_norm_store(x, None, w[nk], w[nv], None, None, *to)
            else:
                wa.qkv_bias_norm_store(x, w[nq], w[nk], w[nv], w[dim], None, *to, *((other, 0.3) if kind in ("mix", "mix_slice") else ()))
            assert bool((wide[:, C:] == 0).all())
            results.append((x.double(), pool.double() if with_pool else x.double()))
        eps = {torch.float32: 2.0 ** -20, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dtype]
        for a, b in zip(*results):
            assert bool(((a - b).abs() <= eps * (b.abs() + 2.0 ** -10)).all())
