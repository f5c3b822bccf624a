"""The per-token attention and expert kernels (csrc/window_attn.hip, sigmoid_attn.hip, moe.hip) against float64: rows that are and are
not whole 16-byte pieces, windows that begin inside a page, contexts at page and chunk borders, key shares with and without keys."""
import pytest
import torch

from test_gpu_span_attn import _pool, _spans, _want

pytestmark = pytest.mark.gpu

PARTS = [(1, 0, 3), (2, 62, 4), (3, 300, 2), (4, 15, 1), (5, 128, 1)]


def _bound(want, dtype):
    """fp32: rounding of sums of some hundred terms of order one; 16 bits: the result's own rounding (the inputs are the same)."""
    eps = {torch.float32: 2.0 ** -18, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    return 1.1 * eps * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,G,d,dv,window,kind", [(8, 2, 128, 128, 0, "rel"), (8, 1, 576, 512, 70, "sink"), (6, 2, 36, 33, 37, "slopes"),
                                                  (5, 5, 10, 7, 0, "plain"), (16, 1, 64, 64, 48, "gate"), (40, 20, 24, 100, 0, "plain")])
def test_softmax_attention(H, G, d, dv, window, kind, dtype):
    from swiftllm_amd.worker.kernels import window_attn as wa
    g = torch.Generator().manual_seed(d)
    pool, sl, table, ks, vs = _pool([a + n for _, a, n in PARTS], G, G, d, dv, dtype, g)
    seq, pos, _ = _spans(PARTS)
    n = seq.shape[0]
    q = torch.randn(n, H * d, generator=g).to(dtype)
    rel = torch.randn(H, 90, generator=g) if kind == "rel" else None
    gate = torch.randn(n, H * dv, generator=g).to(dtype) if kind == "gate" else None
    spec = wa.AttentionSpec(H, G, d, dv, d ** -0.5, window=window, sink=torch.randn(H, generator=g).cuda() if kind == "sink" else None,
                            slopes=(torch.rand(H, generator=g) * 0.1).cuda() if kind == "slopes" else None)
    for reach in (4096, 64):        # (sixteen key shares; one)
        if kind == "rel":
            mixer = type("Mixer", (), dict(num_q_heads=H, num_kv_heads=G, head_dim=d, value_dim=dv, window=0, scale=d ** -0.5, softcap=0.0))
            o = wa.window_attention(q.cuda(), None, pool, sl, table, seq, pos, mixer, None, reach, rel=rel.cuda())
        else:
            o = wa.masked_attention(q.cuda(), pool, sl, table, seq, pos, spec, None, reach, gate=gate.cuda() if gate is not None else None)
        at = 0
        for b, (_, a, m) in enumerate(PARTS):
            want = _want(q[at:at + m].double().view(m, H, d), ks[b], vs[b], a, spec, rel.double() if rel is not None else None,
                         gate[at:at + m].double() if gate is not None else None)
            assert (o[at:at + m].double().cpu() - want).abs().max() <= _bound(want, dtype), (reach, b)
            at += m


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,G,d,dv", [(8, 2, 128, 128), (6, 3, 36, 33), (40, 20, 24, 100)])
def test_few_tokens_have_the_bits_of_many(H, G, d, dv, dtype):
    """Up to 256 workgroups one serves the heads of a key head, beyond them as many heads as it holds: the same sums."""
    from swiftllm_amd.worker.kernels import window_attn as wa
    g = torch.Generator().manual_seed(H)
    pool, sl, table, _, _ = _pool([a + n for _, a, n in PARTS], G, G, d, dv, dtype, g)
    seq, pos, _ = _spans(PARTS)
    n = seq.shape[0]
    q = torch.randn(n, H * d, generator=g).to(dtype).cuda()
    spec = wa.AttentionSpec(H, G, d, dv, d ** -0.5)
    few = wa.masked_attention(q, pool, sl, table, seq, pos, spec, None, 64)
    times = 256 // n + 1        # (the first count past 256 tokens)
    many = wa.masked_attention(q.repeat(times, 1), pool, sl, table, seq.repeat(times), pos.repeat(times), spec, None, 64)
    assert torch.equal(many.view(times, n, -1), few.expand(times, n, few.shape[1]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("H,G,d,dv,window,mixed", [(8, 2, 128, 128, 0, True), (6, 3, 18, 5, 37, True), (40, 20, 24, 100, 0, False)])
def test_sigmoid_attention(H, G, d, dv, window, mixed, dtype):
    from swiftllm_amd.worker.kernels.sigmoid_attn import sigmoid_attention
    g = torch.Generator().manual_seed(d)
    pool, sl, table, ks, vs = _pool([a + n for _, a, n in PARTS], G, G, d, dv, dtype, g)
    seq, pos, _ = _spans(PARTS)
    n = seq.shape[0]
    q = torch.randn(n, H * d, generator=g).to(dtype)
    talk = torch.eye(H) + 0.2 * torch.randn(H, H, generator=g)
    r1, r2, pb = torch.rand(H, generator=g), torch.rand(H, generator=g), torch.randn(H, generator=g) - 2
    mixer = type("Mixer", (), dict(num_q_heads=H, num_kv_heads=G, head_dim=d, value_dim=dv, window=window, scale=d ** -0.5))
    for reach in (4096, 64):
        o = sigmoid_attention(q.cuda(), pool, sl, table, seq, pos, mixer, talk.cuda() if mixed else None, r1.cuda(), r2.cuda(), pb.cuda(),
                              None, reach)
        at = 0
        for b, (_, a, m) in enumerate(PARTS):
            i, j = torch.arange(a, a + m)[:, None], torch.arange(a + m)[None]
            see = (j <= i) & ((i - j < window) if window else torch.ones(m, a + m, dtype=torch.bool))
            w = []
            for h in range(H):
                s = q[at:at + m, h * d:(h + 1) * d].double() @ ks[b][:, h // (H // G)].T * d ** -0.5
                s = s - float(r1[h]) * torch.log1p(float(r2[h]) * (i - j).clamp(min=0)) + float(pb[h])
                w.append(torch.sigmoid(s) * see)
            w = torch.stack(w)
            w = torch.einsum("hg,gij->hij", talk.double(), w) if mixed else w
            want = torch.stack([w[h] @ vs[b][:, h // (H // G)] for h in range(H)], 1).reshape(m, -1)
            # (nothing is normalised: errors of the weights add up over the keys)
            size = float((w.abs().sum(-1)).max()) * 4
            eps = 2.0 ** -20 if dtype == torch.float32 else 2.0 ** -20 + 2.0 ** -11 / size * max(1.0, float(want.abs().max()))
            assert (o[at:at + m].double().cpu() - want).abs().max() <= 1.1 * eps * size, (reach, b)
            at += m


@pytest.mark.parametrize("width,ff,top", [(64, 48, 2), (37, 18, 3), (1024, 20, 2), (130, 257, 1)])
@pytest.mark.parametrize("form", ["relu2", "silu", "clamped_in"])
def test_experts_by_assignment(width, ff, top, form):
    from swiftllm_amd.worker.kernels import moe
    g = torch.Generator().manual_seed(width)
    n, experts = 5, 6
    h = torch.randn(n, width, generator=g)
    up = torch.randn(experts, ff * (1 if form == "relu2" else 2), width, generator=g) / width ** 0.5
    down = torch.randn(experts, width, ff, generator=g) / ff ** 0.5
    idx = torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(n)])
    wts = torch.rand(n, top, generator=g) + 0.1
    args = (h.cuda(), idx.to(torch.int32).cuda(), wts.cuda(), up.cuda(), down.cuda())
    if form == "relu2":
        got = moe.moe_experts_relu2(*args)
    else:
        got = moe.moe_experts(*args, 1.5, moe.ACT_SILU if form == "silu" else moe.ACT_CLAMPED, weigh_inputs=form == "clamped_in")
    want = torch.zeros(n, width, dtype=torch.float64)
    for j in range(top):
        z = torch.einsum("tk,tfk->tf", h.double() * (wts[:, j:j + 1] if form == "clamped_in" else 1.0), up.double()[idx[:, j]])
        if form == "relu2":
            y = torch.relu(z) ** 2
        else:
            a, u = z[:, :ff], z[:, ff:]
            y = a * torch.sigmoid(a) * u if form == "silu" else a.clamp(max=1.5) * torch.sigmoid(1.702 * a.clamp(max=1.5)) * (u.clamp(-1.5, 1.5) + 1)
        want += (1.0 if form == "clamped_in" else wts[:, j:j + 1].double()) * torch.einsum("tf,twf->tw", y, down.double()[idx[:, j]])
    # two fp32 sums of up to 1024 terms of order one, one behind the other
    assert (got.double().cpu() - want).abs().max() <= 2.0 ** -17 * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("H,G,GV,d,dv,kind", [(4, 4, 2, 128, 128, "slopes"), (4, 2, 2, 128, 128, "gate"), (8, 2, 2, 128, 128, "rel"), (8, 1, 1, 128, 128, "chunk"),
                                              (3, 3, 3, 64, 64, "rel"), (6, 3, 3, 64, 64, "window"), (4, 1, 1, 64, 64, "sink"), (16, 2, 1, 64, 64, "cap"),
                                              (8, 8, 4, 64, 128, "window"), (8, 4, 2, 64, 128, "cap"), (8, 2, 1, 64, 128, "gate"), (8, 1, 1, 64, 128, "sink"),
                                              (3, 1, 1, 128, 128, "odd")])
def test_heads_of_a_key_head_in_fp32(H, G, GV, d, dv, kind):
    """The kernel that takes the heads of one key head (1, 2, 4 or 8 of them; three stay with the other), in one and in many key shares;
    what stands in a sequence's last page behind its keys does not count, whatever it is."""
    from swiftllm_amd.worker.kernels import window_attn as wa
    g = torch.Generator().manual_seed(H * d + dv)
    lens = [a + n for _, a, n in PARTS]
    pool, sl, table, ks, vs = _pool(lens, G, GV, d, dv, torch.float32, g)
    for i, n in enumerate(lens):
        if n % 16:
            blk = int(table[i + 1, n // 16])
            pool[blk, sl.k_offset:sl.k_offset + 16 * G * d].view(G, 16, d)[:, n % 16:] = float("nan")
            pool[blk, sl.v_offset:sl.v_offset + 16 * GV * dv].view(GV, dv, 16)[:, :, n % 16:] = float("nan")
    seq, pos, _ = _spans(PARTS)
    n = seq.shape[0]
    wide = torch.randn(n, H * d + 8, generator=g)
    q = wide[:, 4:4 + H * d]
    rel = torch.randn(H, 90, generator=g) if kind == "rel" else None
    out_dim = dv - 5 if kind in ("gate", "slopes") else dv
    gate = torch.randn(n, H * out_dim, generator=g) if kind == "gate" else None
    spec = wa.AttentionSpec(H, G, d, dv, d ** -0.5, window={"window": 70, "chunk": 100}.get(kind, 0), num_v_heads=GV, softcap=1.5 if kind == "cap" else 0.0,
                            mask_kind=wa.MASK_CHUNK if kind == "chunk" else wa.MASK_WINDOW, out_f32=kind == "cap", out_dim=out_dim,
                            sink=torch.randn(H, generator=g).cuda() if kind == "sink" else None,
                            slopes=(torch.rand(H, generator=g) * 0.1).cuda() if kind == "slopes" else None)
    for reach in (4096, 64):        # (sixteen key shares; one)
        if kind == "rel":
            mixer = type("Mixer", (), dict(num_q_heads=H, num_kv_heads=G, head_dim=d, value_dim=dv, window=0, scale=d ** -0.5, softcap=0.0,
                                           q_size=H * d, k_size=0, v_size=0))
            o = wa.window_attention(q.cuda().contiguous(), None, pool, sl, table, seq, pos, mixer, None, reach, rel=rel.cuda())
        else:
            o = wa.masked_attention(wide.cuda()[:, 4:4 + H * d], pool, sl, table, seq, pos, spec, None, reach, gate=gate.cuda() if gate is not None else None)
        at = 0
        for b, (_, a, m) in enumerate(PARTS):
            want = _want(q[at:at + m].double().reshape(m, H, d), ks[b], vs[b], a, spec, rel.double() if rel is not None else None,
                         gate[at:at + m].double() if gate is not None else None)
            assert (o[at:at + m].double().cpu() - want).abs().max() <= _bound(want, torch.float32), (reach, b)
            at += m


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dv,cut,extra,kind", [(64, 0, 0, "sink"), (64, 5, 3, "gate"), (128, 0, 4, "gate"), (128, 2, 0, "f32"), (256, 0, 8, "sink"), (256, 1, 1, "f32"),
                                               (100, 0, 0, "sink")])
def test_sums_of_key_shares(dv, cut, extra, kind, dtype):
    """Every number of key shares against float64: there is a token that sees as many pages (all its shares hold keys), and for most tokens some are
    empty; rows of 64, 128 and 256 columns, and others; columns that do not count, results in a column slice; the per-token entry and, where it
    serves, the tiles'."""
    from swiftllm_amd import _hip
    from swiftllm_amd.worker.kernels import window_attn as wa
    g = torch.Generator().manual_seed(dv + extra)
    H, G, d = 4, 2, 64
    parts = PARTS + [(6, 16 * s - 5, 1) for s in range(1, 65)]
    pool, sl, table, ks, vs = _pool([a + n for _, a, n in PARTS] + [1024], G, G, d, dv, dtype, g)
    seq, pos, (row0, cnt) = _spans(parts)
    n, out_dim = seq.shape[0], dv - cut
    q = torch.randn(n, H * d, generator=g).to(dtype)
    sink = torch.randn(H, generator=g).cuda() if kind == "sink" else None
    gate = torch.randn(n, H * out_dim + extra, generator=g).to(dtype) if kind == "gate" else None
    spec = wa.AttentionSpec(H, G, d, dv, d ** -0.5, sink=sink, out_dim=out_dim)
    rows = torch.cumsum(torch.tensor([0] + [m for _, _, m in parts]), 0).tolist()
    want = torch.cat([_want(q[r:r + m].double().view(m, H, d), ks[b - 1], vs[b - 1], a, spec, None, gate[r:r + m, :H * out_dim].double() if gate is not None else None)
                      for (b, a, m), r in zip(parts, rows)])
    # sums of some hundred fp32 terms, the tiles' weights in two 16-bit terms (2^-17 of values of up to four); a 16-bit result's own rounding.
    # (a share of 64 holds a sixty-fourth of the weights: without it a result moves by some 2^-8)
    bound = 1.1 * (2.0 ** -18 * max(1.0, float(want.abs().max())) if dtype == torch.float32 else 2.0 ** -15 + (0 if kind == "f32" else 2.0 ** -8) * want.abs())
    q, gate, at, size = q.cuda(), gate.cuda() if gate is not None else None, pool.data_ptr(), pool.element_size()
    wide = gate is None and out_dim % 4 == 0 and (H * out_dim + extra) % 4      # (the tiles' stores of four elements)
    tiled = dtype != torch.float32 and not wide and bool(_hip.load().swl_masked_attn_tiles_supported(H, G, G, d, dv, _hip.dtype_code(dtype)))
    for shares in range(1, 65):
        for entry in ("tokens", "tiles")[:1 + tiled]:
            out = torch.full((n, H * out_dim + extra), 7.0, dtype=torch.float32 if kind == "f32" else dtype, device="cuda")
            scratch = torch.full((shares * n * H * (dv + 2),), float("nan"), device="cuda")
            head = (_hip.ptr(out), _hip.ptr(q), at + sl.k_offset * size, at + sl.v_offset * size, _hip.ptr(table), _hip.ptr(seq), _hip.ptr(pos))
            tail = (out_dim, out.stride(0), _hip.ptr(gate), gate.stride(0) if gate is not None else 0)
            f32 = 1 if kind == "f32" else 0
            if entry == "tokens":
                _hip.call("swl_masked_attn_shares", *head, 0, 0, 0, n, H, G, d, dv, H * d, 0, d ** -0.5, 0.0, table.shape[1], pool.shape[1], 0,
                          _hip.ptr(sink), G, f32, 0, *tail, shares, _hip.ptr(scratch), _hip.dtype_code3(dtype), _hip.stream())
            else:
                _hip.call("swl_masked_attn_tiles", *head, _hip.ptr(row0), _hip.ptr(cnt), 0, 0, 0, row0.shape[0], H, G, d, dv, H * d, 0, d ** -0.5, 0.0,
                          table.shape[1], pool.shape[1], shares, _hip.ptr(scratch), n, 0, _hip.ptr(sink), G, f32, 4, 0, *tail, _hip.dtype_code(dtype),
                          _hip.stream())
            assert bool((out[:, H * out_dim:] == 7.0).all())
            err = (out[:, :H * out_dim].double().cpu() - want).abs()
            assert bool((err <= bound).all()), (shares, entry, float(err.max()))
