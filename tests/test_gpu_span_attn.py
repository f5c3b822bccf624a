"""The prompt form of the paged attention (csrc/span_attn.hip) against the same attention in float64: edges of the 32-token spans and
32-key stages, every kind of row grouping (query heads a key head), masks, bias, slopes, cap, sink, gate, narrow outputs, key shares."""
import math
import random

import pytest
import torch

pytestmark = pytest.mark.gpu


def _pool(lens, G, GV, d, dv, dtype, g):
    """-> (pool, slice, block table, keys and values per sequence): pages in shuffled blocks, offsets inside a block not zero."""
    from swiftllm_amd.worker.kernels.window_attn import PoolSlice
    blocks = [-(-n // 16) for n in lens]
    order = torch.randperm(sum(blocks) + 3, generator=g)
    off = 64
    pool = torch.zeros((sum(blocks) + 3, off + 16 * (G * d + GV * dv) + 8), dtype=dtype)
    table = torch.zeros((len(lens) + 1, max(blocks) + 2), dtype=torch.int32)
    ks, vs, at = [], [], 0
    for i, n in enumerate(lens):
        k, v = torch.randn(n, G, d, generator=g).to(dtype), torch.randn(n, GV, dv, generator=g).to(dtype)
        ks.append(k.double())
        vs.append(v.double())
        for b in range(blocks[i]):
            blk, rows = int(order[at]), slice(16 * b, min(16 * b + 16, n))
            at += 1
            table[i + 1, b] = blk
            page_k, page_v = torch.zeros(16, G, d, dtype=dtype), torch.zeros(16, GV, dv, dtype=dtype)
            page_k[:k[rows].shape[0]], page_v[:k[rows].shape[0]] = k[rows], v[rows]
            pool[blk, off:off + 16 * G * d] = page_k.transpose(0, 1).reshape(-1)
            pool[blk, off + 16 * G * d:off + 16 * (G * d + GV * dv)] = page_v.permute(1, 2, 0).reshape(-1)
    return pool.cuda(), PoolSlice(off, off + 16 * G * d), table.cuda(), ks, vs


def _want(q, k, v, start, spec, rel, gate):
    """q [n, H, d] at positions start .. of a sequence whose keys are k [N, G, d]; float64."""
    n, H, _ = q.shape
    G, GV = k.shape[1], v.shape[1]
    pos, key = torch.arange(start, start + n)[:, None], torch.arange(k.shape[0])[None]
    see = key <= pos
    if spec.window and spec.mask_kind == 0:
        see &= pos - key < spec.window
    elif spec.window:
        see &= pos // spec.window == key // spec.window
    dist = (pos - key).clamp(min=0)
    out = []
    for h in range(H):
        s = q[:, h] @ k[:, h // (H // G)].T * spec.scale
        if spec.softcap:
            s = spec.softcap * torch.tanh(s / spec.softcap)
        if rel is not None:
            s = s + rel[h][dist.clamp(max=rel.shape[1] - 1)]
        if spec.slopes is not None:
            s = s - float(spec.slopes[h]) * dist
        s = s.masked_fill(~see, -math.inf)
        if spec.sink is not None:
            s = torch.cat((s, torch.full((n, 1), float(spec.sink[h]), dtype=s.dtype)), 1)
        p = torch.softmax(s, 1)[:, :k.shape[0]]
        out.append(p @ v[:, h // (H // G) % GV])
    o = torch.stack(out, 1)[:, :, :spec.out_dim].reshape(n, -1)
    return o * torch.sigmoid(gate) if gate is not None else o


def _spans(parts, dtype=torch.int32):
    """parts: (table row, start, tokens) of every portion -> (tok_seq, tok_pos, StepTiles) on the device."""
    from swiftllm_amd.worker.kernels.window_attn import StepTiles
    seq = torch.cat([torch.full((n,), i) for i, _, n in parts])
    pos = torch.cat([torch.arange(a, a + n) for _, a, n in parts])
    start = torch.cat([torch.full((n,), a) for _, a, n in parts])

    def runs(size):
        row0, cnt, at = [], [], 0
        for _, _, n in parts:
            row0 += range(at, at + n, size)
            cnt += [min(size, n - r) for r in range(0, n, size)]
            at += n
        return torch.tensor(row0, dtype=dtype).cuda(), torch.tensor(cnt, dtype=dtype).cuda()
    tiles = StepTiles(*runs(16), (*runs(32), start.to(dtype).cuda()), max(a + n for _, a, n in parts))
    return seq.to(dtype).cuda(), pos.to(dtype).cuda(), tiles


CASES = [       # H, G, GV, d, dv, features
    (8, 2, 2, 128, 128, {}),
    (8, 2, 2, 128, 128, dict(rel=True)),
    (4, 4, 4, 64, 64, dict(rel=True, window=37)),
    (6, 2, 2, 128, 64, dict(softcap=9.0, window=50)),
    (8, 4, 2, 64, 128, dict(window=48, mask_kind=1, out_f32=True)),
    (10, 2, 2, 128, 128, dict(slopes=True, window=40, mask_kind=1)),
    (16, 1, 1, 192, 128, dict(sink=True, window=33)),
    (5, 5, 5, 128, 128, dict(gate=True, out_dim=100)),
    (4, 2, 2, 64, 128, dict(out_dim=97)),
    (8, 1, 1, 576, 512, dict(window=70)),
    (40, 1, 1, 320, 256, dict(sink=True)),
    (3, 1, 1, 576, 512, {}),
    (8, 2, 2, 64, 64, dict(rel=True)),          # (a wave's 32 rows: 16 queries of two heads)
    (6, 2, 2, 64, 128, dict(rel=True, window=45, softcap=7.0)),
    (5, 1, 1, 128, 64, dict(sink=True, slopes=True)),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("parts", [[(1, 0, 1), (2, 0, 200), (3, 0, 33)], [(1, 96, 31), (2, 0, 64), (3, 250, 1), (4, 15, 130)]])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_span_attention(case, parts, dtype):
    from swiftllm_amd.worker.kernels import window_attn
    from swiftllm_amd.worker.kernels.window_attn import AttentionSpec
    H, G, GV, d, dv, f = CASES[case]
    g = torch.Generator().manual_seed(case)
    pool, sl, table, ks, vs = _pool([a + n for _, a, n in parts], G, GV, d, dv, dtype, g)
    seq, pos, tiles = _spans(parts)
    n, out_dim = seq.shape[0], f.get("out_dim", dv)
    cols = H * out_dim
    q = torch.randn(n, H * d + 8, generator=g).to(dtype)
    rel = torch.randn(H, 90, generator=g) if f.get("rel") else None
    gate = torch.randn(n, cols + 4, generator=g).to(dtype) if f.get("gate") else None
    spec = AttentionSpec(H, G, d, dv, d ** -0.5, window=f.get("window", 0), mask_kind=f.get("mask_kind", 0), num_v_heads=GV,
                         softcap=f.get("softcap", 0.0), sink=torch.randn(H, generator=g).cuda() if f.get("sink") else None,
                         out_f32=f.get("out_f32", False), slopes=(torch.rand(H, generator=g) * 0.1).cuda() if f.get("slopes") else None,
                         out_dim=out_dim)
    esize = pool.element_size()
    for splits in ("rule", "one"):
        rows = torch.full((n, (cols + 7) // 4 * 4), 7.0, dtype=torch.float32 if spec.out_f32 else dtype, device="cuda")
        longest = tiles.longest
        if splits == "one":
            tiles.longest = 0       # (no key shares)
        qd = q.cuda()
        assert window_attn._span_launch(qd, rows, pool.data_ptr() + sl.k_offset * esize, pool.data_ptr() + sl.v_offset * esize, pool,
                                        table, seq, pos, tiles, H, G, GV, d, dv, spec.window, spec.mask_kind, spec.scale,
                                        spec.softcap, rel=rel.cuda() if rel is not None else None, sink=spec.sink, slopes=spec.slopes,
                                        out_f32=spec.out_f32, out_dim=out_dim, gate=gate.cuda()[:, :cols] if gate is not None else None)
        tiles.longest = longest
        got, at = rows.double().cpu(), 0
        assert bool((got[:, cols:] == 7.0).all())
        for i, a, m in parts:
            qi = q[at:at + m, :H * d].double().view(m, H, d)
            want = _want(qi, ks[parts.index((i, a, m))], vs[parts.index((i, a, m))], a, spec, rel.double() if rel is not None else None,
                         gate[at:at + m, :cols].double() if gate is not None else None)
            # the weights keep 16 bits or more in two terms, the sums are fp32: what is left is one rounding of the result, of a row
            # that is a convex combination of values of order one (fp32 results: the weights' 2^-16)
            eps = 2.0 ** -15 if spec.out_f32 else 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
            err = (got[at:at + m, :cols] - want).abs().max()
            assert err <= 1.1 * eps * max(1.0, float(want.abs().max())), (splits, i, float(err))
            at += m


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shares", [2, 3, 8, 40])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_key_shares(case, shares, dtype, monkeypatch):
    """The same with the pages shared out, also over more workgroups than a row sees pages: windows, chunks and sinks whose shares hold no
    visible key of a row, or none at all. (No element of the scratch counts that no share has written.)"""
    from swiftllm_amd.worker.kernels import window_attn
    used = []

    def forced(device, splits, floats):
        used.append(shares)
        return shares, torch.full((shares * floats,), float("nan"), device=device)
    monkeypatch.setattr(window_attn, "share_scratch", forced)
    test_span_attention(case, [(1, 96, 31), (2, 0, 64), (3, 250, 1), (4, 15, 130)], dtype)
    assert used == [shares, shares]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shares", [1, 3])
@pytest.mark.parametrize("case", [i for i, c in enumerate(CASES) if c[3] + c[4] <= 320])
def test_steps_of_many_workgroups(case, shares, dtype, monkeypatch):
    """The same at more than 640 workgroups of 64 rows, where rows of up to 320 elements take the form of one wave a row group (128 rows):
    portions of 1 to 70 tokens, with and without keys before them."""
    from swiftllm_amd.worker.kernels import window_attn
    H, G = CASES[case][:2]
    queries, pick, parts, spans = 64 >> (H // G - 1).bit_length(), random.Random(case), [], 0
    while spans * G * 32 <= 640 * queries:
        n = pick.choice([1, 15, 31, 32, 33, 47, 64, 70])
        parts.append((len(parts) + 1, pick.choice([0, 0, 16, 37, 100]), n))
        spans += -(-n // 32)
    if shares > 1:
        monkeypatch.setattr(window_attn, "share_scratch", lambda device, splits, floats: (
            shares, torch.full((shares * floats,), float("nan"), device=device)))
    test_span_attention(case, parts, dtype)


@pytest.mark.parametrize("case", [i for i, c in enumerate(CASES) if c[3] + c[4] <= 320])
def test_portions_of_many_pages(case):
    """More pages than one load of block ids holds (64), from the first page on and behind cached tokens."""
    test_span_attention(case, [(1, 0, 1300), (2, 1037, 40)], torch.bfloat16)


@pytest.mark.parametrize("scale", [1e-38, 1e-30, 1e-19, -0.05, 0.0])
def test_scales_of_any_size(scale):
    """Masked keys weigh nothing whatever the scale: next to none at all, the visible values' mean, and negative ones."""
    from swiftllm_amd.worker.kernels import window_attn
    from swiftllm_amd.worker.kernels.window_attn import AttentionSpec
    parts, g = [(1, 0, 40), (2, 21, 77)], torch.Generator().manual_seed(2)
    pool, sl, table, ks, vs = _pool([a + n for _, a, n in parts], 2, 2, 64, 64, torch.bfloat16, g)
    seq, pos, tiles = _spans(parts)
    q = torch.randn(seq.shape[0], 4 * 64, generator=g).to(torch.bfloat16)
    spec = AttentionSpec(4, 2, 64, 64, scale, window=50)
    out = window_attn.masked_attention(q.cuda(), pool, sl, table, seq, pos, spec, tiles)
    at = 0
    for k, v, (_, a, n) in zip(ks, vs, parts):
        want = _want(q[at:at + n].double().view(n, 4, 64), k, v, a, spec, None, None)
        assert (out[at:at + n].double().cpu() - want).abs().max() <= 1.1 * 2.0 ** -8 * max(1.0, float(want.abs().max()))
        at += n


@pytest.mark.parametrize("H,G,d,dv,window", [(8, 2, 128, 128, 0), (4, 4, 64, 64, 100), (6, 2, 192, 128, 0), (8, 1, 576, 512, 300),
                                             (2, 1, 320, 256, 0), (3, 1, 64, 128, 0)])
def test_spans_in_any_order(H, G, d, dv, window):
    """Steps of more than 64 spans take them up in the plan's order: the same bits as last to first (which the oracle checks above), for
    fewer workgroups than CUs, up to two a CU (taken from both ends) and more, whole and broken runs of spans and all key heads."""
    from swiftllm_amd.worker.batch_plan import StepEntry, plan_step
    from swiftllm_amd.worker.kernels import window_attn
    g = torch.Generator().manual_seed(H)
    for parts in ([(1, 0, 1500), (2, 33, 700), (3, 77, 1)], [(1, 0, 2000), (2, 0, 1999), (3, 5, 1), (4, 100, 1234)],
                  [(i, 16 * i, 1700 - 100 * i) for i in range(8)]):
        pool, sl, table, _, _ = _pool([a + n for _, a, n in parts], G, G, d, dv, torch.bfloat16, g)
        seq, pos, tiles = _spans(parts)
        order = plan_step([StepEntry(i, [1] * n, a) for i, a, n in parts]).span_order()
        assert sorted(order) == list(range(tiles.spans[0].shape[0]))
        q = torch.randn(seq.shape[0], H * d, generator=g).to(torch.bfloat16).cuda()
        tiles.longest = 0           # (no key shares)
        out = []
        for tiles.span_order in (None, torch.from_numpy(order).cuda()):
            out.append(torch.full((seq.shape[0], H * dv), 7.0, dtype=torch.bfloat16, device="cuda"))
            assert window_attn._span_launch(q, out[-1], pool.data_ptr() + sl.k_offset * 2, pool.data_ptr() + sl.v_offset * 2, pool, table, seq,
                                            pos, tiles, H, G, G, d, dv, window, 0, d ** -0.5, 0.0)
        assert torch.equal(out[0], out[1]) and not bool((out[0] == 7.0).all(1).any())
