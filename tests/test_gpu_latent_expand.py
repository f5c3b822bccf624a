"""Latent attention on expanded pages (csrc/latent_expand.hip, kernels/latent.py): the pages against float64 products of the cached rows, and the
attention of whole steps (portions with and without earlier tokens, beside decoded ones) against the folded form's oracle."""
import math
from types import SimpleNamespace

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
UNIT = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}      # half a unit in the last place, relative


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,d,dr,e,r,pad,pages", [(2, 128, 64, 128, 512, 0, 21), (3, 64, 64, 64, 64, 0, 8), (1, 136, 8, 200, 128, 8, 1),
                                                  (2, 8, 56, 128, 192, 40, 9), (5, 256, 64, 256, 64, 0, 17)])
def test_pages(H, d, dr, e, r, pad, pages, dtype):
    from swiftllm_amd import _hip
    g = torch.Generator().manual_seed(pages)
    k_dim, off = r + dr + pad, 24
    blocks = pages + 5
    pool = torch.randn(blocks, off + 16 * k_dim + 16, generator=g).to(dtype)
    uk, uv = (torch.randn(H, n, r, generator=g).div(math.sqrt(r)).to(dtype) for n in (d, e))
    table = torch.randperm(blocks, generator=g)[:2 * ((pages + 1) // 2)].view(2, -1).int()
    row = torch.tensor([i % 2 for i in range(pages)]).int()
    no = torch.tensor([i // 2 for i in range(pages)]).int()
    dst = (torch.randperm(pages + 2, generator=g)[:pages]).int()
    page = 16 * H * (d + dr + e)
    out = torch.full((pages + 2, page), 3.0, dtype=dtype, device="cuda")
    dev = [t.cuda() for t in (pool, uk, uv, table, row, no, dst)]
    _hip.call("swl_latent_expand", out.data_ptr(), dev[0].data_ptr() + off * 2, *[t.data_ptr() for t in dev[1:]], pages, H, d, e, dr, r, k_dim,
              table.shape[1], pool.shape[1], _hip.dtype_code(dtype), _hip.stream())
    out = out.cpu()
    for i in range(pages):
        c = pool[int(table[int(row[i]), int(no[i])]), off:off + 16 * k_dim].view(16, k_dim)
        lat = c[:, :r].double()
        got_k = out[int(dst[i]), :16 * H * (d + dr)].view(H, 16, d + dr)
        got_v = out[int(dst[i]), 16 * H * (d + dr):].view(H, e, 16)
        for got, want, mag in ((got_k[:, :, :d], torch.einsum("tr,hdr->htd", lat, uk.double()), torch.einsum("tr,hdr->htd", lat.abs(), uk.double().abs())),
                               (got_v, torch.einsum("tr,her->het", lat, uv.double()), torch.einsum("tr,her->het", lat.abs(), uv.double().abs()))):
            # one rounding of a sum of r fp32 terms
            assert bool(((got.double() - want).abs() <= UNIT[dtype] * want.abs() + r * 2.0 ** -23 * mag + 1e-7).all())
        assert torch.equal(got_k[:, :, d:], c[None, :, r:r + dr].expand(H, 16, dr))
    untouched = [i for i in range(pages + 2) if i not in dst.tolist()]
    assert bool((out[untouched] == 3.0).all())


def _step(parts, window, max_pages=1 << 20):
    """-> (plan, device views) of portions (sequence, start, tokens)."""
    from swiftllm_amd.worker.batch_plan import LatentExpansion, StepEntry, plan_step
    plan = plan_step([StepEntry(s, [1] * n, a, ()) for s, a, n in parts])
    expanded = plan.latent_expansion(LatentExpansion(128, 64, 128, 512, window, max_pages))
    dev = {n: torch.from_numpy(np.ascontiguousarray(getattr(plan, n))).cuda() for n in plan.SEGMENTS}
    dev["portions"], dev["longest"], dev["expanded"] = (plan.target_lens_list, plan.seq_cnt), max(plan.target_lens_list), expanded
    if expanded is not None:
        dev.update({n: torch.from_numpy(np.ascontiguousarray(v)).cuda() for n, v in expanded.arrays.items()})
    return plan, dev


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("window,sink,half", [(0, True, False), (70, False, True)])
@pytest.mark.parametrize("parts,rows", [([(1, 0, 200), (2, 0, 16), (0, 0, 33)], 249), ([(2, 0, 40), (1, 130, 190), (0, 99, 1), (3, 16, 1)], 230),
                                        ([(0, 0, 128), (1, 40, 5), (2, 0, 64)], 128), ([(0, 60, 1), (1, 0, 64)], 0)])
def test_steps(parts, rows, window, sink, half, dtype):
    """Whatever rows are expanded, the results are those of 64-bit attention on the cached rows."""
    check_step(parts, rows, window, sink, half, dtype, 4, 128)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("window,sink,half,H,e", [(0, True, False, 16, 128), (70, False, True, 8, 128), (0, False, True, 20, 64), (33, True, True, 3, 272)])
@pytest.mark.parametrize("parts", [[(2, 0, 1)], [(1, 15, 1), (0, 16, 1), (3, 17, 1)], [(s, (37 * s) % 300, 1) for s in range(20)],
                                   [(s, 5 + 9 * s, 1) for s in range(33)], [(0, 4500, 1), (1, 3000, 1)], [(0, 0, 40), (1, 99, 1), (2, 250, 1)],
                                   [(s, s, 1) for s in range(70)]])
def test_single_tokens(parts, window, sink, half, H, e, dtype):
    """Steps of single tokens, and behind expanded portions (csrc/latent_decode.hip): shares with and without keys, from one page a share on,
    tokens and heads around the kernels' groups of 4 and 16, and more tokens than are folded beside the rotary."""
    check_step(parts, sum(n for _, _, n in parts if n > 1), window, sink, half, dtype, H, e)


def check_step(parts, rows, window, sink, half, dtype, H, e):
    from swiftllm_amd.worker.kernels.latent import ExpandedStep, LatentAttention
    from swiftllm_amd.worker.kernels.window_attn import AttentionSpec, PoolSlice, StepTiles
    g = torch.Generator().manual_seed(rows + window)
    d, dr, r = 128, 64, 512
    mx = SimpleNamespace(num_q_heads=H, head_dim=d, rot_dim=dr, value_dim=e, kv_rank=r, window=window,
                         rot=SimpleNamespace(dims=dr, half=half, multiplier=1.0))
    uk, uv = (torch.randn(H, n, r, generator=g).div(math.sqrt(r)).to(dtype) for n in (d, e))
    freq = 10000.0 ** (-torch.arange(0, dr, 2, dtype=torch.float64) / dr)
    w = SimpleNamespace(uk=uk.cuda(), uk_t=uk.transpose(1, 2).contiguous().cuda(), uv=uv.cuda(), uv_t=uv.transpose(1, 2).contiguous().cuda(), freq=freq.cuda(),
                        c_norm=torch.ones(r, device="cuda"))
    sinks = torch.randn(H, generator=g) if sink else None
    spec = AttentionSpec(H, 1, r + dr, r, (d + dr) ** -0.5, window=window, sink=sinks.cuda() if sink else None)
    plan, dev = _step(parts, window)
    ex = ExpandedStep.of(dev)
    assert (ex.rows if ex else 0) == rows
    # earlier tokens' rows in shuffled blocks, stale rows behind the ends
    total = sum(-(-(a + n) // 16) for _, a, n in parts) + 2
    blocks, block = torch.randperm(total, generator=g), 16 * (2 * r + dr)
    pool = torch.randn(total, block, generator=g).to(dtype)
    pool[:, 16 * (r + dr):] = pool[:, :16 * (r + dr)].view(total, 16, r + dr)[:, :, :r].transpose(1, 2).reshape(total, -1)
    table = torch.zeros(max(s for s, _, _ in parts) + 1, max(-(-(a + n) // 16) for _, a, n in parts) + 1, dtype=torch.int32)
    at = 0
    for s, a, n in parts:
        pages = -(-(a + n) // 16)
        table[s, :pages] = blocks[at:at + pages]
        at += pages
    n = plan.num_tokens
    gate_col = H * (d + dr) + r + dr
    rows_in = torch.randn(n, -(-(gate_col + H) // 8) * 8, generator=g).to(dtype)
    pool_dev, proj = pool.cuda(), rows_in.cuda()
    ctx = SimpleNamespace(pool=pool_dev, block_table=table.cuda(), tok_seq=dev["tok_seq"], tok_pos=dev["tok_pos"], tiles=StepTiles.of(dev),
                          expanded=ex)
    attend = LatentAttention(mx, w, spec, 1e-6, PoolSlice(0, 16 * (r + dr)), 8192, H * (d + dr))
    got = attend(proj, proj[:, gate_col:gate_col + H], ctx).cpu().double()
    pool = pool_dev.cpu()
    folded_rows = SimpleNamespace(**{**ctx.__dict__, "expanded": None})
    other = LatentAttention(mx, w, spec, 1e-6, PoolSlice(0, 16 * (r + dr)), 8192, H * (d + dr))
    other.decodes = False
    proj = rows_in.cuda()
    folded = other(proj, proj[:, gate_col:gate_col + H], folded_rows).cpu().double()
    row = 0
    worst, worst_folded = 0.0, 0.0
    for s, a, cnt in parts:
        cached = torch.cat([pool[int(table[s, b]), :16 * (r + dr)].view(16, r + dr) for b in range(-(-(a + cnt) // 16))])[:a + cnt].double()
        k = torch.cat((torch.einsum("tr,hdr->htd", cached[:, :r], uk.double()), cached[None, :, r:].expand(H, -1, -1)), 2)
        v = torch.einsum("tr,her->hte", cached[:, :r], uv.double())
        q = rows_in[row:row + cnt, :H * (d + dr)].view(cnt, H, d + dr).double()
        ang = torch.arange(a, a + cnt, dtype=torch.float64)[:, None] * freq
        cs, sn = torch.cos(ang)[:, None].float().double(), torch.sin(ang)[:, None].float().double()
        x, y = (q[..., d:d + dr // 2], q[..., d + dr // 2:]) if half else (q[..., d::2], q[..., d + 1::2])
        u, z = x * cs - y * sn, y * cs + x * sn
        rot = torch.cat((u, z), -1) if half else torch.stack((u, z), -1).flatten(-2)
        q = torch.cat((q[..., :d], rot.to(dtype).double()), -1)
        sc = torch.einsum("qhd,hkd->hqk", q, k) * spec.scale
        pos, key = torch.arange(a, a + cnt)[:, None], torch.arange(a + cnt)[None]
        see = (key <= pos) & ((pos - key < window) if window else torch.ones_like(key <= pos))
        sc = sc.masked_fill(~see, -math.inf)
        if sink:
            sc = torch.cat((sc, sinks.double()[:, None, None].expand(H, cnt, 1)), 2)
        results = []
        for without in (slice(0), slice(max(a - a % 16 - 16, 0), a - a % 16)):     # (a whole page's keys left out: what a result that lost them would be)
            x = sc.clone()
            x[:, :, without] = -math.inf
            o = torch.einsum("hqk,hke->qhe", torch.softmax(x, 2)[:, :, :a + cnt], v)
            results.append((o * torch.sigmoid(rows_in[row:row + cnt, gate_col:gate_col + H].double())[:, :, None]).reshape(cnt, -1))
        want, lost = results
        # a key's and a value's products are rounded once (as folded queries and latent results are): scores move by sqrt(d) of such
        # roundings of |q| |k| ~ 1, results by one of the largest |v| ~ 4, and by what the scores' weights move
        bound = 24 * UNIT[dtype]
        err = (got[row:row + cnt] - want).abs().max().item()
        # averages over many keys are small: the 2-norm of a portion's error against its result's. Rounded are the keys or the queries (scores of order
        # one move by 0.6 of a unit), the values, their sums and the result: some five times 0.6 of a unit, in squares
        size = 4 * UNIT[dtype] * want.norm()
        for name, o in (("got", got), ("folded", folded)):
            assert (o[row:row + cnt] - want).norm() <= size, (name, s, a, cnt, float((o[row:row + cnt] - want).norm() / want.norm()))
        if cnt == 1 and a >= 16 and not window:
            assert (lost - want).norm() > 2 * size
        worst += float(((got[row:row + cnt] - want) ** 2).sum())
        worst_folded += float(((folded[row:row + cnt] - want) ** 2).sum())
        assert err <= bound, (s, a, cnt, err, bound)
        row += cnt
    print(f"largest error {math.sqrt(worst):.4e}, folded {math.sqrt(worst_folded):.4e}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("window", [0, 4999])
@pytest.mark.parametrize("H,e,shares", [(16, 128, 1), (3, 64, 1), (20, 16, 1), (16, 128, 2)])
def test_shares_of_many_pages(H, e, shares, window, dtype):
    """A share whose pages are more than a wave loads the ids of at a time (64 of its every fourth one): 5000 and 9000 keys, windows that begin
    inside a page, and a sequence of few beside them."""
    from swiftllm_amd import _hip
    g = torch.Generator().manual_seed(H + shares)
    r, dr = 512, 64
    lens = [5000, 37, 9011]
    pages = [-(-n // 16) for n in lens]
    pool = torch.randn(sum(pages) + 2, 16 * (r + dr), generator=g).to(dtype)
    blocks, table = torch.randperm(sum(pages) + 2, generator=g).int(), torch.zeros(len(lens), max(pages), dtype=torch.int32)
    for s, n in enumerate(pages):
        table[s, :n] = blocks[sum(pages[:s]):sum(pages[:s]) + n]
    q = torch.randn(len(lens), H * (r + dr), generator=g).to(dtype)
    uv = torch.randn(H, e, r, generator=g).div(math.sqrt(r)).to(dtype)
    scale = (r + dr) ** -0.5
    dev = [t.cuda() for t in (q, pool, table, torch.arange(len(lens)).int(), torch.tensor(lens).int() - 1, uv)]
    scratch = torch.full((shares * len(lens) * H * (r + 2),), float("nan"), device="cuda")
    y = torch.empty(len(lens), H * e, dtype=dtype, device="cuda")
    code, stream = _hip.dtype_code(dtype), _hip.stream()
    _hip.call("swl_latent_decode", _hip.ptr(scratch), *[_hip.ptr(t) for t in dev[:5]], len(lens), H, q.shape[1], window, scale, table.shape[1], pool.shape[1],
              shares, code, stream)
    _hip.call("swl_latent_unfold", _hip.ptr(y), _hip.ptr(scratch), _hip.ptr(dev[5]), 0, 0, 0, len(lens), H, e, shares, code, stream)
    for s, n in enumerate(lens):
        c = torch.cat([pool[int(b)].view(16, r + dr) for b in table[s, :pages[s]]])[:n].double()
        sc = q[s].view(H, -1).double() @ c.T * scale
        if window:
            sc[:, :max(n - window, 0)] = -math.inf
        want = torch.einsum("hr,her->he", torch.softmax(sc, 1) @ c[:, :r], uv.double())
        err = (y[s].cpu().double().view(H, e) - want).norm(dim=1) / want.norm(dim=1)
        # the sum's and the result's rounding; a page of 16 keys of n is some sqrt(16 / n) of the result, 4 % and more
        assert float(err.max()) <= 2 * UNIT[dtype], (s, float(err.max()))


@pytest.mark.parametrize("r,dr,e,pad,dtype,held", [(512, 64, 128, 0, torch.bfloat16, "uk_t uv"), (512, 64, 128, 0, torch.float32, ""), (128, 64, 128, 0, torch.float16, "uv"),
                                                   (96, 64, 128, 0, torch.bfloat16, ""), (512, 64, 24, 0, torch.bfloat16, ""),
                                                   (512, 64, 128, 32, torch.bfloat16, "uv")])
def test_up_projections_are_held_the_way_they_are_read(r, dr, e, pad, dtype, held):
    """Beside the two of the folded form a layer keeps the matrices that its kernels read, once for all of its runs."""
    from swiftllm_amd.worker.kernels.latent import LatentAttention
    from swiftllm_amd.worker.kernels.window_attn import AttentionSpec, PoolSlice
    H, d = 4, 128
    mx = SimpleNamespace(num_q_heads=H, head_dim=d, rot_dim=dr, value_dim=e, kv_rank=r)
    uk, uv = torch.randn(H, d, r).to(dtype).cuda(), torch.randn(H, e, r).to(dtype).cuda()
    w = SimpleNamespace(uk=uk, uk_t=None, uv=None, uv_t=uv.transpose(1, 2).contiguous())
    spec = AttentionSpec(H, 1, r + dr + pad, r + pad, 0.1)
    kept = []
    for _ in range(2):
        LatentAttention(mx, w, spec, 1e-6, PoolSlice(0, 16 * (r + dr + pad)), 4096, 0)
        assert " ".join(n for n in ("uk_t", "uv") if getattr(w, n) is not None) == held
        assert w.uk_t is None or torch.equal(w.uk_t, uk.transpose(1, 2))
        assert w.uv is None or torch.equal(w.uv, uv)
        kept.append((w.uk_t, w.uv))
    assert all(a is b for a, b in zip(*kept))


def test_the_weights_of_a_layer_in_fp32_are_held_once(tmp_path):
    import rosilix_oracle as O
    from test_gpu_rosilix import make_model
    cfg = O.make_config([O.latent_mixer(heads=2, dim=128, rot_dim=64, vdim=128, kv_rank=512)])
    for dtype, held in (("float32", False), ("bfloat16", True)):
        lw = make_model(tmp_path / dtype, cfg, O.make_weights(cfg), dtype).weight.layers[0]
        assert (lw.uk_t is not None, lw.uv is not None) == (held, held)


def test_portions_past_the_scratch_limit_stay_folded():
    parts = [(0, 0, 64), (1, 0, 64), (2, 0, 64)]
    for pages, rows in ((12, 192), (11, 128), (4, 64), (3, 0)):
        ex = _step(parts, 0, pages)[1]["expanded"]
        assert (ex.rows if ex else 0) == rows
