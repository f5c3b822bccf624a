"""The linear recurrence of heads with 64 or 128 key channels, 64 columns a workgroup (csrc/linear_scan.hip), against float64: columns that fill no
workgroup and no wave, portions around a tile's and a segment's end, more portions than a wave counts at once, carried states, operands that
the wide kernels do not take."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def oracle(q, k, v, decay, s, u=None):
    """One portion: [n, H, d], [n, H, d], [n, H, dv], [n, H, d], state [H, d, dv] (changed) -> [n, H, dv]; float64."""
    out = torch.empty_like(v)
    for t in range(q.shape[0]):
        kv = k[t].unsqueeze(-1) * v[t].unsqueeze(-2)
        if u is None:
            s.mul_(decay[t].unsqueeze(-1)).add_(kv)
            out[t] = (q[t].unsqueeze(-2) @ s).squeeze(-2)
        else:
            out[t] = (q[t].unsqueeze(-2) @ (s + u.unsqueeze(-1) * kv)).squeeze(-2)
            s.mul_(decay[t].unsqueeze(-1)).add_(kv)
    return out


LONG = [401, 1, 16, 384, 17]
MANY = [1] * 70 + [390, 2, 375]


@pytest.mark.parametrize("lens,H,G,d,dv,bonus,scalar,aligned", [
    (LONG, 2, 1, 128, 72, False, False, True), (LONG, 3, 3, 64, 8, True, False, True), (MANY, 1, 1, 64, 136, False, True, True), (MANY, 2, 2, 128, 64, True, False, True),
    (LONG, 2, 2, 128, 72, False, False, False), (LONG, 1, 1, 128, 12, False, True, True), ([1, 15, 33, 16], 2, 1, 128, 128, False, False, True)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_wide_scan(lens, H, G, d, dv, bonus, scalar, aligned, dtype):
    from swiftllm_amd.worker.kernels import linear_scan
    from swiftllm_amd.worker.kernels.rms_stream import StateRef
    g = torch.Generator().manual_seed(d + dv + len(lens))
    n, off = sum(lens), 8
    rows, counts, tile0, seq_row0, pos, slots = [], [], [], [], [], []
    at = 0
    for s, c in enumerate(lens):
        seq_row0.append(at)
        tile0.append(len(rows))
        for o in range(0, c, 16):
            rows.append(at + o)
            counts.append(min(16, c - o))
        first = 7 * (s % 2)         # (every other sequence has a state)
        pos += range(first, first + c)
        slots += [2 * (len(lens) - 1 - s)] * c
        at += c
    state = torch.randn(len(lens), H, d, dv, generator=g)
    pool = torch.full((len(lens), off + H * d * dv), float("nan"))
    for s in range(len(lens)):
        if s % 2:
            pool[len(lens) - 1 - s, off:] = state[s].flatten()
    pool = pool.cuda()
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")      # noqa: E731
    st = StateRef(pool, ints(pos), None, ints(slots), None, ints(seq_row0), ints(lens), (ints(rows), ints(counts), ints(tile0)), max(lens))
    wide = torch.randn(n, 2 * G * d + H * dv + 1, generator=g).to(dtype)
    if not aligned:
        wide = wide[:, 1:]
    elif wide.shape[1] % 8:
        wide = torch.cat([wide, wide.new_zeros(n, -wide.shape[1] % 8)], dim=1)
    q, k, v = (wide[:, a:b] for a, b in ((0, G * d), (G * d, 2 * G * d), (2 * G * d, 2 * G * d + H * dv)))
    decay = torch.rand(n, H if scalar else H * d, generator=g) ** 0.02
    decay[torch.rand(decay.shape, generator=g) < 0.002] = 0.0
    scale = torch.rand(n, H, generator=g) if scalar else None
    skip = torch.randn(H, generator=g) if scalar else None
    u = torch.randn(H, d, generator=g) if bonus else None
    dev = wide.cuda() if aligned else torch.cat([wide.new_zeros(n, 1), wide], dim=1).cuda()[:, 1:]
    part = lambda a, b: dev[:, a:b]     # noqa: E731
    y = linear_scan.linear_recurrence(part(0, G * d), part(G * d, 2 * G * d), part(2 * G * d, 2 * G * d + H * dv), decay.cuda(), st, off, H, d, dv, q_scale=0.3,
                                      bonus=u.cuda() if bonus else None, k_scale=scale.cuda() if scalar else None,
                                      dskip=skip.cuda() if scalar else None, num_qk_heads=G).cpu().double()
    got_state = pool.cpu()[:, off:].double().view(len(lens), H, d, dv)
    heads = lambda x: x.double().view(n, G, d).repeat_interleave(H // G, dim=1)     # noqa: E731
    qq, kk, vv = 0.3 * heads(q), heads(k), v.double().reshape(n, H, dv)
    if scalar:
        kk = kk * scale.double().unsqueeze(-1)
    dd = decay.double().view(n, H, -1).expand(n, H, d)
    at = 0
    for s, c in enumerate(lens):
        S = state[s].double() if s % 2 else torch.zeros(H, d, dv, dtype=torch.float64)
        want = oracle(qq[at:at + c], kk[at:at + c], vv[at:at + c], dd[at:at + c], S, u.double() if bonus else None)
        if scalar:
            want = want + skip.double().view(1, H, 1) * vv[at:at + c]
        # fp32 products and sums: the bound of the walk without segments
        assert (y[at:at + c] - want.reshape(c, -1)).abs().max() < 3e-5 * max(1.0, float(want.abs().max())), (s, c)
        assert (got_state[len(lens) - 1 - s] - S).abs().max() < 3e-5 * max(1.0, float(S.abs().max())), (s, c)
        at += c


@pytest.mark.parametrize("shift,dv,want", [(0, 64, (21, 3)), (1, 64, (7, 9)), (0, 60, (7, 9))])
def test_segments_are_those_of_the_walk_that_runs(shift, dv, want, monkeypatch):
    """Values that lie on no 16 bytes, or are no whole pieces of 16, take the walk of 16 columns a workgroup: portions are cut as its workgroups need it."""
    from swiftllm_amd.worker.kernels import linear_scan
    from swiftllm_amd.worker.kernels.rms_stream import StateRef
    n, H, d = 1000, 4, 128
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")      # noqa: E731
    starts = range(0, n, 16)
    st = StateRef(torch.zeros(1, H * d * dv, device="cuda"), ints(range(n)), None, ints([0] * n), None, ints([0]), ints([n]),
                  (ints(starts), ints([min(16, n - s) for s in starts]), ints([0])), n)
    cut, got = linear_scan.scan_segments, []

    def keep(*a):
        got.append(cut(*a))
        return got[-1]
    monkeypatch.setattr(linear_scan, "scan_segments", keep)
    v = torch.zeros(n, H * dv + 8, dtype=torch.bfloat16, device="cuda")[:, shift:shift + H * dv]
    q = torch.zeros(n, H * d, dtype=torch.bfloat16, device="cuda")
    linear_scan.linear_recurrence(q, q, v, torch.ones(n, H, device="cuda"), st, 0, H, d, dv)
    assert got[0][:2] == want


@pytest.mark.parametrize("lens", [[401, 1, 16, 384, 17], [33, 20, 50]])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_value_that_is_no_number_stays_in_its_column(lens, dtype):
    """NaN and infinity among the values of one sequence, infinities in another's keys: other sequences, heads, columns and the tiles before have the bits that
    they have without."""
    from swiftllm_amd.worker.kernels import linear_scan
    from swiftllm_amd.worker.kernels.rms_stream import StateRef
    g = torch.Generator().manual_seed(1)
    n, H, d, dv = sum(lens), 2, 64, 72
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")      # noqa: E731
    rows, counts, tile0, seq_row0, at = [], [], [], [], 0
    for c in lens:
        seq_row0.append(at)
        tile0.append(len(rows))
        for o in range(0, c, 16):
            rows.append(at + o)
            counts.append(min(16, c - o))
        at += c
    q, k, v = (torch.randn(n, H * s, generator=g).to(dtype) for s in (d, d, dv))
    decay = torch.rand(n, H * d, generator=g) ** 0.02
    bad_v, bad_k = v.clone(), k.clone()
    bad_v[20, dv + 70] = float("nan")          # the first sequence, second head, column 70, second tile
    last = seq_row0[-1] + 16
    bad_v[last, 3], bad_k[seq_row0[1], 5] = float("inf"), float("inf")
    results = []
    for vv, kk in ((v, k), (bad_v, bad_k)):
        pool = torch.zeros(len(lens), H * d * dv, device="cuda")
        st = StateRef(pool, ints([p for c in lens for p in range(c)]), None, ints([2 * s for s, c in enumerate(lens) for _ in range(c)]), None, ints(seq_row0), ints(lens),
                      (ints(rows), ints(counts), ints(tile0)), max(lens))
        y = linear_scan.linear_recurrence(q.cuda(), kk.cuda(), vv.cuda(), decay.cuda(), st, 0, H, d, dv)
        results.append((y.cpu().view(n, H, dv), pool.cpu().view(len(lens), H, d, dv)))
    (y, s), (bad_y, bad_s) = results
    same, states = torch.ones_like(y, dtype=torch.bool), torch.ones_like(s, dtype=torch.bool)
    same[16:lens[0], 1, 70], states[0, 1, :, 70] = False, False
    same[last:, 0, 3], states[-1, 0, :, 3] = False, False
    same[seq_row0[1]:seq_row0[1] + lens[1], 0], states[1, 0] = False, False
    assert torch.equal(bad_y[same], y[same]) and torch.equal(bad_s[states], s[states])
    assert not bool(bad_y[20:lens[0], 1, 70].isfinite().any()) and not bool(bad_s[0, 1, :, 70].isfinite().any())
    assert not bool(bad_y[last:, 0, 3].isfinite().any()) and not bool(bad_s[-1, 0, :, 3].isfinite().any())
    assert not bool(bad_y[seq_row0[1]:seq_row0[1] + lens[1], 0].isfinite().any())
