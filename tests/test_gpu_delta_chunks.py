"""The delta rule by tiles (csrc/delta_chunks.hip) against the recurrence in float64, and beside the token-by-token walk: portions around
the 16-token tiles, states carried between steps, decays and rates at the ends of their range, keys that repeat."""
import pytest
import torch

from test_gpu_lorulix import Slots

pytestmark = pytest.mark.gpu


def _ref(slots, portions, tiles=True):
    st = slots.ref(portions)
    if tiles:
        row0, cnt, first, at = [], [], [], 0
        for _, _, n in portions:
            first.append(len(row0))
            row0 += range(at, at + n, 16)
            cnt += [min(16, n - r) for r in range(0, n, 16)]
            at += n
        st.tiles = tuple(torch.tensor(x, dtype=torch.int32, device="cuda") for x in (row0, cnt, first))
        st.longest = max(n for _, _, n in portions)
    return st


def _scan(q, k, v, beta, g, S):
    """One head in float64: q, k [n, d], v [n, dv], S [d, dv] -> (o, S)."""
    out = []
    for i in range(q.shape[0]):
        S = g[i] * S
        u = beta[i] * (v[i] - S.T @ k[i])
        S = S + k[i][:, None] * u
        out.append(S.T @ q[i])
    return torch.stack(out), S


@pytest.mark.parametrize("H,G,d,dv", [(4, 2, 128, 128), (3, 1, 64, 64), (2, 2, 128, 48), (5, 5, 64, 16), (9, 3, 64, 208)])
@pytest.mark.parametrize("kind", ["plain", "ends", "repeats"])
@pytest.mark.parametrize("steps", [[[(1, 0, 200), (2, 0, 16), (3, 0, 1)], [(2, 16, 33), (3, 1, 15), (1, 200, 64)]],
                                   [[(1, 0, 49)], [(1, 49, 63), (2, 0, 31)], [(2, 31, 17), (1, 112, 96)]]])
def test_delta_rule_by_tiles(H, G, d, dv, kind, steps):
    from swiftllm_amd.worker.kernels.delta_rule import delta_rule_scan
    gen = torch.Generator().manual_seed(H * d + dv)
    randn = lambda *s: torch.randn(*s, generator=gen)
    slots = {by: Slots([d * dv * H + 64], num_slots=3) for by in ("tiles", "tokens")}
    states = {}
    worst = {"tiles": 0.0, "tokens": 0.0}
    for step in steps:
        n = sum(c for _, _, c in step)
        k = randn(n, G, d)
        if kind == "repeats":       # long runs of one key: T far from the identity
            k = k[:1] + 0.01 * k
        q, k = [torch.nn.functional.normalize(x, dim=2) for x in (randn(n, G, d) + 0.5 * k, k)]
        q, v = q * d ** -0.5, randn(n, H, dv)
        beta, g = torch.sigmoid(2 * randn(n, H)), torch.exp(-torch.nn.functional.softplus(randn(n, H)) * 0.3)
        if kind == "ends":
            pick = torch.randint(0, 5, (n, H), generator=gen)
            beta = torch.where(pick == 0, 0.0, torch.where(pick == 1, 1.0, beta))
            g = torch.where(pick == 2, 0.0, torch.where(pick == 3, 1.0, g))
        if kind == "repeats":
            beta, g = 1 - 0.01 * beta, 1 - 0.001 * g
        gpu = [x.contiguous().view(n, -1).cuda() for x in (q, k, (q * k).sum(2), v, beta, g)]
        got, after = {}, {}
        for by in slots:
            st = _ref(slots[by], step, by == "tiles")
            o = torch.full((n, H * dv), float("nan"), device="cuda")
            delta_rule_scan(o, *gpu, st, slots[by].off[0], H, G, d, dv)
            got[by] = o.double().cpu().view(n, H, dv)
            rows = [int(st.tok_state[int(r)]) >> 1 for r in st.seq_row0]
            after[by] = [st.pool[r, slots[by].off[0]:slots[by].off[0] + H * d * dv].double().cpu().view(H, d, dv) for r in rows]
        at = 0
        for p, (s, start, c) in enumerate(step):
            for h in range(H):
                S = states[s, h] if start else torch.zeros(d, dv, dtype=torch.float64)
                want, states[s, h] = _scan(q[at:at + c, h // (H // G)].double(), k[at:at + c, h // (H // G)].double(), v[at:at + c, h].double(),
                                           beta[at:at + c, h].double(), g[at:at + c, h].double(), S)
                for by in got:
                    for a, b in ((got[by][at:at + c, h], want), (after[by][p][h], states[s, h])):
                        worst[by] = max(worst[by], float((a - b).abs().max()) / max(1.0, float(b.abs().max())))
            at += c
    print("worst error, by tiles and by tokens:", worst)
    # fp32 sums of up to 3 dim terms a tile, carried over at most 14 tiles: sqrt(3 * 128 * 14) * 2^-24 = 4.4e-6 if the roundings are
    # independent; as the keys repeat the terms of T cancel, and the walk by tokens (the same rounding, another order) shows by how much
    assert worst["tiles"] <= max(4.4e-6, 2 * worst["tokens"]), worst


def test_short_steps_walk_by_tokens():
    """A step of few tokens a portion gives the same bits with and without its tiles."""
    from swiftllm_amd.worker.kernels.delta_rule import delta_rule_scan
    gen = torch.Generator().manual_seed(1)
    H = G = 2
    d = dv = 64
    for step in ([(1, 0, 47)], [(i, 0, 17) for i in range(1, 10)]):
        n = sum(c for _, _, c in step)
        q, k = [torch.nn.functional.normalize(torch.randn(n, G, d, generator=gen), dim=2) for _ in range(2)]
        gpu = [x.contiguous().view(n, -1).cuda() for x in (q, k, (q * k).sum(2), torch.randn(n, H, dv, generator=gen),
                                                           torch.rand(n, H, generator=gen), torch.rand(n, H, generator=gen))]
        out = []
        for tiles in (False, True):
            slots = Slots([d * dv * H], num_slots=10)
            out.append(torch.empty((n, H * dv), device="cuda"))
            delta_rule_scan(out[-1], *gpu, _ref(slots, step, tiles), slots.off[0], H, G, d, dv)
        assert torch.equal(out[0], out[1])
