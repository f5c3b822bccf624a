"""The prompt form of attention with mixed heads (csrc/mix_attn.hip) against the same attention in float64: heads that fill a wave's share
or not, edges of the 16-token tiles and 32-key stages, windows, cap, distance penalties, key shares; and what the form leaves to others."""
import math

import pytest
import torch

from test_gpu_span_attn import _pool, _spans

pytestmark = pytest.mark.gpu


class Mixer:
    def __init__(self, H, G, d, dv, window, softcap):
        self.num_q_heads, self.num_kv_heads, self.head_dim, self.value_dim, self.window = H, G, d, dv, window
        self.softcap, self.scale = softcap, d ** -0.5


def _want(q, k, v, start, mixer, talk, r1, r2, pb, sigmoid):
    n, H, _ = q.shape
    rep = H // k.shape[1]
    pos, key = torch.arange(start, start + n)[:, None], torch.arange(k.shape[0])[None]
    see = (key <= pos) & (pos - key < (mixer.window or 1 << 30))
    s = torch.stack([q[:, h] @ k[:, h // rep].T * mixer.scale for h in range(H)])
    if sigmoid:
        if r1 is not None:
            s = s - r1[:, None, None] * torch.log1p(r2[:, None, None] * (pos - key).clamp(min=0))
        w = torch.sigmoid(s + (pb[:, None, None] if pb is not None else 0.0)) * see
        w = torch.einsum("hg,gqk->hqk", talk, w)
    else:
        if mixer.softcap:
            s = mixer.softcap * torch.tanh(s / mixer.softcap)
        w = torch.softmax(torch.einsum("hg,gqk->hqk", talk, s).masked_fill(~see, -math.inf), 2)
    return torch.stack([w[h] @ v[:, h // rep] for h in range(H)], 1).reshape(n, -1)


CASES = [       # H, G, d, dv, window, softcap (softmax) / penalties (sigmoid)
    (16, 4, 128, 128, 0, True),
    (16, 8, 64, 64, 37, False),
    (8, 2, 128, 64, 50, True),
    (8, 8, 64, 128, 0, False),
    (6, 3, 64, 64, 0, True),
    (12, 2, 128, 128, 200, True),
    (10, 1, 64, 128, 33, False),
    (1, 1, 128, 128, 0, True),
    (3, 1, 64, 64, 16, True),
]


@pytest.mark.parametrize("sigmoid", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("parts", [[(1, 0, 1), (2, 0, 200), (3, 0, 33)], [(1, 96, 31), (2, 0, 64), (3, 250, 1), (4, 15, 130)]])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_mixed_attention(case, parts, dtype, sigmoid):
    from swiftllm_amd.worker.kernels import window_attn
    H, G, d, dv, window, extra = CASES[case]
    g = torch.Generator().manual_seed(case)
    pool, sl, table, ks, vs = _pool([a + n for _, a, n in parts], G, G, d, dv, dtype, g)
    seq, pos, tiles = _spans(parts)
    n, esize = seq.shape[0], pool.element_size()
    q = torch.randn(n, H * d + 8, generator=g).to(dtype)
    talk = torch.eye(H) + 0.3 * torch.randn(H, H, generator=g)
    r1, r2, pb = [torch.rand(H, generator=g) if sigmoid and extra else None for _ in range(3)]
    mixer = Mixer(H, G, d, dv, window, 9.0 if extra and not sigmoid else 0.0)
    gpu = [t.cuda() if t is not None else None for t in (talk, r1, r2, pb)]
    qd = q.cuda()
    for longest in (tiles.longest, 0):      # shares of the keys by the rule; none
        tiles.longest = longest
        out = torch.full((n, H * dv), 7.0, dtype=dtype, device="cuda")
        args = (qd, out, pool.data_ptr() + sl.k_offset * esize, pool.data_ptr() + sl.v_offset * esize, pool, table, seq, pos, tiles, mixer)
        assert window_attn.mix_launch("swl_mix_sigmoid_attn", *args, gpu, (), dv) if sigmoid else \
            window_attn.mix_launch("swl_mix_attn", *args, gpu[:1], (float(mixer.softcap),), dv + 2)
        got, at = out.double().cpu(), 0
        for j, (i, a, m) in enumerate(parts):
            want = _want(q[at:at + m, :H * d].double().view(m, H, d), ks[j], vs[j], a, mixer,
                         *[t.double() if t is not None else None for t in (talk, r1, r2, pb)], sigmoid)
            # weights in two 16-bit terms (2^-16 of each), fp32 sums: one rounding of the result is left, relative to its size
            eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
            err = (got[at:at + m] - want).abs().max()
            assert err <= 1.1 * eps * max(1.0, float(want.abs().max())), (longest, i, float(err))
            at += m


@pytest.mark.parametrize("H,G,d,dv,parts,shift", [
    (9, 3, 64, 64, [(1, 0, 40)], 0),            # a wave's two heads on two key heads
    (17, 1, 64, 64, [(1, 0, 40)], 0),           # more than 16 heads
    (8, 2, 96, 64, [(1, 0, 40)], 0),            # a head size that is not compiled
    (8, 2, 64, 64, [(1, 40, 1), (2, 9, 3)], 0),     # few tokens a portion
    (8, 2, 64, 64, [(1, 0, 40)], 4),            # queries on 8 bytes
])
def test_other_steps_keep_their_kernels(H, G, d, dv, parts, shift):
    from swiftllm_amd.worker.kernels import window_attn
    g = torch.Generator().manual_seed(H)
    pool, sl, table, ks, vs = _pool([a + n for _, a, n in parts], G, G, d, dv, torch.bfloat16, g)
    seq, pos, tiles = _spans(parts)
    n, esize = seq.shape[0], pool.element_size()
    q = torch.randn(n, H * d + 8, generator=g).to(torch.bfloat16).cuda()
    talk = torch.eye(H) + 0.3 * torch.randn(H, H, generator=g)
    mixer = Mixer(H, G, d, dv, 0, 0.0)
    out = torch.empty((n, H * dv), dtype=torch.bfloat16, device="cuda")
    qs = q[:, shift:]
    assert not window_attn.mix_launch("swl_mix_attn", qs, out, pool.data_ptr() + sl.k_offset * esize,
                                      pool.data_ptr() + sl.v_offset * esize, pool, table, seq, pos, tiles, mixer, (talk.cuda(),), (0.0,),
                                      dv + 2)
    got = window_attn.window_attention(qs, talk.cuda(), pool, sl, table, seq, pos, mixer, tiles=tiles).double().cpu()
    at = 0
    for j, (i, a, m) in enumerate(parts):
        want = _want(qs[at:at + m, :H * d].double().cpu().view(m, H, d), ks[j], vs[j], a, mixer, talk.double(), None, None, None, False)
        assert (got[at:at + m] - want).abs().max() <= 1.1 * 2.0 ** -8 * max(1.0, float(want.abs().max()))
        at += m
