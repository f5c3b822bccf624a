"""Decode steps whose heads are the rows of the matrix-core tile (csrc/window_attn_mfma.hip) against float64: groups of two to more than
sixteen heads of a key head, shared values, masks, bias, slopes, sink, gate, with and without key shares."""
import pytest
import torch

from test_gpu_span_attn import _pool, _spans, _want

pytestmark = pytest.mark.gpu

CASES = [       # H, G, GV, d, dv, features
    (32, 8, 4, 64, 128, dict(window=300, mask_kind=0)),
    (8, 2, 2, 128, 128, dict(rel=True)),
    (8, 4, 4, 64, 64, dict(rel=True, window=37)),
    (6, 2, 2, 128, 64, dict(softcap=9.0, window=50)),
    (6, 2, 1, 64, 128, dict(window=48, mask_kind=1, out_f32=True)),
    (34, 2, 2, 64, 64, dict(slopes=True, sink=True)),
    (40, 1, 1, 576, 512, dict(gate=True)),
    (10, 5, 5, 96, 128, dict(gate=True, out_dim=100)),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_head_rows(case, dtype, monkeypatch):
    from swiftllm_amd.worker.kernels import window_attn
    from swiftllm_amd.worker.kernels.window_attn import AttentionSpec
    H, G, GV, d, dv, f = CASES[case]
    g = torch.Generator().manual_seed(case)
    parts = [(1, 0, 1), (2, 15, 1), (3, 16, 1), (4, 499, 1)]
    pool, sl, table, ks, vs = _pool([a + n for _, a, n in parts], G, GV, d, dv, dtype, g)
    seq, pos, tiles = _spans(parts)
    n, out_dim = len(parts), f.get("out_dim", dv)
    q = torch.randn(n, H * d + 4, generator=g).to(dtype)
    rel = torch.randn(H, 90, generator=g) if f.get("rel") else None
    gate = torch.randn(n, H * out_dim, generator=g).to(dtype) if f.get("gate") else None
    spec = AttentionSpec(H, G, d, dv, d ** -0.5, window=f.get("window", 0), mask_kind=f.get("mask_kind", 0), num_v_heads=GV,
                         softcap=f.get("softcap", 0.0), sink=torch.randn(H, generator=g).cuda() if f.get("sink") else None,
                         out_f32=f.get("out_f32", False), slopes=(torch.rand(H, generator=g) * 0.1).cuda() if f.get("slopes") else None,
                         out_dim=out_dim)
    assert window_attn.head_rows(spec, tiles[0], n)
    for slots in (window_attn.HEAD_ROWS_SLOTS, 1):      # shares of the keys by the rule; none
        monkeypatch.setattr(window_attn, "HEAD_ROWS_SLOTS", slots)
        if rel is None:
            got = window_attn.masked_attention(q.cuda(), pool, sl, table, seq, pos, spec, tiles, 500, gate=gate.cuda() if gate is not None else None)
        else:
            got = window_attn.window_attention(q.cuda(), None, pool, sl, table, seq, pos, spec, tiles, 500, rel.cuda())
        got = got.double().cpu()
        for j, (i, a, m) in enumerate(parts):
            want = _want(q[j:j + 1, :H * d].double().view(1, H, d), ks[j], vs[j], a, spec, rel.double() if rel is not None else None,
                         gate[j:j + 1].double() if gate is not None else None)
            # (as for the prompt form: one rounding of a convex combination of values of order one; fp32 results: the weights' 2^-16)
            eps = 2.0 ** -15 if spec.out_f32 else 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
            assert (got[j:j + 1] - want).abs().max() <= 1.1 * eps * max(1.0, float(want.abs().max())), (slots, i)
