"""The linear recurrence with long portions cut into segments that run side by side (csrc/linear_scan.hip) against float64: portions that end
inside, at and just after a segment, short ones beside them, states carried into and out of the step."""
import pytest
import torch

import vafozen_oracle as O
from test_gpu_vafozen import Step, state_manager

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,d,dv,bonus", [(2, 2, 128, 128, False), (4, 2, 64, 48, True), (1, 1, 20, 260, False), (2, 1, 200, 16, True),
                                            (1, 1, 320, 20, False)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_segments(H, G, d, dv, bonus, dtype):
    from swiftllm_amd.worker.kernels import linear_scan
    g = torch.Generator().manual_seed(d)
    u = torch.randn(H, d, generator=g) if bonus else None
    mgr = state_manager()
    off = mgr.add_region(H * d * dv)
    step, data, at = Step(mgr), {}, {}
    lens = {0: 960, 2: 945, 3: 3}
    for s, n in lens.items():
        q, k, v = (torch.randn(n, c, generator=g).to(dtype) for c in (G * d, G * d, H * dv))
        decay = torch.rand(n, H * d, generator=g) ** 0.02
        decay[torch.rand(decay.shape, generator=g) < 0.001] = 0.0
        rep = lambda x: x.double().view(n, G, d).repeat_interleave(H // G, dim=1)       # noqa: E731
        args = 0.3 * rep(q), rep(k), v.double().view(n, H, dv), decay.double().view(n, H, d)
        want = (O.bonus_scan(*args, u.double()) if bonus else O.linear_scan(*args)).reshape(n, H * dv)
        data[s], at[s] = (q, k, v, decay, want), 0
    for counts in ({0: 400, 2: 385, 3: 1}, {0: 432, 3: 1}, {2: 560, 0: 128, 3: 1}):
        parts = [(s, at[s], c) for s, c in counts.items()]
        pick = lambda j: torch.cat([data[s][j][a:a + c] for s, a, c in parts]).cuda()       # noqa: E731
        st = step.ref(parts)
        st.longest = max(counts.values())
        segments, seg_tiles, _ = linear_scan.scan_segments(st, H, d, dv)
        assert segments > 1 and segments * seg_tiles * 16 >= st.longest
        y = linear_scan.linear_recurrence(pick(0), pick(1), pick(2), pick(3), st, off, H, d, dv, q_scale=0.3,
                                          bonus=u.cuda() if bonus else None, num_qk_heads=G).cpu().double()
        o = 0
        for s, a, c in parts:
            want = data[s][4]
            # fp32 products and sums from 16-bit or fp32 operands, the bound of the walk without segments
            assert (y[o:o + c] - want[a:a + c]).abs().max() < 3e-5 * float(want.abs().max()), (s, a, c)
            o += c
            at[s] += c


def test_rule():
    """Portions stay whole when there are enough of them, or too short ones."""
    from swiftllm_amd.worker.kernels import linear_scan

    class Ref:
        pass
    st = Ref()
    st.pool = torch.empty(1, device="cuda")
    for longest, portions, heads, vdim, cut in ((368, 1, 8, 128, False), (369, 1, 8, 128, True), (1000, 32, 16, 128, False), (1000, 3, 16, 128, False),
                                                (4096, 1, 16, 128, True), (4096, 8, 32, 128, False)):
        st.longest, st.tiles, st.seq_row0 = longest, (torch.empty(portions * -(-longest // 16)),), torch.empty(portions)
        segments, seg_tiles, _ = linear_scan.scan_segments(st, heads, 128, vdim)
        assert (segments > 1) == cut and (not cut or segments * seg_tiles * 16 >= longest)
