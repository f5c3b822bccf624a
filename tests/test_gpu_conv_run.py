"""Kernels whose workgroups take four tokens in a row in steps of many (csrc/conv_tail.h, ConvRun) against steps of fewer, a token a workgroup:
the same bits of every result and of the carried inputs, with portions that begin and end between the four."""
import pytest
import torch

pytestmark = pytest.mark.gpu
LENS = [1, 2, 1, 5, 3, 1500, 1, 1, 1532, 3, 1500, 2, 1598, 1, 3]    # (6153 tokens: rows of any width are many; the last workgroup has one)
CUTS = [6, 10, 12]      # (1512, 1537, 1502 and 1602 tokens: few of any width)


def _steps():
    """(portions of every step) for a step of all LENS and for the same cut in four: a few tokens ahead of half the sequences, and one behind all."""
    ahead = [(s, 0, 3) for s in range(0, len(LENS), 2)]
    main = [(s, 3 if s % 2 == 0 else 0, c) for s, c in enumerate(LENS)]
    behind = [(s, a + c, 1) for s, a, c in main]
    return [ahead, main, behind], [ahead] + [main[a:b] for a, b in zip([0] + CUTS, CUTS + [len(LENS)])] + [behind]


def _same(run, channels, taps):
    """run(rows' slice, StateRef, tail offset) -> tensors, over both ways to take the same tokens."""
    from test_gpu_lorulix import Slots
    results = []
    for steps in _steps():
        slots, parts, at = Slots([2 * (taps - 1) * channels], num_slots=len(LENS)), [], 0
        for portions in steps:
            n = sum(c for _, _, c in portions)
            parts.append(run(slice(at, at + n), slots.ref(portions), slots.off[0]))
            at += n
        results.append([torch.cat(p) for p in zip(*parts)])
    for a, b in zip(*results):
        assert bool(torch.isfinite(a.float()).all()) and torch.equal(a, b)


TOTAL = sum(c for _, _, c in sum(_steps()[0], []))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("taps,channels,add", [(4, 1024, True), (1, 40, False), (3, 2056, True), (2, 8, False), (5, 64, True)])
def test_causal_conv(taps, channels, add, dtype):
    from swiftllm_amd.worker.kernels.rms_stream import causal_conv_state
    g = torch.Generator().manual_seed(channels + taps)
    h, w = torch.randn(TOTAL, channels + 8, generator=g).to(dtype).cuda(), torch.randn(taps, channels, generator=g).cuda()
    _same(lambda rows, st, off: (causal_conv_state(h[rows, :channels], w, st, off, add),), channels, taps)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,G,d,dv,taps", [(8, 2, 128, 128, 4), (3, 1, 24, 8, 2), (4, 4, 64, 40, 3), (2, 2, 20, 16, 1), (8, 8, 64, 24, 3)])
def test_delta_prep(H, G, d, dv, taps, dtype):
    from swiftllm_amd import _hip
    g = torch.Generator().manual_seed(d + taps)
    C = 2 * G * d + H * dv
    proj = torch.randn(TOTAL, (C + H * dv + 2 * H + 7) // 8 * 8, generator=g).to(dtype).cuda()
    conv, a_log, dt = (torch.randn(*s, generator=g).cuda() for s in ((taps, C), (H,), (H,)))

    def run(rows, st, off):
        x = proj[rows]
        n = x.shape[0]
        qn, kn, kq, vv, beta, decay = (torch.empty(n, c, device="cuda") for c in (G * d, G * d, G, H * dv, H, H))
        _hip.call("swl_delta_prep", *(_hip.ptr(t) for t in (qn, kn, kq, vv, beta, decay, x)), x.stride(0), _hip.ptr(conv), _hip.ptr(a_log),
                  _hip.ptr(dt), _hip.ptr(st.pool), st.pool.stride(0), off, _hip.ptr(st.tok_pos), _hip.ptr(st.tok_start), _hip.ptr(st.tok_state),
                  _hip.ptr(st.tok_seq), n, H, G, d, dv, taps, _hip.dtype_code3(dtype), _hip.stream())
        return qn, kn, kq, vv, beta, decay
    _same(run, C, taps)
