"""Causal convolutions with carried inputs (csrc/conv_tail.h) against float64: one to six taps, eight channels a thread and one, portions
shorter than the taps, several sequences a step."""
import pytest
import torch

from test_gpu_lorulix import Slots

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("channels", [8, 12, 1024, 1032, 2056])
@pytest.mark.parametrize("taps", [1, 2, 3, 4, 6])
def test_portions(taps, channels, dtype):
    from swiftllm_amd.worker.kernels.rms_stream import causal_conv_state
    g = torch.Generator().manual_seed(taps * channels)
    w = torch.randn(taps, channels, generator=g)
    slots = Slots([2 * (taps - 1) * channels], num_slots=3)
    rows = {s: torch.randn(n, channels, generator=g).to(dtype) for s, n in ((1, 40), (2, 7))}
    at = {1: 0, 2: 0}
    for counts in ({1: 1}, {1: 2, 2: 1}, {2: 3, 1: 17}, {1: 1, 2: 1}, {2: 2, 1: 19}):
        parts = [(s, at[s], c) for s, c in counts.items()]
        h = torch.cat([rows[s][a:a + c] for s, a, c in parts]).cuda()
        out = causal_conv_state(h, w.cuda(), slots.ref(parts), slots.off[0], True).double().cpu()
        o = 0
        for s, a, c in parts:
            full = torch.cat((torch.zeros(taps - 1, channels, dtype=torch.float64), rows[s].double()))
            want = sum(full[j:j + rows[s].shape[0]] * w[j].double() for j in range(taps)) + rows[s].double()
            got = out[o:o + c]
            # up to seven fp32 terms, then one rounding to the type
            eps = 1e-6 if dtype == torch.float32 else 2.0 ** -8
            assert ((got - want[a:a + c]).abs() <= eps * want[a:a + c].abs() + 2e-6).all(), (s, a, c)
            o += c
            at[s] += c
