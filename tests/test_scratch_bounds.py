"""What memory profiling sets aside for scratch covers every step within the limits, however its tokens are shared out over portions."""
import random
from types import SimpleNamespace

import pytest

from swiftllm_amd.worker.kernels import delta_rule, window_attn
from swiftllm_amd.worker.kernels.linear_scan import SEGMENT_MAX_SCRATCH
from swiftllm_amd.worker.kernels.window_attn import SHARE_MAX_SCRATCH


def test_shares_stay_within_their_bound():
    for splits, floats in ((1, 10), (16, 1000), (8, 8192 * 514), (16, 1 << 24), (16, 1 << 27), (2, 0)):
        got, scratch = window_attn.share_scratch("meta", splits, floats)
        assert 1 <= got <= splits and (scratch is None) == (got == 1)
        assert scratch is None or (scratch.numel() == got * floats and 4 * scratch.numel() <= SHARE_MAX_SCRATCH)
        # as many as the bound leaves
        assert got == splits or 4 * (got + 1) * floats > SHARE_MAX_SCRATCH


@pytest.mark.parametrize("heads,dim,vdim", [(8, 128, 128), (3, 64, 16), (64, 128, 1024)])
def test_tiles_of_any_portions(heads, dim, vdim):
    from swiftllm_amd import _hip
    mixer = SimpleNamespace(num_heads=heads, head_dim=dim, value_dim=vdim)
    rng = random.Random(heads)
    for _ in range(300):
        tokens, batch = rng.randint(1, 20000), rng.randint(1, 300)
        portions = min(rng.randint(1, batch), tokens)
        cuts = sorted(rng.sample(range(1, tokens), portions - 1)) if rng.random() < 0.5 else list(range(1, portions))
        lens = [b - a for a, b in zip([0] + cuts, cuts + [tokens])]
        need = _hip.load().swl_delta_rule_tiles_scratch_bytes(sum(-(-n // 16) for n in lens), heads, dim, vdim)
        if need <= delta_rule.TILES_MAX_SCRATCH:        # (else the step walks token by token)
            assert need <= delta_rule.most_tiles_scratch(tokens, batch, mixer)


def test_what_the_designs_set_aside():
    from swiftllm_amd.worker.kekapel_model import KekapelModel
    from swiftllm_amd.worker.lorulix_model import LorulixModel
    from swiftllm_amd.worker.ratilorn_model import RatilornModel
    from swiftllm_amd.worker.vafozen_model import VafozenModel

    def aside(kind, layers=(), tokens=8192):
        model = kind.__new__(kind)
        model.model_config = SimpleNamespace(layers=layers)
        return model._scratch_bytes(tokens, 64)
    assert aside(KekapelModel) == SHARE_MAX_SCRATCH
    assert aside(RatilornModel) == aside(VafozenModel) == max(SHARE_MAX_SCRATCH, SEGMENT_MAX_SCRATCH)
    delta = SimpleNamespace(type="delta", mixer=SimpleNamespace(num_heads=32, head_dim=128, value_dim=128))
    attention = SimpleNamespace(type="attention", mixer=None)
    assert aside(LorulixModel, [attention]) == SHARE_MAX_SCRATCH
    assert SHARE_MAX_SCRATCH < aside(LorulixModel, [attention, delta]) < aside(LorulixModel, [delta], 1 << 20) == delta_rule.TILES_MAX_SCRATCH
