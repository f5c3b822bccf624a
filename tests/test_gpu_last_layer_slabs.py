"""The slabs of the last layer's down projection in steps with prompts: added into the residual and normed in one launch, with the bits of the three
steps apart."""
import pytest
import torch

from oracle import synth
from test_gpu_model import _make_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_last_layer(tmp_path, dtype, monkeypatch):
    from swiftllm_amd.worker import model as M
    from swiftllm_amd.worker.kernels.linear import SplitKPartials
    from swiftllm_amd.worker.kernels.rmsnorm import rmsnorm_inplace
    cfg = synth.make_config(**dict(synth.SMALL128, hidden_size=1024, num_attention_heads=8, num_key_value_heads=2, intermediate_size=4096, num_hidden_layers=2))
    tdtype = getattr(torch, dtype)
    model = _make_model(tmp_path, cfg, synth.make_state_dict(cfg, seed=3, dtype=tdtype), num_blocks=64, dtype=dtype, max_tokens_in_batch=1024)
    g = torch.Generator().manual_seed(1)
    prompts = [torch.randint(0, cfg["vocab_size"], (n,), generator=g).tolist() for n in (140, 1, 131)]
    fused, calls = M.fused_add_rmsnorm_from_splitk, []

    def count(partials, *a):
        calls.append(partials.shape)
        return fused(partials, *a)

    def apart(partials, residual, weight, eps):
        x = materialize(partials)
        x += residual
        rmsnorm_inplace(x, weight, eps)
        return x

    materialize = SplitKPartials.materialize
    monkeypatch.setattr(SplitKPartials, "materialize", lambda self: pytest.fail("a launch that only adds slabs up"))
    results = []
    for stand_in in (count, apart):
        monkeypatch.setattr(M, "fused_add_rmsnorm_from_splitk", stand_in)
        toks = model.forward(prompts, [0, 1, 2], [])
        mixed = model.forward([prompts[0] + prompts[2], [toks[0]], [toks[2]]], [3, 0, 2], [141, 132])
        results.append((toks, mixed, [t.clone() for t in model.post_layer.logits_tap]))
        model.post_layer.logits_tap.clear()
        model.free_seqs_resources([0, 1, 2, 3])
    assert calls == [(272, 1024), (273, 1024)]
    assert results[0][:2] == results[1][:2]
    assert all(torch.equal(a, b) for a, b in zip(results[0][2], results[1][2]))
