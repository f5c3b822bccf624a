"""Captured decode steps of the step-planned workers when the step's metadata outgrows its buffer: the captures are taken again."""
import pytest
import torch

import lorulix_oracle as O
from test_gpu_lorulix import F32_TOL, entry, make_model, rel_err, tokens_for

pytestmark = pytest.mark.gpu


def test_a_large_step_between_captured_decode_steps(tmp_path):
    cfg = O.make_config()
    W = O.make_weights(cfg)
    model = make_model(tmp_path / "m", cfg, W, "float32", num_blocks=90, max_seqs=6, graph=True)
    toks = tokens_for(cfg, 40, 1)
    want = O.forward(cfg, W, toks)[0]
    got = [model.step([entry(0, toks[:30], 0)])]
    for i in range(30, 34):
        got.append(model.step([entry(0, toks[i:i + 1], i)]).clone())
    held = model._meta_dev.numel()
    model.step([entry(s, tokens_for(cfg, 250, s), 0, (249,)) for s in (1, 2, 3, 4)])
    assert model._meta_dev.numel() > held and model.graph_captures == 1
    for i in range(34, 40):
        got.append(model.step([entry(0, toks[i:i + 1], i)]).clone())
        torch.cuda.synchronize()
    assert model.graph_captures == 2
    assert rel_err(torch.cat(got), want) < F32_TOL


def test_a_step_on_expanded_pages_between_captured_decode_steps(tmp_path):
    """Memory profiling runs a step of the most tokens without a pool, and so without the arrays of the expansion: the buffer it sizes has
    room for them, and the largest step leaves the captures in place."""
    import rosilix_oracle
    from swiftllm_amd.worker.batch_plan import plan_step
    from test_gpu_rosilix import make_model as make_rosilix
    cfg = rosilix_oracle.make_config([rosilix_oracle.latent_mixer(heads=2, dim=64, rot_dim=64, vdim=64, kv_rank=256)])
    W = rosilix_oracle.make_weights(cfg)
    model = make_rosilix(tmp_path / "m", cfg, W, "bfloat16", num_blocks=130, graph=True)
    model.profile_num_blocks()
    toks, got = tokens_for(cfg, 520, 1), []
    model.step([entry(0, toks[:30], 0)])
    for i in range(30, 34):
        got.append(model.step([entry(0, toks[i:i + 1], i)]).clone())
    assert model.graph_captures == 1
    held = model._meta_dev
    prompts = [tokens_for(cfg, 341, s) for s in (1, 2, 3)]
    assert plan_step([entry(s, prompts[s - 1], 0, (340,)) for s in (1, 2, 3)]).latent_expansion(model.latent_expansion).seqs == 3
    model.step([entry(s, prompts[s - 1], 0, (340,)) for s in (1, 2, 3)])                # 1023 tokens of 1024
    model.step([entry(s, tokens_for(cfg, 170, s), 341, (169,)) for s in (1, 2, 3)])     # (three times the pages of its tokens)
    model.free_seqs_resources([1, 2, 3])
    for i in range(34, 40):
        got.append(model.step([entry(0, toks[i:i + 1], i)]).clone())
    assert model.graph_captures == 1 and model._meta_dev is held
    fresh = make_rosilix(tmp_path / "m", cfg, W, "bfloat16", num_blocks=130)
    fresh.step([entry(0, toks[:30], 0)])
    for i, logits in zip(range(30, 40), got):
        assert torch.equal(logits, fresh.step([entry(0, toks[i:i + 1], i)]))
