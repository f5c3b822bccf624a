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
