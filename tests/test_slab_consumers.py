"""Where a prompt-sized step asks for a product's K shares as slabs: only where the step behind it adds them up."""
from types import SimpleNamespace

import pytest
import torch


@pytest.mark.parametrize("fuse", [True, False])
@pytest.mark.parametrize("layer", [0, 1])
def test_llama_layers(fuse, layer, monkeypatch):
    from swiftllm_amd.worker.layers import transformer_layer as T
    asked = []
    weight = SimpleNamespace(o_proj="o", up_gate_proj="up_gate", down_proj="down", ffn_norm=None)
    monkeypatch.setattr(T, "linear_tile_partial", lambda a, w: asked.append(w))
    monkeypatch.setattr(T, "linear", lambda a, w, skinny=False: torch.zeros(300, 16))
    for name in ("linear_silu_gate", "linear_gated"):
        monkeypatch.setattr(T, name, lambda *a, **k: None)
    for name in ("fused_add_rmsnorm_inplace", "silu_and_mul_inplace"):
        monkeypatch.setattr(T, name, lambda *a, **k: None)
    cfg = SimpleNamespace(num_layers=2, ffn_inter_dim=8, rms_norm_eps=1e-5)
    op = T.LlamaTransformerLayer(cfg, SimpleNamespace(use_skinny_gemm=True, fuse_splitk_consumers=fuse), weight, None, layer)
    out = op._forward_after_attention(torch.zeros(300, 16), torch.zeros(300, 16), False, None)
    assert isinstance(out, torch.Tensor)
    assert asked == (["o", "down"] if fuse else [])


@pytest.mark.parametrize("rows,asks", [(8192, True), (8448, False)])
def test_stepped_designs(rows, asks, monkeypatch):
    from swiftllm_amd.worker.layers import kekapel_layer as K
    asked = []
    monkeypatch.setattr(K, "linear_tile_partial", lambda a, w: asked.append(w))
    monkeypatch.setattr(K, "linear", lambda a, w, skinny=False: torch.zeros(a.shape[0], w.shape[0]))
    K._project_partials(torch.zeros(257, 8, dtype=torch.bfloat16), torch.zeros(rows, 8, dtype=torch.bfloat16), True)
    assert bool(asked) == asks
