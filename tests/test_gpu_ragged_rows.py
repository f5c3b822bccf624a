"""Prompt-sized steps of models whose matrices have a number of rows that is no multiple of 8: products of them are rows one behind the other, which the
kernels behind them read (csrc/polynorm.hip, swl_logit_softcap, the residual steps)."""
import pytest
import torch

import kekapel_oracle as K
import rokevik_oracle as R
import test_gpu_kekapel as TK
import test_gpu_rokevik as TR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(257, 682, 256), (300, 1001, 512), (4500, 4, 256), (257, 9, 1024)])
def test_products_are_contiguous(m, n, k, dtype):
    from swiftllm_amd.worker.kernels.linear import linear
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn((m, k), generator=g, device="cuda").to(dtype)
    w = (torch.randn((n, k), generator=g, device="cuda") / k ** 0.5).to(dtype)
    y, z = linear(x, w, True), x.double() @ w.double().T
    assert y.shape == (m, n) and y.is_contiguous()
    # fp32 sums in any order (each addition rounds by 2^-24 of the magnitudes' sum), rounded once
    bound = (2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7) * z.abs() + 2.0 ** -24 * k * (x.double().abs() @ w.double().abs().T) + 2.0 ** -24
    assert bool(((y.double() - z).abs() <= bound).all())


def test_kekapel_with_ragged_feed_forward(tmp_path):
    cfg = K.make_config(width=256, vocab=97, layers=[K.attention_layer(dim=64, vdim=64, mlp=K.dense_mlp(682)), K.attention_layer(dim=64, vdim=64, mlp=K.dense_mlp(681))],
                        max_positions=320)
    W = K.random_weights(cfg, seed=3)
    toks = TK.tokens_for(cfg, 300, 5)
    want = K.forward(cfg, W, toks)
    model = TK.make_model(tmp_path / "m", cfg, W, "bfloat16")
    assert TK.rel_err(model.step([TK.entry(0, toks, 0)]), want) < TK.BF16_TOL


def test_rokevik_with_capped_logits_of_a_ragged_vocabulary(tmp_path):
    cfg = R.make_config(layers=[R.attention_layer(dim=64, rot_dims=32), R.min_gru_layer(width=256)], width=256, vocab=301, groups=2, streams=2, loop=None)
    W = R.random_weights(cfg, seed=4)
    toks = TR.tokens_for(cfg, 290, 6)
    want = R.forward(cfg, TR.f64(W), toks)
    model = TR.make_model(tmp_path / "m", cfg, W, "bfloat16")
    got = model.step([TR.entry(0, toks, 0)])
    assert got.dtype == torch.float32 and TR.close(got, want, "bfloat16")
