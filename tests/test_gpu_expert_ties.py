"""What a row of logits owes to the choice of experts: in 16 bits a token whose best scores lie closer together than rounding may take
another expert than the oracle, and its row then differs by an expert's share, not by rounding. Every choice is the router's rule applied
to the scores of the model's own rows, these scores are the oracle's up to rounding, and rows that see no
token with another expert differ from the oracle's by rounding alone."""
import pytest
import torch

import ratilorn_oracle as O
from test_gpu_ratilorn import BF16_TOL, entry, f64, make_model, row_err, tokens_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("groups", [(4, 2), None])
def test_rows_that_differ_are_ties(tmp_path, monkeypatch, groups):
    import swiftllm_amd.worker.layers.ratilorn_layer as layer
    moe = O.moe_mlp(64, 8, 2, groups, 64)
    cfg = O.make_config(layers=[O.attention_layer(heads=8, kv_heads=4, dim=64, vdim=64, mlp=moe),
                                O.parallel_layer(heads=8, kv_heads=4, dim=64, vdim=64, s_heads=2, s_vdim=64, state=32, mlp=moe),
                                O.attention_layer(heads=8, kv_heads=4, dim=64, vdim=64, mlp=moe)], width=128, max_positions=512)
    W = O.random_weights(cfg, seed=7)
    prompts, n = 40, 12
    toks = [tokens_for(cfg, n, seed) for seed in range(prompts)]
    ours, theirs = [], []
    route, moe_ff = layer.moe_route_grouped, O.moe_ff

    def gpu_route(h, *rest):
        out = route(h, *rest)
        ours.append((h.double().cpu(), out[0].long().cpu()))
        return out

    def oracle_ff(h, W, p, mlp):
        theirs.append((h, W[p + "router"], W[p + "correction"], mlp["router"]))
        return moe_ff(h, W, p, mlp)
    monkeypatch.setattr(layer, "moe_route_grouped", gpu_route)
    monkeypatch.setattr(O, "moe_ff", oracle_ff)
    want = torch.cat([O.forward(f64(W), cfg, t)[0] for t in toks])
    model = make_model(tmp_path / "m", cfg, W, "bfloat16", max_seqs=prompts)
    err = row_err(model.step([entry(i, t, 0) for i, t in enumerate(toks)]), want)

    clean = torch.ones(prompts, n, dtype=torch.bool)        # no token of the prompt up to this one has taken another expert so far
    for i, (h, chosen) in enumerate(ours):
        ref = torch.cat([t[0] for t in theirs[i::len(ours)]])
        _, router, correction, r = theirs[i]
        scores, oracle_scores = (torch.sigmoid(x @ router.T) + correction for x in (h, ref))
        rule = O.route(h @ router.T, correction, r["top"], r.get("groups"))[0]
        # the kernel's scores are fp32 sums: it may differ from the rule in 64 bits where two of them lie within 1e-5
        for t in (rule.sort(1).values != chosen.sort(1).values).any(1).nonzero().flatten().tolist():
            gaps = [scores[t].sort().values.diff().abs().min()]
            if groups:
                gaps.append(scores[t].view(groups[0], -1).topk(2, 1).values.sum(1).sort().values.diff().abs().min())
            assert min(gaps) < 1e-5, (t, scores[t])
        # a row that is off by BF16_TOL moves a logit of size 2 by 0.16, and its sigmoid by a quarter of that
        assert (scores - oracle_scores)[clean.flatten()].abs().max() < 0.5 * BF16_TOL
        best = O.route(ref @ router.T, correction, r["top"], r.get("groups"))[0]
        same = (best.sort(1).values == chosen.sort(1).values).all(1).view(prompts, n)
        clean &= same.long().cumprod(1).bool()
    clean = clean.flatten()
    print("rows that owe nothing to another expert:", int(clean.sum()), "largest error %.4f" % float(err[clean].max()),
          "largest of the others %.4f" % float(err[~clean].max()))
    assert clean.double().mean() > 0.5 and not clean.all()
    assert err[clean].max() < BF16_TOL
