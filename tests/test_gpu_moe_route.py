"""Routers at the edges of the choice (csrc/moe.hip): expert counts around the steps of the wave's arg-max, more choices than lanes, equal
scores, against the same choice in float64 on the CPU."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("experts,top", [(1, 1), (2, 1), (3, 2), (4, 4), (5, 2), (8, 2), (9, 3), (16, 4), (17, 2), (33, 6), (64, 64), (65, 65), (72, 66), (130, 8)])
def test_choice(experts, top):
    from swiftllm_amd.worker.kernels.moe import moe_route, moe_route_grouped, moe_route_scores
    g = torch.Generator().manual_seed(experts)
    h = torch.randn(37, 68, generator=g)
    h[5] = 0                            # (equal scores: the lowest experts, in order)
    router = torch.randn(experts, 68, generator=g) / 68 ** 0.5
    h_gpu, r_gpu, none = h.cuda(), router.cuda(), torch.zeros(experts, device="cuda")
    logits = h.double() @ router.double().T
    order = logits.sort(dim=1, descending=True, stable=True)
    # fp32 sums of 68 products of size ~1/8: errors below 68 * 2^-24 * 4 = 2e-5; rows with scores closer than that may choose either way
    gap = (order.values[:, :-1] - order.values[:, 1:])[:, :top]
    clear = (gap > 4e-5).all(dim=1) if experts > 1 else torch.ones(37, dtype=torch.bool)
    clear[5] = True
    assert experts > 20 or clear.sum() > 30
    chosen = order.values[:, :top]
    for route, want in ((moe_route(h_gpu, r_gpu, none, top), chosen.softmax(1)),
                        (moe_route_scores(h_gpu, r_gpu, top, 1.5), 1.5 * logits.softmax(1).gather(1, order.indices[:, :top])),
                        (moe_route_grouped(h_gpu, r_gpu, None, top), chosen.sigmoid() / chosen.sigmoid().sum(1, keepdim=True))):
        idx, weights = (x.cpu() for x in route)
        assert torch.equal(idx[clear].long(), order.indices[clear, :top])
        # weights: relative error of the exponential's argument (4e-5 over both terms) and of the sum
        torch.testing.assert_close(weights[clear].double(), want[clear], rtol=1e-4, atol=1e-7)


@pytest.mark.parametrize("count,per,keep,top", [(2, 4, 1, 3), (3, 1, 2, 2), (5, 3, 2, 4), (9, 2, 8, 16), (17, 4, 3, 5)])
def test_groups(count, per, keep, top):
    from swiftllm_amd.worker.kernels.moe import moe_route_grouped
    g = torch.Generator().manual_seed(count)
    experts = count * per
    h, router, corr = torch.randn(41, 68, generator=g), torch.randn(experts, 68, generator=g) / 68 ** 0.5, torch.randn(experts, generator=g)
    score = (h.double() @ router.double().T).sigmoid()
    choice = (score + corr.double()).view(41, count, per)
    group = choice.topk(min(2, per), dim=2).values.sum(2)
    kept = group.sort(dim=1, descending=True).indices[:, :keep]
    mask = torch.zeros(41, count, dtype=torch.bool).scatter_(1, kept, True)
    order = choice.masked_fill(~mask[:, :, None], float("-inf")).view(41, experts).sort(dim=1, descending=True).indices[:, :top]
    want = score.gather(1, order)
    idx, weights = (x.cpu() for x in moe_route_grouped(h.cuda(), router.cuda(), corr.cuda(), top, count, keep))
    same = (idx.long() == order).all(dim=1)
    assert same.float().mean() > 0.95      # (scores closer than fp32 sums tell apart may choose either way)
    torch.testing.assert_close(weights[same].double(), (want / want.sum(1, keepdim=True))[same], rtol=1e-4, atol=1e-7)


@pytest.mark.parametrize("experts,top", [(2, 2), (8, 2), (9, 3), (72, 66)])
def test_scores_that_are_no_numbers(experts, top):
    """Tokens whose scores are NaN or -inf name experts that exist (what reads the experts' weights takes the ids as they are), with a weight
    of 0 or NaN, and leave the other tokens alone."""
    from swiftllm_amd.worker.kernels.moe import moe_experts, moe_route, moe_route_grouped, moe_route_scores
    g = torch.Generator().manual_seed(experts)
    h, router = torch.randn(13, 64, generator=g), torch.randn(experts, 64, generator=g) / 8
    bias = torch.zeros(experts)
    bad = h.clone()
    bad[3], bad[7, 5], bad[9, 0] = float("nan"), float("inf"), float("-inf")
    fine = [t for t in range(13) if t not in (3, 7, 9)]
    gate_up, down = torch.randn(experts, 2 * 32, 64, generator=g) / 8, torch.randn(experts, 64, 32, generator=g) / 6
    for route in (lambda x, b: moe_route(x, router.cuda(), b, top), lambda x, b: moe_route_scores(x, router.cuda(), top, 1.5),
                  lambda x, b: moe_route_grouped(x, router.cuda(), b, top)):
        want, got = route(h.cuda(), bias.cuda()), route(bad.cuda(), bias.cuda())
        assert int(got[0].min()) >= 0 and int(got[0].max()) < experts
        for a, b in zip(want, got):
            assert torch.equal(a[fine], b[fine])
        out = [moe_experts(x.cuda(), i, w, gate_up.cuda(), down.cuda(), 7.0).cpu() for x, (i, w) in ((h, want), (bad, got))]
        assert torch.equal(out[0][fine], out[1][fine]) and torch.isnan(out[1][3]).all()
    closed = torch.full((experts,), float("-inf"))      # every expert but one is closed
    closed[1] = 0.0
    idx, weights = (x.cpu() for x in moe_route(h.cuda(), router.cuda(), closed.cuda(), top))
    assert (idx[:, 0] == 1).all() and (weights[:, 0] == 1).all() and int(idx.min()) >= 0 and int(idx.max()) < experts
    assert (weights[:, 1:] == 0).all()
