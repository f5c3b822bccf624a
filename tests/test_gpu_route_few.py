"""Routers of steps of many tokens (csrc/moe.hip, two or four tokens a wave): the same bits as the kernels of fewer tokens, which the same rows meet
in slices, for ties, scores that are no numbers, groups of every size, ragged widths and row counts."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3073, 4609, 4614, 5633, 6601, 6606])
@pytest.mark.parametrize("experts,top,count,keep", [(8, 2, 4, 2), (6, 3, 3, 2), (6, 2, 2, 1), (8, 8, 2, 2), (5, 1, 1, 1), (8, 2, 8, 3), (4, 4, 2, 2), (1, 1, 1, 1)])
@pytest.mark.parametrize("width,dtype", [(260, torch.bfloat16), (1024, torch.float16), (100, torch.float32)])
def test_same_bits(n, experts, top, count, keep, width, dtype):
    from swiftllm_amd.worker.kernels.moe import moe_route, moe_route_grouped, moe_route_scores
    g = torch.Generator().manual_seed(n + experts + width)
    router, bias = torch.randn(experts, width, generator=g).cuda(), (0.3 * torch.randn(experts, generator=g)).cuda()
    if experts == 8:
        router[3], bias[3] = router[5], bias[5]     # ties
    if experts == 5:
        router[0, 0] = float("nan")
    if experts == 6:
        bias[1] = float("-inf")
    h = torch.randint(-2, 3, (n, width), generator=g).to(dtype).cuda()
    for f in (lambda x: moe_route(x, router, bias, top), lambda x: moe_route_scores(x, router, top, 0.7),
              lambda x: moe_route_grouped(x, router, bias, top, count, keep), lambda x: moe_route_grouped(x, router, None, top, count, keep, False)):
        got, want = f(h), [f(h[i:i + 1000].contiguous()) for i in range(0, n, 1000)]
        assert torch.equal(got[0], torch.cat([x[0] for x in want]))
        w = torch.cat([x[1] for x in want])
        assert torch.equal(got[1].isnan(), w.isnan()) and torch.equal(got[1].nan_to_num(), w.nan_to_num())
