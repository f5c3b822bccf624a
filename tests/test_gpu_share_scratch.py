"""The scratch of key shares belongs to one call: launches from several streams or threads at once give what each gives alone, a captured
step keeps its own, and prompts that grow from step to step leave no memory behind."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


class Case:
    """`tokens` decoded tokens, each at the end of a sequence of `keys` keys: 8 heads of 64 over 2."""
    H, G, D = 8, 2, 64

    def __init__(self, tokens, keys, dtype, seed):
        from swiftllm_amd.worker.kernels.window_attn import AttentionSpec, PoolSlice
        g = torch.Generator(device="cuda").manual_seed(seed)
        blocks = -(-keys // 16)
        rand = lambda *shape: torch.randn(*shape, generator=g, device="cuda").to(dtype)      # noqa: E731
        self.pool, self.q = rand(tokens * blocks, 2 * 16 * self.G * self.D), rand(tokens, self.H * self.D)
        self.slice = PoolSlice(0, 16 * self.G * self.D)
        self.table = torch.randperm(tokens * blocks, generator=g, device="cuda").view(tokens, blocks).int()
        self.seq = torch.arange(tokens, dtype=torch.int32, device="cuda")
        self.pos = torch.full((tokens,), keys - 1, dtype=torch.int32, device="cuda")
        self.spec = AttentionSpec(self.H, self.G, self.D, self.D, self.D ** -0.5)
        one = torch.ones(tokens, dtype=torch.int32, device="cuda")
        self.tiles = (self.seq, one)

    def run(self, q=None):
        from swiftllm_amd.worker.kernels.window_attn import masked_attention
        return masked_attention(self.q if q is None else q, self.pool, self.slice, self.table, self.seq, self.pos, self.spec, self.tiles, 1024)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("streams", [1, 2])
def test_threads_at_once(dtype, streams):
    """Two workers on two streams, or on one stream from two threads (the calls give up the interpreter between their launches)."""
    cases = [Case(3 + i, 500, dtype, i) for i in range(2)]
    alone = [c.run() for c in cases]
    torch.cuda.synchronize()
    lanes = [torch.cuda.Stream() for _ in range(streams)]
    got, errors = [[], []], []

    def work(i):
        try:
            with torch.cuda.stream(lanes[i % streams]):
                for _ in range(60):
                    got[i].append(cases[i].run())
        except Exception as e:      # noqa: BLE001
            errors.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for i in range(2):
        assert len(got[i]) == 60 and all(torch.equal(x, alone[i]) for x in got[i])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_captured_shares_between_eager_ones(dtype):
    case, other = Case(3, 500, dtype, 0), Case(5, 300, dtype, 1)
    q = case.q.clone()
    want_other = other.run()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        case.run(q)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = case.run(q)
    for k in range(4):
        q.copy_(case.q * (1 + k))
        want = case.run(q).clone()
        assert torch.equal(other.run(), want_other)
        graph.replay()
        assert torch.equal(other.run(), want_other)
        torch.cuda.synchronize()
        assert torch.equal(out, want), k


def test_growing_prompts_leave_no_memory():
    """A conversation whose prompts grow: the shares of latent heads want more scratch every turn, and each gives it back."""
    from swiftllm_amd.worker.kernels.window_attn import AttentionSpec, PoolSlice, StepTiles, masked_attention
    H, d, dv, most = 8, 576, 512, 1040
    pool = torch.zeros(most // 16 + 1, 16 * (d + dv), dtype=torch.bfloat16, device="cuda")
    table = torch.arange(most // 16 + 1, dtype=torch.int32, device="cuda")[None]
    spec = AttentionSpec(H, 1, d, dv, d ** -0.5)

    def turn(n):
        runs = lambda size: (torch.arange(0, n, size, dtype=torch.int32, device="cuda"),      # noqa: E731
                             torch.tensor([min(size, n - i) for i in range(0, n, size)], dtype=torch.int32, device="cuda"))
        start = torch.zeros(n, dtype=torch.int32, device="cuda")
        tiles = StepTiles(*runs(16), (*runs(32), start), n)
        q = torch.ones(n, H * d, dtype=torch.bfloat16, device="cuda")
        masked_attention(q, pool, PoolSlice(0, 16 * d), table, start, torch.arange(n, dtype=torch.int32, device="cuda"), spec, tiles, 4096)
        torch.cuda.synchronize()
    turn(16)
    before = torch.cuda.memory_allocated()
    for n in range(200, most, 70):
        turn(n)
        assert torch.cuda.memory_allocated() == before, n


def test_profile_sets_scratch_aside(tmp_path, monkeypatch):
    import lorulix_oracle as O
    from test_gpu_lorulix import make_model
    cfg = O.make_config()
    model = make_model(tmp_path / "m", cfg, O.make_weights(cfg, seed=1))
    ecfg = model.engine_config
    want = model._scratch_bytes(ecfg.max_tokens_in_batch, ecfg.max_batch_size)
    model.profile_num_blocks()
    with_it = model.profile_num_blocks()
    monkeypatch.setattr(model, "_scratch_bytes", lambda tokens, batch: 0)
    without = model.profile_num_blocks()
    block = model.block_elems * model.dtype.itemsize
    # (what the two runs' free memory may differ by)
    assert abs((without - with_it) * block - want) <= block + (32 << 20)
