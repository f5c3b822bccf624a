"""GPU parity tests of the whole data plane: swiftllm_amd.LlamaModel (HIP kernels through the C ABI)
against (a) the golden run of the reference's own LlamaModel.forward and (b) the oracle model, on
random-init checkpoints. Bar: greedy token ids identical, pre-argmax
logits within 1e-3 (fp16; bf16 is held to its own rounding: 8 mantissa bits)."""
import os

import pytest
import torch

from oracle import synth
from oracle.ref_model import RefLlamaModel

pytestmark = pytest.mark.gpu


def _engine_config(path, **kw):
    from swiftllm_amd import EngineConfig
    base = dict(model_path=path, use_dummy=False, block_size=16, gpu_mem_utilization=0.9,
                num_cpu_blocks=8, max_seqs_in_block_table=16, max_blocks_per_seq=32, max_batch_size=8,
                max_tokens_in_batch=256)
    base.update(kw)
    return EngineConfig(**base)


def _make_model(tmp_path, cfg, sd, num_blocks=24, **kw):
    from swiftllm_amd import LlamaModel
    synth.write_model_dir(str(tmp_path), cfg, sd)
    model = LlamaModel(_engine_config(str(tmp_path), **kw))
    model.load_weights()
    model.init_kvcache_and_swap(num_blocks)
    model.post_layer.logits_tap = []
    return model


@pytest.mark.parametrize("opts", [dict(), dict(fuse_qkv=False, use_skinny_gemm=False),
                                  dict(fuse_qkv=False), dict(use_skinny_gemm=False),
                                  dict(tuning=dict(fuse_rope_kvstore=False)), dict(use_hip_graph=False),
                                  dict(tuning=dict(fuse_rope_into_attention=False)), dict(pack_decode_weights=False)],
                         ids=["default", "reference_blas_calls", "unfused_qkv", "blas_gemm", "unfused_rope",
                              "eager_launches", "rope_kernel", "row_major_weights"])
def test_forward_matches_reference_golden(tmp_path, golden, opts):
    """The scripted run frozen from the reference (fp16, BASELINE configs[0] model)."""
    g = golden("e2e_tiny_fp16.pt")
    cfg, e = g["config"], g["engine"]
    model = _make_model(tmp_path, cfg, synth.make_state_dict(cfg, seed=g["seed"]), e["num_gpu_blocks"],
                        num_cpu_blocks=e["num_cpu_blocks"], max_seqs_in_block_table=e["max_seqs_in_block_table"],
                        max_blocks_per_seq=e["max_blocks_per_seq"], **opts)
    worst = 0.0
    for step in g["steps"]:
        toks = model.forward(step["input_ids"], step["seq_ids"], step["dec_lens"])
        logits = model.post_layer.logits_tap[-1].float().cpu()
        worst = max(worst, (logits - step["logits"]).abs().max().item())
        assert toks == step["tokens"], (step["kind"], toks, step["tokens"])
    assert worst <= 1e-3, worst


def _run_script(model, prompts, decode_steps, seq_ids=None):
    seq_ids = seq_ids or list(range(len(prompts)))
    out = [model.forward(prompts, seq_ids, [])]
    lens = [len(p) for p in prompts]
    for _ in range(decode_steps):
        lens = [n + 1 for n in lens]
        out.append(model.forward([[t] for t in out[-1]], seq_ids, list(lens)))
    return out


@pytest.mark.parametrize("shape", ["TINY", "SMALL64", "SMALL128"])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_forward_matches_oracle_model(tmp_path, shape, dtype):
    """head_dim 32 / 64 / 128 (all kernel specialisations), prompts crossing block and tile
    boundaries, 20 decode steps, both dtypes: identical greedy tokens, close logits."""
    cfg = synth.make_config(**getattr(synth, shape))
    tdtype = torch.float16 if dtype == "float16" else torch.bfloat16
    sd = synth.make_state_dict(cfg, seed=5, dtype=tdtype)
    from swiftllm_amd import LlamaModelConfig
    ecfg = dict(max_blocks_per_seq=32, max_tokens_in_batch=1024, dtype=dtype)
    model = _make_model(tmp_path, cfg, sd, 64, **ecfg)
    ref = RefLlamaModel(LlamaModelConfig(cfg), _engine_config("", **ecfg), sd, tdtype)
    ref.init_kvcache_and_swap(64)
    g = torch.Generator().manual_seed(2)
    prompts = [torch.randint(0, cfg["vocab_size"], (n,), generator=g).tolist() for n in (1, 16, 17, 130, 65)]
    got = _run_script(model, prompts, 20)
    taps = model.post_layer.logits_tap
    # |dlogit| <= atol + rtol*|logit|. Against the CPU oracle the GEMMs differ too (hipBLASLt vs
    # CPU fp32 summation order: 1-ulp flips of 16-bit activations that propagate), so the budget is
    # two ulps of the storage dtype at |logit| ~ 1; the north_star's 1e-3 is held where it is
    # defined — against the reference's own run, test_forward_matches_reference_golden.
    atol, rtol = (2e-3, 2e-3) if dtype == "float16" else (1.6e-2, 1.6e-2)

    def excess(ours, theirs):
        return ((ours.float().cpu() - theirs).abs() - rtol * theirs.abs()).max().item()
    want, worst = [], 0.0
    want.append(ref.forward(prompts, list(range(5)), []))
    worst = max(worst, excess(taps[0], ref.last_logits))
    lens = [len(p) for p in prompts]
    for i in range(20):
        lens = [n + 1 for n in lens]
        # teacher-forced with OUR tokens so one near-tie cannot derail the comparison of later steps
        want.append(ref.forward([[t] for t in got[i]], list(range(5)), list(lens)))
        worst = max(worst, excess(taps[i + 1], ref.last_logits))
    assert worst <= atol, worst
    assert got == want


def test_mixed_batches_free_and_reuse(tmp_path):
    """Piggybacked prefill+decode batches (two-stream path), freeing and re-using sequence slots and
    blocks, vs the oracle model step by step."""
    cfg = synth.make_config(**synth.SMALL64)
    sd = synth.make_state_dict(cfg, seed=9)
    from swiftllm_amd import LlamaModelConfig
    model = _make_model(tmp_path, cfg, sd, 40, max_tokens_in_batch=1024)
    ref = RefLlamaModel(LlamaModelConfig(cfg), _engine_config("", max_tokens_in_batch=1024), sd, torch.float16)
    ref.init_kvcache_and_swap(40)
    g = torch.Generator().manual_seed(4)
    rp = lambda n: torch.randint(0, cfg["vocab_size"], (n,), generator=g).tolist()   # noqa: E731

    def both(ids, sids, dlens):
        a = model.forward(ids, sids, dlens)
        b = ref.forward(ids, sids, dlens)
        d = (model.post_layer.logits_tap[-1].float().cpu() - ref.last_logits).abs()
        assert (d - 2e-3 * ref.last_logits.abs()).max().item() <= 1e-3
        assert a == b
        return a

    t = both([rp(40), rp(7)], [2, 5], [])
    lens = {2: 40, 5: 7}
    for _ in range(3):
        for s in lens:
            lens[s] += 1
        t = both([[t[0]], [t[1]]], [2, 5], [lens[2], lens[5]])
    # a new prompt rides along with the two decoding sequences
    for s in lens:
        lens[s] += 1
    t = both([rp(33), [t[0]], [t[1]]], [0, 2, 5], [lens[2], lens[5]])
    lens[0] = 33
    # sequence 5 finishes: free it on both sides, its blocks must be handed out again (lowest first)
    model.free_seqs_resources([5])
    ref.free_seqs_resources([5])
    assert model.gpu_block_manager.num_free_blocks == ref.gpu_block_manager.num_free_blocks
    del lens[5]
    for s in lens:
        lens[s] += 1
    t = both([rp(50), [t[0]], [t[1]]], [5, 0, 2], [lens[0], lens[2]])
    torch.cuda.synchronize()
    bm, rbm = model.gpu_block_manager, ref.gpu_block_manager
    assert torch.equal(bm.num_seq_allocated_blocks.cpu(), rbm.num_seq_allocated_blocks)
    assert torch.equal(bm.is_block_free.cpu(), rbm.is_block_free)
    for s in (0, 2, 5):
        n = int(rbm.num_seq_allocated_blocks[s])
        assert bm.block_table[s, :n].cpu().tolist() == rbm.block_table[s, :n].tolist()
    assert model.forward([], [], []) == []


def test_swap_out_and_in_preserves_generation(tmp_path):
    """encode -> erase -> decode: swap a sequence out to the host pool, let another sequence overwrite
    the GPU blocks it held, swap it back in (different block ids) and continue decoding: tokens must
    equal an undisturbed run."""
    cfg = synth.make_config(**synth.SMALL64)
    sd = synth.make_state_dict(cfg, seed=6)
    g = torch.Generator().manual_seed(8)
    pa = torch.randint(0, cfg["vocab_size"], (37,), generator=g).tolist()
    pb = torch.randint(0, cfg["vocab_size"], (60,), generator=g).tolist()

    clean = _make_model(tmp_path / "a", cfg, sd, 16)
    want = [x[0] for x in _run_script(clean, [pa], 8, [3])]

    model = _make_model(tmp_path / "b", cfg, sd, 16)
    got = [x[0] for x in _run_script(model, [pa], 3, [3])]
    model.swap_out_seqs([3])
    assert model.gpu_block_manager.num_free_blocks == 16
    assert model.cpu_block_manager.num_free_blocks == 8 - 3
    _run_script(model, [pb], 2, [1])                    # tramples the freed GPU blocks
    model.swap_in_seqs([3])
    assert model.cpu_block_manager.num_free_blocks == 8
    n = len(pa) + 3
    last = got[-1]
    for _ in range(5):
        n += 1
        last = model.forward([[last]], [3], [n])[0]
        got.append(last)
    assert got == want


def test_profile_num_blocks_and_dummy_weights(tmp_path):
    from swiftllm_amd import LlamaModel
    cfg = synth.make_config(**synth.SMALL128)
    synth.write_model_dir(str(tmp_path), cfg)
    model = LlamaModel(_engine_config(str(tmp_path), use_dummy=True, gpu_mem_utilization=0.5,
                                      max_batch_size=4, max_tokens_in_batch=512, dtype="bfloat16"))
    model.load_weights()
    n = model.profile_num_blocks()
    free, total = torch.cuda.mem_get_info()
    block_bytes = 16 * model.model_config.get_kvslot_size(torch.bfloat16)
    assert 0 < n * block_bytes <= 0.5 * total
    model.init_kvcache_and_swap(min(n, 64))
    toks = model.forward([[1, 2, 3, 4, 5]], [0], [])
    assert len(toks) == 1 and 0 <= toks[0] < cfg["vocab_size"]


def test_positions_beyond_the_rope_table_raise_on_the_host(tmp_path):
    """max_position_embeddings 512 (+128 slack): a 700-token prompt must be refused with a Python
    exception, not a device memory fault."""
    cfg = synth.make_config()
    model = _make_model(tmp_path, cfg, synth.make_state_dict(cfg), 64, max_blocks_per_seq=64,
                        max_tokens_in_batch=1024)
    with pytest.raises(RuntimeError, match="rotary table"):
        model.forward([[1] * 700], [0], [])
    assert model.forward([[1, 2, 3]], [0], []) is not None


@pytest.mark.parametrize("mode", ["plain", "piggyback", "hipgraph"])
def test_engine_serving_matches_offline_generation(tmp_path, mode):
    """The control plane over the real data plane: 7 requests of different lengths through Engine
    (continuous batching, max_batch_size 3 so requests queue and join mid-flight; with `piggyback`
    prefills and decodes share a forward) must each produce the tokens an isolated offline greedy
    generation of the same prompt produces."""
    import asyncio
    from swiftllm_amd import Engine, RawRequest
    cfg = synth.make_config(**synth.SMALL64)
    sd = synth.make_state_dict(cfg, seed=9)
    model = _make_model(tmp_path, cfg, sd, 48, max_batch_size=3, max_tokens_in_batch=200,
                        use_hip_graph=(mode == "hipgraph"))
    model.post_layer.logits_tap = None
    g = torch.Generator().manual_seed(4)
    shapes = [(5, 9), (33, 4), (64, 12), (1, 7), (100, 3), (17, 1), (48, 10)]
    prompts = [torch.randint(0, cfg["vocab_size"], (n,), generator=g).tolist() for n, _ in shapes]

    expected = []
    for p, (_, n_out) in zip(prompts, shapes):
        steps = _run_script(model, [p], n_out - 1, seq_ids=[15])
        expected.append([s[0] for s in steps])
        model.free_seqs_resources([15])

    async def serve():
        eng = Engine(model.engine_config, model=model, piggyback=(mode == "piggyback"))
        await eng.initialize()
        loops = asyncio.ensure_future(eng.start_all_event_loops())
        jobs = [asyncio.ensure_future(eng.add_request_and_wait(RawRequest("", n_out, p)))
                for p, (_, n_out) in zip(prompts, shapes)]
        done = await asyncio.wait_for(asyncio.gather(*jobs), timeout=120)
        loops.cancel()
        return eng, [toks for _, toks in done]
    eng, got = asyncio.run(serve())
    assert got == expected
    assert eng.num_forwards < sum(n for _, n in shapes)      # requests really shared forwards
    assert model.gpu_block_manager.num_free_blocks == 48     # everything released


def test_streaming_weight_loader_equals_per_tensor_loader(tmp_path):
    """Pinned-ring streaming safetensors loader: same tensors on the device as the reference's per-tensor path,
    fused [q;k;v] and [up;gate] assembled in place."""
    from swiftllm_amd import LlamaModelConfig
    from swiftllm_amd.worker.weight import load_weights
    cfg = synth.make_config(**synth.SMALL128)
    sd = synth.make_state_dict(cfg, seed=21)
    synth.write_model_dir(str(tmp_path), cfg, sd)
    mc = LlamaModelConfig.load_from_model_path(str(tmp_path))
    a = load_weights(mc, torch.float16, str(tmp_path), device="cuda", fuse_qkv=True, streaming=True)
    b = load_weights(mc, torch.float16, str(tmp_path), device="cuda", fuse_qkv=True, streaming=False)
    for attr in ("wte", "lm_head", "final_norm"):
        assert torch.equal(getattr(a, attr), getattr(b, attr)) and getattr(a, attr).is_cuda
    for la, lb in zip(a.layers, b.layers):
        for attr in ("attn_norm", "qkv_proj", "o_proj", "ffn_norm", "up_gate_proj", "down_proj"):
            assert torch.equal(getattr(la, attr), getattr(lb, attr))


@pytest.mark.parametrize("dtype,copies", [("float16", 4), ("bfloat16", 4), ("bfloat16", 6)],
                         ids=["float16-batch32", "bfloat16-batch32", "bfloat16-batch48"])
def test_full_width_layers_fast_path_equals_reference_op_sequence(tmp_path, dtype, copies):
    """Llama-3-8B layer geometry (hidden 4096, 32/8 heads of 128, FFN 14336; 2 layers, 8k vocabulary so the CPU
    side stays small): here every decode projection really splits K (4-8 slabs), runs the ring kernel, the
    split-K consumers and the attention kernel fed by qkv slabs — none of which the small test models reach. The
    default path must give the tokens of the reference's op sequence (separate q/k/v, every linear on hipBLASLt,
    one kernel per operator), with logits inside the storage dtype's rounding, with hipGraph replay (the default) and
    with eager launches; and replay must be BIT-equal to eager launches at the same flash-decoding split geometry."""
    cfg = synth.make_config(num_hidden_layers=2, hidden_size=4096, num_attention_heads=32, num_key_value_heads=8,
                            intermediate_size=14336, vocab_size=8192, max_position_embeddings=2048,
                            rope_theta=500000.0)
    tdtype = torch.float16 if dtype == "float16" else torch.bfloat16
    sd = synth.make_state_dict(cfg, seed=31, dtype=tdtype)
    g = torch.Generator().manual_seed(8)
    lens = [1, 15, 16, 17, 100, 257, 640, 33] * copies            # batch 32 (one token block) or 48 (medium-batch GEMM), ragged
    prompts = [torch.randint(0, cfg["vocab_size"], (n,), generator=g).tolist() for n in lens]
    base = dict(max_blocks_per_seq=64, max_tokens_in_batch=8192, max_batch_size=48, max_seqs_in_block_table=48,
                dtype=dtype)
    from swiftllm_amd import LlamaModel
    synth.write_model_dir(str(tmp_path), cfg, sd)
    del sd
    seq_ids = list(range(len(prompts)))

    def run(opts, forced=None, bucketed=False):
        """prefill + 6 decode steps; `forced` = token lists to feed instead of the run's own (teacher forcing: one
        near-tie must not make the later steps incomparable)"""
        model = LlamaModel(_engine_config(str(tmp_path), **base, **opts))
        model.load_weights()
        model.init_kvcache_and_swap(48 * 48)
        model._eager_uses_graph_buckets = bucketed
        model.post_layer.logits_tap = []
        tap = model.post_layer.logits_tap
        toks = [model.forward(prompts, seq_ids, [])]
        logits = [tap[-1].float().cpu()]        # copied at once: under hipGraph replay the tapped tensor is reused
        cur = list(lens)
        for step in range(6):
            cur = [n + 1 for n in cur]
            feed = forced[step] if forced is not None else toks[-1]
            toks.append(model.forward([[t] for t in feed], seq_ids, list(cur)))
            logits.append(tap[-1].float().cpu())
        del model
        torch.cuda.empty_cache()
        return toks, logits

    ref_toks, ref_logits = run(dict(fuse_qkv=False, use_skinny_gemm=False, use_hip_graph=False))
    eps = 2.0 ** -10 if dtype == "float16" else 2.0 ** -7
    results = {}
    for name, opts, bucketed in (("hipgraph", dict(), False), ("eager", dict(use_hip_graph=False), False),
                                 ("eager_bucketed", dict(use_hip_graph=False), True)):
        toks, logits = run(opts, forced=ref_toks, bucketed=bucketed)
        results[name] = (toks, logits)
        for step, (a, b) in enumerate(zip(logits, ref_logits)):
            # budget: a few ulps of the storage dtype AT THE SCALE OF THE ROW (16-bit activation flips upstream move
            # small logits by as much as large ones)
            scale = b.abs().amax(dim=1, keepdim=True).clamp(min=1.0)
            excess = ((a - b).abs() - 4 * eps * scale).max().item()
            assert excess <= 0, (name, step, excess)
        # greedy ids: identical except where the reference run itself has a near-tie
        for step, (a, b) in enumerate(zip(toks, ref_toks)):
            for seq, (x, y) in enumerate(zip(a, b)):
                if x != y:
                    top2 = ref_logits[step][seq].topk(2).values
                    assert float(top2[0] - top2[1]) <= 8 * eps * float(top2[0].abs().clamp(min=1.0)), (name, step, seq)
    # Graph replay buckets the flash-decoding split geometry (model._graph_bucket: width rounded to a 1/16..1/32
    # quantum, count to a power of two), so its fp32 summation order may differ from the eager plan's; at the SAME
    # geometry replay and eager launches are the same kernels on the same data: bit-equal logits and tokens.
    assert results["hipgraph"][0] == results["eager_bucketed"][0]
    for step, (a, b) in enumerate(zip(results["hipgraph"][1], results["eager_bucketed"][1])):
        assert torch.equal(a, b), ("graph replay != eager launches at the replay geometry", step)


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("batch", [1, 2])
def test_tiny_batch_decode_path_equals_the_consumer_path(tmp_path, dtype, batch):
    """The tiny_decode_batches switch (EngineConfig.tuning) at Llama-3-8B layer geometry (2 layers): the <= 4-sequence path (projections that
    sum the previous projection's slabs themselves, residual ping-pong) against the same engine with it switched off —
    same greedy tokens over 8 decode steps with and without hipGraph replay, logits within the storage dtype's rounding
    (the only arithmetic difference is the fp32 summation order of the sums of squares)."""
    cfg = synth.make_config(num_hidden_layers=2, hidden_size=4096, num_attention_heads=32, num_key_value_heads=8,
                            intermediate_size=14336, vocab_size=4096, max_position_embeddings=2048, rope_theta=500000.0)
    tdtype = torch.float16 if dtype == "float16" else torch.bfloat16
    sd = synth.make_state_dict(cfg, seed=17, dtype=tdtype)
    g = torch.Generator().manual_seed(4)
    lens = [300, 17, 1, 64][:batch]
    prompts = [torch.randint(0, cfg["vocab_size"], (n,), generator=g).tolist() for n in lens]
    base = dict(max_blocks_per_seq=32, max_tokens_in_batch=512, max_batch_size=4, max_seqs_in_block_table=8, dtype=dtype)
    synth.write_model_dir(str(tmp_path), cfg, sd)
    del sd
    from swiftllm_amd import LlamaModel

    def run(opts, forced=None):
        model = LlamaModel(_engine_config(str(tmp_path), **base, **opts))
        model.load_weights()
        model.init_kvcache_and_swap(64)
        model.post_layer.logits_tap = []
        seq_ids = list(range(batch))
        toks = [model.forward(prompts, seq_ids, [])]
        logits = []
        cur = list(lens)
        for step in range(8):
            cur = [n + 1 for n in cur]
            feed = forced[step] if forced is not None else toks[-1]
            toks.append(model.forward([[t] for t in feed], seq_ids, list(cur)))
            logits.append(model.post_layer.logits_tap[-1].float().cpu())
        del model
        torch.cuda.empty_cache()
        return toks, logits

    # (rows_decode off on both sides: with it on, bfloat16 batches of <= 8 never reach the tiny path — tests/test_gpu_rows.py)
    ref_toks, ref_logits = run(dict(tuning=dict(tiny_decode_batches=False, rows_decode=False)))
    eps = 2.0 ** -10 if dtype == "float16" else 2.0 ** -7
    for opts in (dict(tuning=dict(rows_decode=False)), dict(use_hip_graph=False, tuning=dict(rows_decode=False))):
        toks, logits = run(opts, forced=ref_toks)
        for step, (a, b) in enumerate(zip(logits, ref_logits)):
            scale = b.abs().amax(dim=1, keepdim=True).clamp(min=1.0)
            assert ((a - b).abs() <= 4 * eps * scale).all(), (opts, step, ((a - b).abs() / scale).max().item())
        for step, (x, y) in enumerate(zip(toks, ref_toks)):
            for seq, (tx, ty) in enumerate(zip(x, y)):
                if tx != ty:
                    top2 = ref_logits[step - 1][seq].topk(2).values if step else None
                    assert top2 is not None and float(top2[0] - top2[1]) <= 8 * eps * float(top2[0].abs().clamp(min=1.0))


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_decode_fast_path_survives_realistic_norm_weights_and_residual_outliers(tmp_path, dtype):
    """the deferred-RMSNorm decode path stores round(residual * norm_weight) BEFORE the 1/rms is
    applied. In float16 a residual outlier of 1e3-1e4 times a norm weight of up to 3 leaves the format's range (inf), and
    rows with small rms lose bits to subnormals — the reference's path (rmsnorm.py:59-64) has neither problem, and
    synthetic norm weights of ~1 never show it. The deferred form is therefore bfloat16-only (kernels/rmsnorm.py:
    deferred_norm_ok); this test pins the behaviour: norm weights log-uniform in [0.01, 3], embedding rows with outliers
    of 1e3-1e4, hidden 1024 (every projection on the split-K fast path), both dtypes — finite logits, the oracle's greedy
    ids (per-row near-tie rule), logits within a few storage-dtype ulps of the row scale."""
    from swiftllm_amd import LlamaModelConfig
    cfg = synth.make_config(num_hidden_layers=2, hidden_size=1024, num_attention_heads=8, num_key_value_heads=2,
                            intermediate_size=2048, vocab_size=512, max_position_embeddings=1024)
    tdtype = torch.float16 if dtype == "float16" else torch.bfloat16
    sd = synth.make_state_dict(cfg, seed=21, dtype=tdtype)
    g = torch.Generator().manual_seed(6)
    for name in list(sd):
        if name.endswith("layernorm.weight") or name == "model.norm.weight":
            sd[name] = torch.exp(torch.empty(1024).uniform_(-4.6, 1.1, generator=g)).to(tdtype)      # 0.01 .. 3
    emb = sd["model.embed_tokens.weight"].float()
    rows = torch.randint(0, 512, (64,), generator=g)
    cols = torch.randint(0, 1024, (64,), generator=g)
    emb[rows, cols] = torch.empty(64).uniform_(1e3, 1e4, generator=g) * torch.where(torch.rand(64, generator=g) < 0.5, -1.0, 1.0)
    sd["model.embed_tokens.weight"] = emb.to(tdtype)
    ecfg = dict(max_blocks_per_seq=32, max_tokens_in_batch=1024, dtype=dtype, max_batch_size=8, max_seqs_in_block_table=8)
    model = _make_model(tmp_path, cfg, sd, 64, **ecfg)
    ref = RefLlamaModel(LlamaModelConfig(cfg), _engine_config("", **ecfg), sd, tdtype)
    ref.init_kvcache_and_swap(64)
    # prompts that hit the outlier rows
    prompts = [rows[i * 8:(i + 1) * 8].tolist() + torch.randint(0, 512, (5 + 7 * i,), generator=g).tolist() for i in range(6)]
    seq_ids = list(range(6))
    eps = 2.0 ** -10 if dtype == "float16" else 2.0 ** -7
    want = ref.forward(prompts, seq_ids, [])
    got = model.forward(prompts, seq_ids, [])
    lens = [len(p) for p in prompts]
    for step in range(10):
        a, b = model.post_layer.logits_tap[-1].float().cpu(), ref.last_logits
        assert torch.isfinite(a).all() and torch.isfinite(b).all(), step
        d = (a - b).abs()
        scale = b.abs().amax(dim=1, keepdim=True).clamp(min=1.0)
        assert (d <= 6 * eps * scale).all(), (step, float((d / scale).max()))
        for i, (x, y) in enumerate(zip(got, want)):
            if x != y:
                top2 = b[i].topk(2).values
                assert float(top2[0] - top2[1]) <= 2 * float(d[i].max()), (step, i)
        lens = [n + 1 for n in lens]
        got = model.forward([[t] for t in want], seq_ids, list(lens))       # teacher-forced with the oracle's tokens
        want = ref.forward([[t] for t in want], seq_ids, list(lens))


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_decode_lookahead_changes_nothing_but_the_host_path(tmp_path, dtype):
    """LlamaModel prepares the next decode step's metadata while the GPU runs the current one (model.py:
    _prepare_next_decode) and skips plan + upload when the next call is exactly that step. Same graphs, same kernels, same
    data: tokens and logits must be BIT-equal to the model with the look-ahead off, through block-boundary crossings,
    graph-bucket changes, a call that breaks the prediction (other input tokens), a freed-and-reused sequence slot, a
    prefill in between, and a shrinking batch; and the fast path must actually have been taken."""
    cfg = synth.make_config(**synth.SMALL64)
    tdtype = torch.float16 if dtype == "float16" else torch.bfloat16
    sd = synth.make_state_dict(cfg, seed=13, dtype=tdtype)
    g = torch.Generator().manual_seed(9)
    prompts = [torch.randint(0, cfg["vocab_size"], (n,), generator=g).tolist() for n in (14, 31, 1, 60)]
    extra = torch.randint(0, cfg["vocab_size"], (9,), generator=g).tolist()
    os.environ["SWL_HOST_PROFILE"] = "1"
    try:
        def run(lookahead):
            model = _make_model(tmp_path / ("on" if lookahead else "off"), cfg, sd, 64, max_blocks_per_seq=32,
                                max_tokens_in_batch=512, dtype=dtype)
            model._decode_lookahead = lookahead
            tap = model.post_layer.logits_tap
            trace = []

            def fwd(ids, seqs, lens):
                toks = model.forward(ids, seqs, lens)
                trace.append((toks, tap[-1].float().cpu().clone()))
                return toks
            seqs = [0, 1, 2, 3]
            toks = fwd(prompts, seqs, [])
            lens = [len(p) for p in prompts]
            for step in range(40):          # crosses 16-token block boundaries of every sequence
                lens = [n + 1 for n in lens]
                feed = [[t] for t in toks]
                if step == 7:
                    feed[1] = [(toks[1] + 1) % cfg["vocab_size"]]      # not what was sampled: the prediction must be dropped
                toks = fwd(feed, seqs, list(lens))
            model.free_seqs_resources([2])                                # slot 2 leaves, a new prompt takes it
            toks2 = fwd([extra], [2], [])
            toks[2], lens[2] = toks2[0], len(extra)
            for step in range(6):
                lens = [n + 1 for n in lens]
                toks = fwd([[t] for t in toks], seqs, list(lens))
            model.free_seqs_resources([0])                                # the batch shrinks
            seqs, toks, lens = seqs[1:], toks[1:], lens[1:]
            for step in range(5):
                lens = [n + 1 for n in lens]
                toks = fwd([[t] for t in toks], seqs, list(lens))
            hits = (model._host_prof or {}).get("lookahead_hits", 0.0)
            del model
            torch.cuda.empty_cache()
            return trace, hits
        base, hits_off = run(False)
        fast, hits_on = run(True)
    finally:
        os.environ.pop("SWL_HOST_PROFILE", None)
    assert hits_off == 0 and hits_on >= 40, (hits_off, hits_on)
    assert len(base) == len(fast)
    for i, ((ta, la), (tb, lb)) in enumerate(zip(base, fast)):
        assert ta == tb, i
        assert torch.equal(la, lb), i


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_llama32_1b_geometry_matches_oracle(tmp_path, dtype):
    """The other model family the reference serves (weight.py:157-163, model.py:183-214): Llama-3.2-1B geometry — hidden
    2048, 32 query / 8 kv heads of 64, FFN 8192, dict-style rope_scaling (the reference's home-grown frequency split) and
    the tied lm_head it implies — 2 layers, an 8k vocabulary so the CPU side stays small. Different tile counts and
    K-splits in every decode projection than the 8B shapes the other tests run (N = 2048 / 3072 / 16384), head_dim 64
    attention kernels, ragged batch of 9: greedy ids of the oracle (per-row near-tie rule), logits within a few storage-
    dtype ulps of the row scale, prefill + 12 decode steps, graph replay (default) and eager launches."""
    from swiftllm_amd import LlamaModelConfig
    cfg = synth.make_config(num_hidden_layers=2, hidden_size=2048, num_attention_heads=32, num_key_value_heads=8,
                            intermediate_size=8192, vocab_size=8192, max_position_embeddings=2048, rope_theta=500000.0,
                            rope_scaling=dict(factor=32.0, low_freq_factor=1.0, high_freq_factor=4.0,
                                              original_max_position_embeddings=64, rope_type="llama3"),
                            tie_word_embeddings=True)
    tdtype = torch.float16 if dtype == "float16" else torch.bfloat16
    sd = synth.make_state_dict(cfg, seed=77, dtype=tdtype)
    g = torch.Generator().manual_seed(12)
    lens = [1, 15, 16, 17, 100, 257, 640, 33, 500]
    prompts = [torch.randint(0, cfg["vocab_size"], (n,), generator=g).tolist() for n in lens]
    seq_ids = list(range(len(lens)))
    ecfg = dict(max_blocks_per_seq=48, max_tokens_in_batch=2048, max_batch_size=16, max_seqs_in_block_table=16, dtype=dtype)
    ref = RefLlamaModel(LlamaModelConfig(cfg), _engine_config("", **ecfg), sd, tdtype, tied_lm_head=True)
    ref.init_kvcache_and_swap(16 * 48)
    want, want_logits = [ref.forward(prompts, seq_ids, [])], [ref.last_logits.clone()]
    cur = list(lens)
    for _ in range(12):
        cur = [n + 1 for n in cur]
        want.append(ref.forward([[t] for t in want[-1]], seq_ids, list(cur)))
        want_logits.append(ref.last_logits.clone())
    eps = 2.0 ** -10 if dtype == "float16" else 2.0 ** -7
    for opts in (dict(), dict(use_hip_graph=False)):
        model = _make_model(tmp_path / ("graph" if not opts else "eager"), cfg, sd, 16 * 48, **ecfg, **opts)
        assert model.weight.lm_head.data_ptr() == model.weight.wte.data_ptr() or torch.equal(model.weight.lm_head, model.weight.wte)
        cur = list(lens)
        for s in range(13):
            ids = prompts if s == 0 else [[t] for t in want[s - 1]]      # teacher-forced with the oracle's tokens
            if s:
                cur = [n + 1 for n in cur]
            got = model.forward(ids, seq_ids, [] if s == 0 else list(cur))
            a, b = model.post_layer.logits_tap[-1].float().cpu(), want_logits[s]
            d = (a - b).abs()
            scale = b.abs().amax(dim=1, keepdim=True).clamp(min=1.0)
            assert (d <= 4 * eps * scale).all(), (opts, s, float((d / scale).max()))
            for i, (x, y) in enumerate(zip(got, want[s])):
                if x != y:
                    top2 = b[i].topk(2).values
                    assert float(top2[0] - top2[1]) <= 2 * float(d[i].max()), (opts, s, i)
        del model
        torch.cuda.empty_cache()


@pytest.mark.parametrize("batch", [100, 200])
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_large_decode_batches_take_the_wide_kernels_and_match_the_oracle(tmp_path, batch, dtype, monkeypatch):
    """Decode batches of 65..256 sequences (r04: csrc/gemm_wide.hip): the projections the measured policy gives to
    swl_gemm_packed_wide really go through it — as split-K slabs into the add+norm consumer and the slab-fed attention kernel where K is
    split, with the SiLU-gate in the epilogue up to 128 tokens — and the forward still matches the CPU oracle, teacher-
    forced over 3 steps, on a model wide enough for every K-split rule (hidden 2048, 16/4 heads of 128, FFN 4096)."""
    monkeypatch.setenv("SWIFTLLM_ROUTE_TUNE", "table")      # (these widths are not in the measured table: pin it, the test
    # asserts WHICH kernels run; kernels/route_tune.py would otherwise time both sides on this box)
    from swiftllm_amd import LlamaModelConfig, _hip
    cfg = synth.make_config(num_hidden_layers=2, hidden_size=2048, num_attention_heads=16, num_key_value_heads=4,
                            intermediate_size=4096, vocab_size=512, max_position_embeddings=512)
    tdtype = torch.float16 if dtype == "float16" else torch.bfloat16
    sd = synth.make_state_dict(cfg, seed=9, dtype=tdtype)
    ecfg = dict(max_blocks_per_seq=8, max_tokens_in_batch=batch * 24, max_batch_size=batch,
                max_seqs_in_block_table=batch + 8, dtype=dtype, use_hip_graph=False)
    model = _make_model(tmp_path, cfg, sd, batch * 3 + 8, **ecfg)
    ref = RefLlamaModel(LlamaModelConfig(cfg), _engine_config("", **ecfg), sd, tdtype, dense_decode_attention=True)
    ref.init_kvcache_and_swap(batch * 3 + 8)
    calls = []
    real = _hip.call

    def spy(name, *a):
        calls.append(name)
        return real(name, *a)
    monkeypatch.setattr(_hip, "call", spy)
    g = torch.Generator().manual_seed(3)
    prompts = [torch.randint(0, cfg["vocab_size"], (3 + i % 17,), generator=g).tolist() for i in range(batch)]
    seq_ids = list(range(batch))
    got = [model.forward(prompts, seq_ids, [])]
    want = [ref.forward(prompts, seq_ids, [])]
    lens = [len(p) for p in prompts]
    mant = 10 if dtype == "float16" else 7
    worst, mism, off_tie = 0.0, 0, []
    del calls[:]
    for i in range(3):
        lens = [n + 1 for n in lens]
        got.append(model.forward([[t] for t in got[-1]], seq_ids, list(lens)))
        want.append(ref.forward([[t] for t in got[-2]], seq_ids, list(lens)))       # teacher-forced with OUR tokens
        d = (model.post_layer.logits_tap[-1].float().cpu() - ref.last_logits).abs().amax(dim=1)
        row_ulp = torch.exp2(torch.floor(torch.log2(ref.last_logits.abs().amax(dim=1))) - mant)
        worst = max(worst, float((d / row_ulp).max()))
        top2 = ref.last_logits.topk(2, dim=1).values
        for r, (a, b) in enumerate(zip(got[-1], want[-1])):
            if a != b:      # a greedy id may differ only on a near-tie of the oracle: top-2 gap within twice the row's distance
                mism += 1
                if float(top2[r, 0] - top2[r, 1]) > 2 * float(d[r]):
                    off_tie.append((i, r, float(top2[r, 0] - top2[r, 1]), float(d[r])))
    # the bar of tests/test_gpu_parity_fullwidth.py: within 3 ulps of the storage dtype at the row's scale of the CPU oracle
    # (hipBLASLt / MFMA vs CPU fp32 summation order: 1-ulp flips of 16-bit activations that propagate; measured r04: 1-2 ulps)
    assert worst <= 3.0, worst
    assert not off_tie and mism <= 3 * batch // 50, (mism, off_tie)
    wide = [c for c in calls if c.startswith("swl_gemm_packed_wide")]
    assert "swl_gemm_packed_wide_partial" in wide, sorted(set(calls))        # K-split projections feed the consumers
    assert "swl_splitk_fused_add_rmsnorm" in calls
    # up to 128 tokens the qkv slabs go straight into the attention kernel's prologue (rotary + KV store + attention in one
    # launch); beyond, this model's qkv projection is the library's and the separate rotary+store launch runs
    assert ("swl_paged_attn_decode_qkv" in calls) == (batch <= 128), sorted(set(calls))
    assert ("swl_rotary_store_kv_decode" in calls or "swl_splitk_rotary_store_kv_decode" in calls) == (batch > 128)
    assert ("swl_gemm_packed_wide_silu_gate" in wide) == (batch <= 128), sorted(set(wide))


def test_a_batch_rounded_up_to_its_bucket_keeps_the_bits_of_its_exact_size(tmp_path):
    """Six sequences of more than 512 tokens over 40 kv heads: 240 workgroups of attention, 320 in the bucket of eight that a replay runs. The
    inert ones are no second round: tokens and logits of a replayed step are those of an eager step of six, bit for bit."""
    cfg = synth.make_config(num_hidden_layers=2, hidden_size=1280, num_attention_heads=40, num_key_value_heads=40,
                            intermediate_size=1024, vocab_size=512, max_position_embeddings=1024)
    sd = synth.make_state_dict(cfg, seed=12, dtype=torch.bfloat16)
    g = torch.Generator().manual_seed(4)
    prompts = [torch.randint(0, cfg["vocab_size"], (600 + 17 * i,), generator=g).tolist() for i in range(6)]
    runs = {}
    for graph in (False, True):
        model = _make_model(tmp_path / f"g{int(graph)}", cfg, sd, 6 * 48 + 8, max_blocks_per_seq=64, max_tokens_in_batch=8192,
                            max_batch_size=8, max_seqs_in_block_table=16, dtype="bfloat16", use_hip_graph=graph)
        toks = _run_script(model, prompts, 4)
        runs[graph] = (toks, [t.clone() for t in model.post_layer.logits_tap])
        if graph:
            assert {k[0] for k in model._decode_graphs} == {8}
        del model
        torch.cuda.empty_cache()
    assert runs[True][0] == runs[False][0]
    for a, b in zip(runs[True][1], runs[False][1]):
        assert torch.equal(a, b)


@pytest.mark.parametrize("batch", [100, 200])
def test_large_decode_batches_replay_their_hip_graph_bit_for_bit(tmp_path, batch, monkeypatch):
    """The product default (hipGraph replay) at decode batches beyond 64: the captured graph — wide GEMMs, their slabs into
    the add+norm consumer and the slab-fed attention prologue — gives the tokens AND the logits of eager launches, bit for
    bit, over 4 steps (bfloat16, the geometry of the test above)."""
    monkeypatch.setenv("SWIFTLLM_ROUTE_TUNE", "table")      # (two model instances must route alike whatever a timing says)
    cfg = synth.make_config(num_hidden_layers=2, hidden_size=2048, num_attention_heads=16, num_key_value_heads=4,
                            intermediate_size=4096, vocab_size=512, max_position_embeddings=512)
    sd = synth.make_state_dict(cfg, seed=9, dtype=torch.bfloat16)
    g = torch.Generator().manual_seed(3)
    prompts = [torch.randint(0, cfg["vocab_size"], (3 + i % 17,), generator=g).tolist() for i in range(batch)]
    runs = {}
    for graph in (False, True):
        model = _make_model(tmp_path / f"g{int(graph)}", cfg, sd, batch * 3 + 8, max_blocks_per_seq=8,
                            max_tokens_in_batch=batch * 24, max_batch_size=batch, max_seqs_in_block_table=batch + 8,
                            dtype="bfloat16", use_hip_graph=graph)
        toks = _run_script(model, prompts, 4)
        runs[graph] = (toks, [t.clone() for t in model.post_layer.logits_tap])
        if graph:
            assert len(model._decode_graphs) >= 1
        del model
        torch.cuda.empty_cache()
    assert runs[True][0] == runs[False][0]
    for a, b in zip(runs[True][1], runs[False][1]):
        assert torch.equal(a, b)


def test_graphs_are_recaptured_after_the_flash_decoding_scratch_grows(tmp_path):
    """A server meets this: decode graphs exist (one short sequence), then a step needs a larger flash-decoding scratch (more
    sequences, split contexts) — the captured graphs point into the old buffer and are dropped. The shared private pool must
    be dropped WITH them: a pool whose last graph is gone sits on the caching allocator's books with use_count 0, and the
    next capture into the same id tripped `it->second->use_count > 0` (r06: tools/serve_bench.py --sweep crashed the model
    thread with it; r05 introduced the shared pool). The steps after the drop replay fresh captures and equal eager launches."""
    cfg = synth.make_config(num_hidden_layers=2, hidden_size=1024, num_attention_heads=8, num_key_value_heads=2,
                            intermediate_size=2048, vocab_size=512, max_position_embeddings=1024)
    sd = synth.make_state_dict(cfg, seed=23, dtype=torch.bfloat16)
    g = torch.Generator().manual_seed(4)
    lens0 = [300, 280, 310, 290, 305, 270]
    prompts = [torch.randint(0, cfg["vocab_size"], (n,), generator=g).tolist() for n in lens0]
    runs = {}
    for graph in (False, True):
        model = _make_model(tmp_path / f"g{int(graph)}", cfg, sd, 200, max_blocks_per_seq=32, max_tokens_in_batch=2048,
                            max_batch_size=8, max_seqs_in_block_table=16, dtype="bfloat16", use_hip_graph=graph)
        seq_ids = list(range(len(prompts)))
        toks = model.forward(prompts, seq_ids, [])
        lens = list(lens0)
        out = []
        for step in range(2):                   # one sequence alone: a graph (and a small scratch) exists
            lens[0] += 1
            toks[0] = model.forward([[toks[0]]], [0], [lens[0]])[0]
            out.append(toks[0])
        pools = []
        if graph:
            assert len(model._decode_graphs) >= 1
            pools.append(model._graph_pool)
            scratch0 = model._scratch.numel() if model._scratch is not None else 0
        for step in range(3):                   # all six: a larger scratch, every graph dropped, new captures
            lens = [n + 1 for n in lens]
            toks = model.forward([[t] for t in toks], seq_ids, list(lens))
            out.append(list(toks))
        if graph:
            assert model._scratch is not None and model._scratch.numel() > scratch0, "the scenario did not grow the scratch"
            assert model._graph_pool is not None and model._graph_pool != pools[0]
        runs[graph] = (out, [t.clone() for t in model.post_layer.logits_tap])
        del model
        torch.cuda.empty_cache()
    assert runs[True][0] == runs[False][0]
    for a, b in zip(runs[True][1], runs[False][1]):
        assert a.shape == b.shape and torch.equal(a, b)


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_decode_batch_buckets_replay_equals_exact_eager_launches(tmp_path, dtype):
    """hipGraph replay rounds a pure-decode batch up to its bucket with inert rows (worker/model.py: _decode_batch_bucket):
    a batch that shrinks 7 -> 6 -> 5 -> 4 -> 3 as sequences finish replays ONE captured graph (batch 8) and returns, step
    for step, the tokens AND the logits of exact-size eager launches, bit for bit (every decode kernel is row-independent
    and treats a length-0 sequence as a no-op); the finished sequences' blocks are freed and the KV of the survivors is
    untouched by the inert rows (they store nothing)."""
    cfg = synth.make_config(num_hidden_layers=2, hidden_size=1024, num_attention_heads=8, num_key_value_heads=2,
                            intermediate_size=2048, vocab_size=512, max_position_embeddings=512)
    tdtype = torch.float16 if dtype == "float16" else torch.bfloat16
    sd = synth.make_state_dict(cfg, seed=21, dtype=tdtype)
    g = torch.Generator().manual_seed(8)
    lens0 = [40, 3, 17, 64, 5, 33, 9]
    prompts = [torch.randint(0, cfg["vocab_size"], (n,), generator=g).tolist() for n in lens0]
    runs = {}
    for graph in (False, True):
        model = _make_model(tmp_path / f"g{int(graph)}", cfg, sd, 96, max_blocks_per_seq=16, max_tokens_in_batch=512,
                            max_batch_size=8, max_seqs_in_block_table=16, dtype=dtype, use_hip_graph=graph)
        seq_ids = list(range(len(prompts)))
        toks = model.forward(prompts, seq_ids, [])
        lens = list(lens0)
        out = [list(toks)]
        for step in range(10):
            if step in (2, 4, 6, 8):            # the last sequence finishes
                model.free_seqs_resources([seq_ids[-1]])
                seq_ids, lens, toks = seq_ids[:-1], lens[:-1], toks[:-1]
            lens = [n + 1 for n in lens]
            toks = model.forward([[t] for t in toks], seq_ids, list(lens))
            assert len(toks) == len(seq_ids)
            out.append(list(toks))
        logits = [t.clone() for t in model.post_layer.logits_tap]
        runs[graph] = (out, logits)
        if graph:
            # one BATCH bucket (8) for the five batch sizes; the split geometry of these short, shrinking sequences adds its
            # own key dimension (_graph_bucket)
            assert {k[0] for k in model._decode_graphs} == {8} and model.graph_captures <= 2, list(model._decode_graphs)
        del model
        torch.cuda.empty_cache()
    assert runs[True][0] == runs[False][0]
    assert len(runs[True][1]) == len(runs[False][1])
    for a, b in zip(runs[True][1], runs[False][1]):
        assert a.shape == b.shape and torch.equal(a, b)
