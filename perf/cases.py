"""The work whose speed counts: what a program that serves models with this package has it do.

Every case is one pass of a worker (`swiftllm_amd.build_model`), driven as an offline program or the engine drives it:

  * `prompts`: whole prompts of several requests in one step, the logits of each prompt's last token, the requests released;
  * `decode`:  `steps` tokens generated one after the other for a batch of running requests, each step fed with the tokens
               that the one before it sampled (contexts are in the caches before the pass);
  * `mixed`:   one step that takes new prompts beside one decoded token of every running request.

All seven designs that the package serves take part, at the layer sizes and with the mechanisms that `bench.py
--compare-designs` gives them (LLaMA: Llama-3-8B's layer), in a stack of four layers, so that every kind of a design's layers
is in it. Weights are random and drawn from a fixed seed (a model is loaded once and serves many batches), prompts from the
case's seed. Sublayers add a quarter of the stream's size or less, as in trained stacks, and the head answers a token with one
particular successor far above the rest, so that sampled tokens do not hang on rounding.
"""
import math
import shutil
import tempfile
import weakref

import torch

F64 = torch.float64
SIZES = {       # width, heads, kv heads, head size, feed-forward width
    "small": dict(w=1024, H=8, G=2, d=128, ff=4096),
    "medium": dict(w=2048, H=16, G=4, d=128, ff=8192),
    "wide": dict(w=4096, H=32, G=8, d=128, ff=14336),
}
VOCAB, DEPTH, POSITIONS, RANK = 32000, 4, 4096, 512
DECAY_RANK = 64
DESIGNS = ("llama", "kekapel", "lorulix", "rosilix", "ratilorn", "rokevik", "vafozen")


def listed():
    def case(name, design, size, kind, dtype="bfloat16", prompts=0, prompt_len=0, batch=0, context=0, steps=0):
        return dict(name=name, design=design, size=size, kind=kind, dtype=dtype, prompts=prompts, prompt_len=prompt_len,
                    batch=batch, context=context, steps=steps)
    return [
        # one user's chat with a Llama-3-8B-shaped model: latency of a token
        case("llama_chat", "llama", "wide", "decode", batch=1, context=700, steps=4),
        # a server under its ordinary load: 32 requests at about 1k tokens
        case("llama_serve", "llama", "wide", "decode", batch=32, context=1088, steps=4),
        # the same server with its batch full
        case("llama_full", "llama", "wide", "decode", batch=120, context=600, steps=4),
        # prompts of five requests arriving together, the reference's own precision
        case("llama_prompts", "llama", "wide", "prompts", "float16", prompts=5, prompt_len=1023),
        # a step of a busy server: new prompts beside running requests
        case("llama_mixed", "llama", "wide", "mixed", prompts=2, prompt_len=900, batch=29, context=1088),
        # documents in, the first token out: head mixing, windows, PolyNorm and experts
        case("kekapel_prompts", "kekapel", "medium", "prompts", prompts=3, prompt_len=1500),
        # the same for the delta rule beside attention with a distance bias
        case("lorulix_prompts", "lorulix", "small", "prompts", prompts=4, prompt_len=2048),
        # generation for a batch: differential and latent attention
        case("rosilix_serve", "rosilix", "medium", "decode", batch=32, context=1024, steps=4),
        # many short prompts: sigmoid attention, state-space recurrence, grouped experts
        case("ratilorn_prompts", "ratilorn", "medium", "prompts", prompts=11, prompt_len=333),
        # prompts through latent attention, keys as values, minGRU and experts in every layer
        case("rokevik_prompts", "rokevik", "small", "prompts", prompts=4, prompt_len=2000),
        # new prompts beside running requests on a design with recurrent state
        case("vafozen_mixed", "vafozen", "small", "mixed", prompts=2, prompt_len=1000, batch=30, context=777),
        # a few requests of a small recurrent model generating in true fp32: launches and latency
        case("lorulix_chat", "lorulix", "small", "decode", "float32", batch=3, context=513, steps=4),
    ]


def draw(rng):
    """Any design, kind, size and type of the above; lengths and batches over their logarithm."""
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    design = rng.choice(DESIGNS)
    kind = rng.choice(("prompts", "prompts", "decode", "decode", "mixed"))
    if design == "llama":
        size, dtype = "wide", rng.choice(("bfloat16", "float16"))
    else:
        dtype = rng.choice(("bfloat16", "bfloat16", "float16", "float32"))
        size = "small" if dtype == "float32" else rng.choice(("small", "medium"))
    case = dict(design=design, size=size, kind=kind, dtype=dtype, prompts=0, prompt_len=0, batch=0, context=0, steps=0)
    if kind != "decode":
        case["prompts"] = log(1, 12)
        case["prompt_len"] = log(8, min(2048, (500 if dtype == "float32" else 5000) // case["prompts"]))
    if kind != "prompts":
        most = 3 if dtype == "float32" else 100 if (design, dtype) == ("llama", "bfloat16") else 32
        case["batch"], case["context"] = log(1, most), log(16, {3: 500, 32: 1100, 100: 700}[most])
        case["steps"] = 4 if kind == "decode" else 0
    return case


# ---- models ----------------------------------------------------------------------------------------------------------------
def config_of(design, size):
    """config.json of the design at this size."""
    s = SIZES[size]
    w, H, G, d, ff = (s[k] for k in ("w", "H", "G", "d", "ff"))
    half, root = d // 2, d ** -0.5
    heads = dict(dim=d, vdim=d, heads=H, kv_heads=G, scale=root)
    dense = dict(kind="dense", ff=ff)
    if design == "llama":
        return dict(model_type="llama", hidden_act="silu", rms_norm_eps=1e-5, rope_scaling=None, tie_word_embeddings=False,
                    num_hidden_layers=DEPTH, hidden_size=w, num_attention_heads=H, num_key_value_heads=G, intermediate_size=ff,
                    vocab_size=VOCAB, max_position_embeddings=POSITIONS, rope_theta=500000.0)
    top = dict(architecture=design.capitalize(), max_positions=POSITIONS, norm=dict(eps=1e-6), vocab=VOCAB, width=w)
    ssm = dict(heads=H, vdim=d, state=d, groups=1, conv=4, norm_groups=1)
    latent = dict(heads=H, dim=d, rot_dim=half, vdim=d, kv_rank=RANK, rot=dict(base=10000.0, dims=half), scale=(d + half) ** -0.5)
    moe = dict(kind="moe", expert=dict(ff=ff // 4), router=dict(experts=8, top=2), shared=dict(ff=ff // 4))
    kinds, mlps = [], [dense, moe]
    if design == "kekapel":
        top.update(embedding=dict(scale=1.0), residual_mult=0.5)
        kinds = [("attention", dict(heads, mask=dict(size=1024), softcap=30.0))]
        mlps = [dense, dict(kind="moe", expert=dict(ff=ff // 4, limit=7.0), router=dict(experts=8, top=2))]
    elif design == "lorulix":
        top.update(canon=dict(taps=3))
        attn = dict(heads, bias_max=1024, q_temp=dict(coef=0.1, every=256))
        kinds = [("attention", attn), ("delta", dict(dim=d, vdim=d, heads=H, kv_heads=G, conv=4)),
                 ("attention", dict(attn, kv_from=0)), ("attention", attn)]
        mlps = [dict(dense, limit=7.0), dict(moe, router=dict(experts=8, top=2, scale=1.0))]
    elif design == "rosilix":
        top.update(embedding=dict(scale=1.0))
        dif = dict(heads=H, kv_heads=G, dim=half, vdim=d, diff=0.3, mask=dict(size=1024), rot=dict(base=10000.0, dims=half),
                   scale=half ** -0.5)
        kinds = [("latent_attention", latent), ("attention", dif), ("attention", dif), ("latent_attention", dict(latent, kv_from=0))]
        mlps = [dense]
    elif design == "ratilorn":
        top.update(logit_scale=0.5)
        kinds = [("attention", dict(heads, v_mix=True)), ("parallel", dict(left=heads, right=ssm)), ("parallel", dict(left=heads, right=ssm))]
        mlps = [dense, dict(moe, router=dict(experts=8, top=2, groups=dict(count=4, keep=2)))]
    elif design == "rokevik":
        top.update(norm=dict(eps=1e-6, groups=2), streams=2, logit_softcap=30.0)
        lat = dict(latent, mask=dict(size=1024), rot=dict(base=200000.0, dims=half, scaling=dict(factor=4.0, original=2048, fast=24.0,
                                                                                           slow=2.0)))
        kinds = [("attention", dict(heads, softcap=30.0, rot=dict(base=10000.0, dims=half))), ("latent_attention", lat),
                 ("latent_attention", lat), ("mingru", dict(width=H * d))]
        mlps = [moe]
    else:
        top.update(embedding=dict(scale=1.0))
        kinds = [("parallel", dict(left=dict(heads, mask=dict(size=1024)), right=dict(heads=H, dim=d, vdim=d, tau=16.0),
                                   left_scale=0.8, right_scale=1.1)),
                 ("parallel_2", dict(left=dict(heads, conv=4, softcap=30.0, rot=dict(base=10000.0, dims=d)),
                                     right=dict(heads=H, dim=d), left_scale=0.8, right_scale=1.1)),
                 ("mamba2", ssm)]
        mlps = [dense]
    top["layers"] = [dict(type=kinds[i % len(kinds)][0], mixer=kinds[i % len(kinds)][1], mlp=mlps[i % len(mlps)]) for i in range(DEPTH)]
    return top


def tensor_specs(design, size):
    """name -> (shape, how it is drawn) of every tensor of a checkpoint. How: (mean, standard deviation), "rand" with (low, high),
    or "in": N(0, gain^2 / inputs)."""
    c, out = config_of(design, size), {}
    s = SIZES[size]
    w = s["w"]

    def mat(name, rows, cols, gain=1.0):
        out[name] = ((rows, cols), (0.0, gain / math.sqrt(cols)))

    def vec(name, n, mean=0.0, std=0.1):
        out[name] = (n if isinstance(n, tuple) else (n,), (mean, std))

    def uni(name, n, low, high):
        out[name] = (n if isinstance(n, tuple) else (n,), (low, high, "rand"))

    if design == "llama":
        vec("model.embed_tokens.weight", (VOCAB, w), 0.0, 1.0)
        vec("lm_head.weight", (VOCAB, w), 0.0, 1.0 / math.sqrt(w))
        vec("model.norm.weight", w, 1.0)
        for i in range(DEPTH):
            p = f"model.layers.{i}."
            vec(p + "input_layernorm.weight", w, 1.0)
            vec(p + "post_attention_layernorm.weight", w, 1.0)
            for n, rows, cols, gain in (("self_attn.q_proj", s["H"] * s["d"], w, 1.0), ("self_attn.k_proj", s["G"] * s["d"], w, 1.0),
                                        ("self_attn.v_proj", s["G"] * s["d"], w, 1.0), ("self_attn.o_proj", w, s["H"] * s["d"], 0.5),
                                        ("mlp.up_proj", s["ff"], w, 1.0), ("mlp.gate_proj", s["ff"], w, 1.0),
                                        ("mlp.down_proj", w, s["ff"], 0.3)):
                mat(p + n + ".weight", rows, cols, gain)
        return out
    vec("embed", (VOCAB, w), 0.0, 1.0)
    if design in ("kekapel", "lorulix", "ratilorn"):
        vec("pos", (POSITIONS, w), 0.0, 0.3)
    if design != "ratilorn":
        vec("head", (VOCAB, w), 0.0, 1.0 / math.sqrt(w))
    off = 0.0 if design in ("lorulix", "ratilorn", "vafozen") else 1.0       # (norm weights stored around zero)
    vec("final.norm", w, off)
    if design == "kekapel":
        vec("final.norm.b", w)
    for i, L in enumerate(c["layers"]):
        p, mx, mlp = f"l{i}.", L["mixer"], L["mlp"]
        m = p + "mix."
        for q in ("1", "2"):
            if design == "vafozen" and q == "2":
                continue
            vec(f"{p}norm{q}", w, off if design != "ratilorn" else -0.75, 0.1 if design != "ratilorn" else 0.05)
            if design in ("kekapel", "lorulix", "rosilix"):
                vec(f"{p}norm{q}b", w, {"kekapel": 0.5, "lorulix": -0.75, "rosilix": 0.25}[design], 0.05)
            if design == "kekapel":
                vec(f"{p}norm{q}.b", w)
                vec(f"{p}norm{q}b.b", w, 0.0, 0.02)
            if design == "lorulix":
                vec(f"{p}canon{q}", (w, c["canon"]["taps"]), 0.0, 0.3)
                mat(f"{p}rg{q}", w, w)
                vec(f"{p}rg{q}.b", w, 0.0, 0.5)
            if design == "rokevik":
                uni(f"{p}hc{q}.in", 2, 0.4, 0.6)
                uni(f"{p}hc{q}.out", 2, 0.15, 0.25)
                uni(f"{p}hc{q}.mix", (2, 2), 0.0, 0.05)
        if design == "ratilorn" and L["type"] == "parallel":
            vec(m + "left.out", w, 1.0)
            vec(m + "right.out", w, 1.0)
        small = 0.25 if design == "vafozen" else 1.0
        if L["type"] in ("parallel", "parallel_2", "mamba2") or (L["type"] == "attention" and design != "rosilix"):
            a, q = (mx["left"], m + "left.") if "left" in mx else (mx, m)
            if L["type"] != "mamba2":
                H, G, d, e = a["heads"], a["kv_heads"], a["dim"], a["vdim"]
                kv = a.get("kv_from") is None
                names = [("q", H * d)] + ([("k", G * d)] if kv else []) + ([("v", G * e)] if kv and design != "rokevik" else [])
                for n, rows in names:
                    mat(q + n, rows, w)
                    if design in ("ratilorn", "rokevik", "vafozen"):
                        vec(q + n + ".b", rows, 0.0, 0.2)
                    if "conv" in a:
                        vec(q + n + ".conv", (rows, a["conv"]), 0.0, 0.5)
                if design == "lorulix":
                    vec(q + "q.norm", H * d, 1.0)
                    if kv:
                        vec(q + "k.norm", G * d, 1.0)
                    vec(q + "rel", (32, H), 0.0, 1.0)
                elif design in ("kekapel", "rokevik") or L["type"] == "parallel":
                    vec(q + "q.norm", d, 1.0)
                    vec(q + "k.norm", d, 1.0)
                if design == "kekapel":
                    vec(q + "talk", (H, H), 0.0, 0.3 / math.sqrt(H))
                if design == "ratilorn" and L["type"] == "attention":
                    uni(q + "vmix", (), 0.2, 0.6)
                    uni(q + "r1", H, 0.2, 0.8)
                    uni(q + "r2", H, 0.05, 0.5)
                    vec(q + "talk", (H, H), 0.0, 0.3 / math.sqrt(H))
                    vec(q + "pb", H, -3.0, 0.5)
                if design == "rokevik":
                    uni(q + "temp", H, 0.6, 1.4)
                    mat(q + "g", H, w)
                if design in ("rokevik", "vafozen"):
                    vec(q + "o.b", w, 0.0, 0.02)
                if L["type"] == "parallel_2":
                    mat(q + "g", H * e, w)
                mat(q + "o", w, H * e, small)
        if L["type"] == "attention" and design == "rosilix":
            H, G, d, e = mx["heads"], mx["kv_heads"], mx["dim"], mx["vdim"]
            mat(m + "q", H * 2 * d, w)
            mat(m + "k", G * 2 * d, w)
            mat(m + "v", G * e, w)
            for n in ("lq1", "lk1", "lq2", "lk2"):
                vec(m + n, d, 0.0, 0.2)
            mat(m + "g", H, w)
            mat(m + "o", w, H * e)
        if L["type"] == "latent_attention":
            H, d, dr, e, r = mx["heads"], mx["dim"], mx["rot_dim"], mx["vdim"], mx["kv_rank"]
            mat(m + "q", H * (d + dr), w)
            if mx.get("kv_from") is None:
                mat(m + "dkv", r + dr, w)
                vec(m + "dkv.norm", r, 1.0)
            mat(m + "uk", H * d, r)
            mat(m + "uv", H * e, r)
            if design == "rosilix":
                vec(m + "sink", H, 0.0, 1.0)
            mat(m + "g", H, w)
            mat(m + "o", w, H * e)
        if L["type"] == "mingru":
            n = mx["width"]
            for k in "zx":
                mat(m + k, n, w)
                vec(m + k + ".b", n, -1.5 if k == "z" else 0.0, 1.0 if k == "z" else 0.3)
            mat(m + "g", n, w)
            mat(m + "o", w, n)
        if L["type"] == "delta":
            H, G, d, e = mx["heads"], mx["kv_heads"], mx["dim"], mx["vdim"]
            for n, rows in (("q", G * d), ("k", G * d), ("v", H * e)):
                mat(m + n, rows, w)
                vec(m + n + ".conv", (rows, mx["conv"]), 0.0, 0.5)
            mat(m + "b", H, w)
            mat(m + "a", H, w)
            uni(m + "A_log", H, -1.0, 0.5)
            uni(m + "dt_bias", H, -4.0, -1.0)
            vec(m + "norm", e, 1.0)
            mat(m + "g", H * e, w)
            mat(m + "o", w, H * e)
        if L["type"] == "mamba2" or (design == "ratilorn" and L["type"] == "parallel"):
            r, q = (mx, m) if L["type"] == "mamba2" else (mx["right"], m + "right.")
            inner, gn = r["heads"] * r["vdim"], r["groups"] * r["state"]
            mat(q + "in", 2 * inner + 2 * gn + r["heads"], w)
            vec(q + "conv", (inner + 2 * gn, r["conv"]), 0.0, 0.5)
            vec(q + "conv.b", inner + 2 * gn, 0.0, 0.2)
            uni(q + "dt_bias", r["heads"], -4.0, -1.0)
            uni(q + "A_log", r["heads"], -1.0, 0.5)
            uni(q + "D", r["heads"], 0.5, 1.5)
            vec(q + "norm", inner, 1.0)
            mat(q + "o", w, inner, small)
        if design == "vafozen" and L["type"] != "mamba2":
            r, q = mx["right"], m + "right."
            n = r["heads"] * r["dim"]
            if L["type"] == "parallel":
                for k in "qkvg":
                    mat(q + k, n, w)
                vec(q + "norm", r["vdim"], 1.0)
                mat(q + "a1", DECAY_RANK, w)
                mat(q + "a2", n, DECAY_RANK, 2.0)
                vec(q + "a2.b", n, 0.0, 0.3)
            else:
                for k in "rkvgw":
                    uni(f"{q}mu.{k}", w, 0.0, 1.0)
                for k in "rkvg":
                    mat(q + k, n, w)
                mat(q + "w1", DECAY_RANK, w)
                mat(q + "w2", n, DECAY_RANK)
                uni(q + "w0", n, -6.0, -1.0)
                vec(q + "u", (r["heads"], r["dim"]), 0.5, 0.5)
                vec(q + "norm", n, 1.0)
            mat(q + "o", w, n, small)
        f = p + "mlp."
        if mlp["kind"] == "dense":
            if design == "vafozen":
                small = 0.4
            for n in ("up",) if design in ("kekapel", "rosilix") else ("gate", "up"):
                mat(f + n, mlp["ff"], w)
            mat(f + "down", w, mlp["ff"], small)
            if design == "kekapel":
                vec(f + "act", 4, 0.5, 0.1)
        else:
            E, ef = mlp["router"]["experts"], mlp["expert"]["ff"]
            names = ("up",) if design == "lorulix" else ("gate", "up")
            for u in [f"e{e}." for e in range(E)] + (["shared."] if "shared" in mlp else []):
                for n in names:
                    mat(f + u + n, ef, w)
                mat(f + u + "down", w, ef)
            mat(f + "router", E, w, 2.0)
            if design == "kekapel":
                vec(f + "router.b", E, 0.0, 0.3)
            if design == "lorulix":
                mat(f + "shared.sg", 1, w)
            if design == "ratilorn":
                vec(f + "correction", E, 0.0, 0.1)
    return out


def successor(tokens):
    """The token that the head of every design but Ratilorn's (whose head is its embedding) puts far above the rest."""
    return (tokens * 7919 + 13) % VOCAB


def weights_of(design, size, dtype):
    """Random weights with the checkpoint's names and type, on the GPU; the same ones at every call."""
    kind = {"float16": torch.float16}.get(dtype, torch.bfloat16)
    g = torch.Generator(device="cuda").manual_seed(20)
    W = {}
    for name, (shape, how) in tensor_specs(design, size).items():
        if how[-1] == "rand":
            t = torch.rand(shape, generator=g, device="cuda") * (how[1] - how[0]) + how[0]
        else:
            t = torch.randn(shape, generator=g, device="cuda") * how[1] + how[0]
        if name.endswith("talk") or (design == "rokevik" and name.endswith(".mix")):
            t += torch.eye(shape[0], device="cuda") * (0.9 if name.endswith(".mix") else 1.0)
        W[name] = t.to(kind)
    embed, head = ("model.embed_tokens.weight", "lm_head.weight") if design == "llama" else ("embed", "head")
    if head in W:
        ids = torch.arange(VOCAB, device="cuda")
        W[head].index_add_(0, successor(ids), (W[embed].float() / math.sqrt(W[embed].shape[1])).to(kind))
    return W


class _Model:
    """A loaded worker and room for the batches of several states: sequence ids in sets that states take and give back."""
    SETS = 4

    def __init__(self, case):
        import json
        import os
        from safetensors.torch import save_file
        from swiftllm_amd import EngineConfig, build_model
        design, size, dtype = case["design"], case["size"], case["dtype"]
        self.set = 160 if (design, dtype) == ("llama", "bfloat16") else 48      # requests of one state, at most
        path = tempfile.mkdtemp(prefix="perf_cases_", dir="/dev/shm" if os.path.isdir("/dev/shm") else None)
        try:
            with open(os.path.join(path, "config.json"), "w", encoding="utf-8") as f:
                json.dump(config_of(design, size), f)
            W = {k: v.cpu() for k, v in weights_of(design, size, dtype).items()}
            save_file(W, os.path.join(path, "model.safetensors"))
            self.worker = build_model(EngineConfig(
                model_path=path, use_dummy=False, block_size=16, gpu_mem_utilization=0.9, num_cpu_blocks=0,
                max_seqs_in_block_table=self.SETS * self.set, max_blocks_per_seq=POSITIONS // 16,
                max_batch_size=64 if design == "llama" and self.set == 48 else 128 if design == "llama" else self.SETS * self.set,
                max_tokens_in_batch=8192, dtype=dtype))
            self.worker.load_weights()
        finally:
            shutil.rmtree(path)
        self.worker.init_kvcache_and_swap(self.SETS * (80000 + 8192 + self.set * 32) // 16)
        self.taps = []
        self.free_sets = list(range(self.SETS))

    def give_back(self, taken, running):
        self.worker.free_seqs_resources(running)
        self.free_sets.append(taken)


_loaded = {}        # at most one model: key -> _Model


class _State:
    """One batch of requests on a loaded worker."""

    def __init__(self, case, seed):
        key = (case["design"], case["size"], case["dtype"])
        if key not in _loaded:
            _loaded.clear()
            torch.cuda.empty_cache()
            _loaded[key] = _Model(case)
        self.case, self.model = case, _loaded[key]
        taken = self.model.free_sets.pop(0)
        base = taken * self.model.set
        self.new, self.contexts = inputs_of(case, seed)
        self.running = [base + i for i in range(case["batch"])]
        self.new_ids = [base + case["batch"] + i for i in range(case["prompts"])]
        self.lens = [len(c) - 1 for c in self.contexts]     # (tokens in the caches)
        weakref.finalize(self, self.model.give_back, taken, list(self.running))
        at = 0
        while at < len(self.running):       # the contexts of the running requests, up to 8192 tokens a step
            to, total = at, 0
            while to < len(self.running) and total + self.lens[to] <= 8192:
                total += self.lens[to]
                to += 1
            self.model.worker.forward([c[:-1] for c in self.contexts[at:to]], self.running[at:to], [])
            at = to
        del self.model.taps[:]


def inputs_of(case, seed):
    """-> (new prompts, contexts of the running requests with the token that they go on from), lists of token ids. Lengths are
    ragged: from a half to one and a half of the case's (at most 2048), drawn with the tokens."""
    g = torch.Generator().manual_seed(int(seed) * 2 + 1)

    def some(count, length):
        lens = (torch.rand(count, generator=g) + 0.5).mul(length).long().clamp(1, 2048)
        if count:       # (the sum stays the case's: what a pass costs does not hang on the seed)
            lens = (lens.float() * (count * length / lens.sum())).long().clamp(1, 2048)
        return [torch.randint(0, VOCAB, (int(n),), generator=g).tolist() for n in lens]
    prompts, contexts = some(case["prompts"], case["prompt_len"]), some(case["batch"], case["context"])
    # a pass of several steps starts again where it started, which a worker allows inside a block of 16 tokens only
    contexts = [c[:len(c) - max(0, len(c) % 16 + case["steps"] - 16)] for c in contexts]
    return prompts, [c + [int(torch.randint(0, VOCAB, (1,), generator=g))] for c in contexts]


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    from swiftllm_amd.worker.batch_plan import StepEntry
    case, worker, taps = state.case, state.model.worker, state.model.taps
    if case["design"] == "llama":
        worker.post_layer.logits_tap = taps
    else:
        worker.logits_tap = taps if case["kind"] == "decode" else None
    if case["kind"] == "decode":
        tokens, sampled = [c[-1] for c in state.contexts], []
        for i in range(case["steps"]):
            tokens = worker.forward([[t] for t in tokens], state.running, [n + 1 + i for n in state.lens])
            sampled.append(tokens)
        out = {"logits": list(taps), "tokens": [torch.tensor(s) for s in sampled]}
        del taps[:]
        return out
    lasts = [[c[-1]] for c in state.contexts]
    if case["design"] == "llama":
        worker.forward(state.new + lasts, state.new_ids + state.running, [n + 1 for n in state.lens])
        logits = taps[0]
    else:
        entries = [StepEntry(i, p, 0, (len(p) - 1,)) for i, p in zip(state.new_ids, state.new)]
        entries += [StepEntry(i, t, n, (0,)) for i, t, n in zip(state.running, lasts, state.lens)]
        logits = worker.step(entries)
    del taps[:]
    worker.free_seqs_resources(state.new_ids)
    return {"logits": logits}


# ---- what a pass cannot do without -----------------------------------------------------------------------------------------
def work(case):
    """Weights read once (of the experts those that can be chosen), cached keys, values and states read and written once, tokens'
    logits written; multiply-adds of the products, of every visible (query, key) pair and of the recurrences."""
    specs = tensor_specs(case["design"], case["size"])
    c, e = config_of(case["design"], case["size"]), 4 if case["dtype"] == "float32" else 2
    s = SIZES[case["size"]]
    P, n, B, ctx = case["prompts"], case["prompt_len"], case["batch"], case["context"]
    steps = max(1, case["steps"])
    rows = P * n + B                    # tokens a step
    wanted = P + B
    token_w, last_w, expert_w = 0, 0, 0
    for name, (shape, _) in specs.items():
        size = math.prod(shape) if shape else 1
        if name in ("embed", "pos", "model.embed_tokens.weight"):
            continue
        if name in ("head", "lm_head.weight"):
            last_w += size
        elif ".mlp.e" in name:
            expert_w += size
        elif len(shape) == 2:
            token_w += size
    if case["design"] == "ratilorn":
        last_w = VOCAB * s["w"]
    used = min(1.0, rows * 2 / 8)
    nbytes = e * (token_w + last_w + expert_w * used + rows * s["w"] + wanted * VOCAB)
    flops = 2.0 * (token_w * rows + last_w * wanted + expert_w * rows / 4)

    def pairs(window):
        """visible pairs of the new prompts and of the running requests, and cached tokens read"""
        k = min(n, window or n)
        cached = B * (min(ctx, window) if window else ctx)
        return P * (n * k - k * (k - 1) / 2) + cached, cached
    for L in (c.get("layers") or [dict(type="llama", mixer=dict(heads=s["H"], kv_heads=s["G"], dim=s["d"], vdim=s["d"]))] * DEPTH):
        mx = L["mixer"]
        a = mx.get("left", mx)
        if "scale" in a or L["type"] == "llama":
            pr, cached = pairs((a.get("mask") or {}).get("size", 0))
            if L["type"] == "latent_attention":     # (the smaller of: all heads' keys and values from the latent rows, or folded)
                H, qk, v, kv = a["heads"], a["dim"] + a["rot_dim"], a["vdim"], a["kv_rank"] + a["rot_dim"]
            else:
                maps = 2 if "diff" in a else 1
                H, qk, v = a["heads"], a["dim"] * maps, a["vdim"] * maps
                kv = a["kv_heads"] * (a["dim"] * maps + (0 if c.get("architecture") == "Rokevik" else a["vdim"]))
            flops += 2.0 * pr * H * (qk + v) + (2.0 * pr * H * H if c.get("architecture") == "Kekapel" else 0.0)
            nbytes += e * kv * (cached + rows)
        r = mx.get("right", mx if L["type"] in ("mamba2", "delta") else None)
        if r is not None:
            st = r["heads"] * r.get("state", r.get("dim")) * r.get("vdim", r.get("dim"))
            flops += rows * st * (6.0 if L["type"] == "delta" else 4.0)
            nbytes += 4 * st * (P + 2 * B)
        if L["type"] == "mingru":
            nbytes += 4 * mx["width"] * (P + 2 * B)
    return {"bytes": nbytes * steps, "flops": flops * steps}


def tolerance(case):
    """About four times the distance of the logits to the same pass in 64 bits, measured over all designs: 0.0057 at most in
    bfloat16, 0.0007 in float16, 1e-6 in float32 (relative, 2-norm). Sampled tokens are the same ones."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-3}
    if case["dtype"] == "float16":
        return {"rel": 0.004, "max": 0.1}
    return {"rel": 0.02, "max": 0.5}


# ---- the same passes in 64 bits --------------------------------------------------------------------------------------------
def _unit(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


def _conv(u, w):
    """u [B, T, C], w [C, taps]: causal, the last column multiplies the current token."""
    out = torch.zeros_like(u)
    for j in range(w.shape[1]):
        back = w.shape[1] - 1 - j
        if back < u.shape[1]:
            out[:, back:] += u[:, :u.shape[1] - back] * w[:, j]
    return out


def _frequencies(rot):
    dims, base = rot["dims"], rot["base"]
    f, sc = [base ** (-2.0 * i / dims) for i in range(dims // 2)], rot.get("scaling")
    if not sc:
        return f, 1.0
    lo, hi = (dims * math.log(sc["original"] / (2 * math.pi * sc[k])) / (2 * math.log(base)) for k in ("fast", "slow"))
    lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), dims - 1)
    ramps = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(dims // 2)]
    return [fi / sc["factor"] * r + fi * (1 - r) for fi, r in zip(f, ramps)], 0.1 * math.log(sc["factor"]) + 1.0


def _rotate(x, rot, pairs=False):
    """x [B, T, heads, d]; pairs: neighbouring elements turn together, else element i with element i + dims / 2."""
    if not rot:
        return x
    f, mult = _frequencies(rot)
    half = rot["dims"] // 2
    ang = torch.arange(x.shape[1], dtype=F64, device=x.device)[:, None] * torch.tensor(f, dtype=F64, device=x.device)
    c, s = (torch.cos(ang) * mult)[:, None, :], (torch.sin(ang) * mult)[:, None, :]
    turned, rest = x[..., :2 * half], x[..., 2 * half:]
    u, v = (turned[..., 0::2], turned[..., 1::2]) if pairs else (turned[..., :half], turned[..., half:])
    a, b = u * c - v * s, v * c + u * s
    turned = torch.stack((a, b), -1).flatten(-2) if pairs else torch.cat((a, b), -1)
    return torch.cat((turned, rest), -1)


def _attend(q, k, v, scores=None, window=0, chunk=0, sink=None, weights=None):
    """q [B, T, H, d], k [B, T, G, d], v [B, T, G, e] -> [B, T, H, e]. scores(s): what becomes of q k^T [H, T, T]; weights(s): in
    the place of the softmax."""
    T, H = q.shape[1], q.shape[2]
    i, j = torch.arange(T, device=q.device)[:, None], torch.arange(T, device=q.device)[None]
    see = j <= i
    if window:
        see &= i - j < window
    if chunk:
        see &= i // chunk == j // chunk
    out = []
    for b in range(q.shape[0]):
        kb, vb = (x[b].transpose(0, 1).repeat_interleave(H // x.shape[2], 0) for x in (k, v))
        s = q[b].transpose(0, 1) @ kb.transpose(1, 2).contiguous()
        s = scores(s, (i - j).clamp(min=0)) if scores else s
        if weights:
            p = weights(s, see)
        else:
            s = s.masked_fill(~see, -math.inf)
            if sink is not None:
                p = torch.softmax(torch.cat((s, sink[:, None, None].expand(-1, T, 1)), -1), -1)[..., :-1]
            else:
                p = torch.softmax(s, -1)
        out.append((p @ vb).transpose(0, 1))
    return torch.stack(out)


def _scan(q, k, v, decay, bonus=None, beta=None):
    """S <- decay S + k u^T and o = S^T q, token by token; u = v, with beta: the delta rule's correction; with a bonus: o from the
    state before the token plus diag(bonus) k v^T. q, k [B, T, H, d], v [B, T, H, e], decay [B, T, H, d or 1]."""
    S = torch.zeros(*q.shape[:1], *q.shape[2:], v.shape[-1], dtype=F64, device=q.device)
    out = torch.empty_like(v)
    for t in range(q.shape[1]):
        kt, vt, qt, dt = k[:, t, :, :, None], v[:, t, :, None], q[:, t, :, None], decay[:, t, :, :, None]
        if bonus is not None:
            kv = kt * vt
            out[:, t] = (qt @ (S + bonus[..., None] * kv))[..., 0, :]
            S = dt * S + kv
            continue
        S = dt * S
        if beta is not None:
            vt = beta[:, t, :, None, None] * (vt - kt.transpose(-1, -2) @ S)
        S = S + kt * vt
        out[:, t] = (qt @ S)[..., 0, :]
    return out


def _cap(s, c):
    return c * torch.tanh(s / c) if c else s


class _Exact:
    def __init__(self, design, size, dtype):
        self.c, self.design = config_of(design, size), design
        self.W = weights_of(design, size, dtype)
        self.eps = self.c["norm"]["eps"] if design != "llama" else 1e-5

    def w(self, name):
        return self.W[name].to(F64)

    def lin(self, x, name, bias=True):
        y = x @ self.w(name).T
        return y + self.w(name + ".b") if bias and name + ".b" in self.W else y

    def heads(self, x, name, n):
        return self.lin(x, name).unflatten(-1, (n, -1))

    # -- mixers
    def attention(self, h, m, mx, i):
        D, eps = self.design, self.eps
        H, G, T = mx["heads"], mx["kv_heads"], h.shape[1]
        scale, rot = mx["scale"], mx.get("rot")
        q = self.heads(h, m + "q", H)
        if D == "lorulix":
            q = (_unit(q.flatten(-2), eps) * self.w(m + "q.norm")).unflatten(-1, (H, -1))
            t = mx["q_temp"]
            pos = torch.arange(T, dtype=F64, device=h.device)
            q = q * (1 + t["coef"] * torch.log(torch.floor((pos + 1) / t["every"]) + 1))[:, None, None]
            if "kv_from" not in mx:
                k = _unit(self.lin(h, m + "k"), eps) * self.w(m + "k.norm")
                self.cache[i] = k.unflatten(-1, (G, -1)), self.heads(h, m + "v", G)
            k, v = self.cache[mx.get("kv_from", i)]
            rel, far = self.w(m + "rel"), mx["bias_max"]
            half = rel.shape[0] // 2
            row = torch.tensor([n if n < half else min(rel.shape[0] - 1, half + math.floor(math.log(n / half) / math.log(far / half)
                                                                                          * (rel.shape[0] - half)))
                                for n in range(T)], device=h.device)
            o = _attend(q, k, v, lambda s, dist: s * scale + rel[row[dist]].permute(2, 0, 1))
            return self.lin(o.flatten(-2), m + "o")
        k = self.heads(h, m + "k", G)
        if D == "ratilorn":
            v = self.lin(h, m + "v")
            lam = self.w(m + "vmix")
            v = v if self.v_first is None else (1 - lam) * v + lam * self.v_first
            self.v_first = v if self.v_first is None else self.v_first
            r1, r2, pb = (self.w(m + n)[:, None, None] for n in ("r1", "r2", "pb"))
            talk = self.w(m + "talk")

            def mixed(s, see):
                return torch.einsum("hg,gij->hij", talk, torch.sigmoid(s) * see)
            o = _attend(_unit(q, eps), _unit(k, eps), v.unflatten(-1, (G, -1)), weights=mixed,
                        scores=lambda s, dist: s * scale - r1 * torch.log(1 + r2 * dist) + pb)
            return self.lin(o.flatten(-2), m + "o")
        v = self.heads(h, m + ("k" if D == "rokevik" else "v"), G)      # (Rokevik: the keys before their norm and rotation)
        if m + "q.norm" in self.W:
            q, k = _unit(q, eps) * self.w(m + "q.norm"), _unit(k, eps) * self.w(m + "k.norm")
        if "conv" in mx:
            q, k, v = (_conv(x.flatten(-2), self.w(m + n + ".conv")).unflatten(-1, (x.shape[2], -1)) for n, x in zip("qkv", (q, k, v)))
        q, k = _rotate(q, rot), _rotate(k, rot)
        size, cap = (mx.get("mask") or {}).get("size", 0), mx.get("softcap", 0.0)
        extra = None
        if D == "kekapel":
            talk = self.w(m + "talk")
            extra = lambda s, dist: torch.einsum("hg,gij->hij", talk, _cap(s * scale, cap))       # noqa: E731
        elif D == "rokevik":
            temp = self.w(m + "temp")[:, None, None]
            extra = lambda s, dist: _cap(s * scale * temp, cap)      # noqa: E731
        elif D == "vafozen" and "mask" in mx:
            slope = torch.tensor([2.0 ** (-8.0 * (n + 1) / H) for n in range(H)], dtype=F64, device=h.device)[:, None, None]
            extra = lambda s, dist: s * scale - slope * dist     # noqa: E731
        else:
            extra = lambda s, dist: _cap(s * scale, cap)      # noqa: E731
        o = _attend(q, k, v, extra, **{"chunk" if D == "vafozen" else "window": size})
        if D == "rokevik":
            o = o * torch.sigmoid(h @ self.w(m + "g").T)[..., None]
        elif D == "vafozen" and "conv" in mx:
            o = o * torch.sigmoid(h @ self.w(m + "g").T).unflatten(-1, (H, -1))
        return self.lin(o.flatten(-2), m + "o")

    def differential(self, h, m, mx):
        H, G = mx["heads"], mx["kv_heads"]
        q, k = (_rotate(self.heads(h, m + n, 2 * x), mx["rot"], pairs=True) for n, x in (("q", H), ("k", G)))
        v = self.heads(h, m + "v", G)
        maps = [_attend(q[:, :, t::2], k[:, :, t::2], v, lambda s, dist: s * mx["scale"], chunk=mx["mask"]["size"]) for t in (0, 1)]
        dot = [float((self.w(m + "lq" + n) * self.w(m + "lk" + n)).sum()) for n in "12"]
        o = maps[0] - (math.exp(dot[0]) - math.exp(dot[1]) + mx["diff"]) * maps[1]
        o = _unit(o, self.eps) * (1 - mx["diff"]) * torch.sigmoid(h @ self.w(m + "g").T)[..., None]
        return self.lin(o.flatten(-2), m + "o")

    def latent(self, h, m, mx, i):
        H, d, r, pairs = mx["heads"], mx["dim"], mx["kv_rank"], self.design == "rosilix"
        q = self.heads(h, m + "q", H)
        q = torch.cat((q[..., :d], _rotate(q[..., d:], mx["rot"], pairs)), -1)
        if "kv_from" not in mx:
            z = self.lin(h, m + "dkv")
            self.cache[i] = _unit(z[..., :r], self.eps) * self.w(m + "dkv.norm"), _rotate(z[..., None, r:], mx["rot"], pairs)
        c, kr = self.cache[mx.get("kv_from", i)]
        k = torch.cat((self.heads(c, m + "uk", H), kr.expand(-1, -1, H, -1)), -1)
        o = _attend(q, k, self.heads(c, m + "uv", H), lambda s, dist: s * mx["scale"], window=(mx.get("mask") or {}).get("size", 0),
                    sink=self.w(m + "sink") if m + "sink" in self.W else None)
        return self.lin((o * torch.sigmoid(h @ self.w(m + "g").T)[..., None]).flatten(-2), m + "o")

    def min_gru(self, h, m, mx, i):
        z, u = torch.sigmoid(self.lin(h, m + "z")), self.lin(h, m + "x")
        cand, S, out = torch.where(u >= 0, u + 0.5, torch.sigmoid(u)), torch.zeros_like(z[:, 0]), torch.empty_like(z)
        for t in range(z.shape[1]):
            S = (1 - z[:, t]) * S + z[:, t] * cand[:, t]
            out[:, t] = S
        return self.lin(out * _silu(self.lin(h, m + "g")), m + "o")

    def delta(self, h, m, mx, i):
        H, G, d = mx["heads"], mx["kv_heads"], mx["dim"]
        q, k, v = (_silu(_conv(self.lin(h, m + n), self.w(m + n + ".conv"))).unflatten(-1, (x, -1)) for n, x in
                   (("q", G), ("k", G), ("v", H)))
        q, k = (x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6) for x in (q, k))
        q, k = (x.repeat_interleave(H // G, 2) for x in (q * d ** -0.5, k))
        decay = torch.exp(-torch.exp(self.w(m + "A_log")) * torch.nn.functional.softplus(self.lin(h, m + "a") + self.w(m + "dt_bias")))
        o = _scan(q, k, v, decay[..., None], beta=torch.sigmoid(self.lin(h, m + "b")))
        o = _unit(o, self.eps) * self.w(m + "norm") * _silu(self.heads(h, m + "g", H))
        return self.lin(o.flatten(-2), m + "o")

    def state_space(self, h, m, r):
        H, P, N = r["heads"], r["vdim"], r["state"]
        inner = H * P
        z, xbc, dt = self.lin(h, m + "in").split((inner, inner + 2 * N, H), -1)
        xbc = _silu(_conv(xbc, self.w(m + "conv")) + self.w(m + "conv.b"))
        x, b, c = xbc.split((inner, N, N), -1)
        x = x.unflatten(-1, (H, P))
        dt = torch.nn.functional.softplus(dt + self.w(m + "dt_bias"))
        decay = torch.exp(-torch.exp(self.w(m + "A_log")) * dt)[..., None]
        y = _scan(c[..., None, :].expand(-1, -1, H, -1), b[..., None, :] * dt[..., None], x, decay) + self.w(m + "D")[:, None] * x
        return self.lin(_unit(y.flatten(-2) * _silu(z), self.eps) * self.w(m + "norm"), m + "o")

    def parallel(self, h, m, mx, i):
        if self.design == "ratilorn":
            left, right = self.attention_plain(h, m + "left.", mx["left"]), self.state_space(h, m + "right.", mx["right"])
            return 0.5 * (_unit(left, self.eps) * self.w(m + "left.out") + _unit(right, self.eps) * self.w(m + "right.out"))
        left, r, p = self.attention(h, m + "left.", mx["left"], i), mx["right"], m + "right."
        H, d = r["heads"], r["dim"]
        if "tau" in r:
            q, k, v = (self.heads(h, p + n, H) for n in "qkv")
            decay = torch.sigmoid(self.lin(self.lin(h, p + "a1"), p + "a2")).pow(1.0 / r["tau"]).unflatten(-1, (H, -1))
            o = _unit(_scan(q * d ** -0.5, k, v, decay), self.eps) * self.w(p + "norm")
            right = self.lin(o.flatten(-2) * _silu(self.lin(h, p + "g")), p + "o")
        else:
            prev = torch.cat((torch.zeros_like(h[:, :1]), h[:, :-1]), 1)
            mix = {n: h + (prev - h) * self.w(f"{p}mu.{n}") for n in "rkvgw"}
            q, k, v = (self.heads(mix[n], p + n, H) for n in "rkv")
            decay = torch.exp(-torch.exp(self.lin(torch.tanh(self.lin(mix["w"], p + "w1")), p + "w2") + self.w(p + "w0")))
            o = _unit(_scan(q, k, v, decay.unflatten(-1, (H, -1)), bonus=self.w(p + "u")), self.eps).flatten(-2)
            right = self.lin(o * self.w(p + "norm") * _silu(self.lin(mix["g"], p + "g")), p + "o")
        return mx["left_scale"] * left + mx["right_scale"] * right

    def attention_plain(self, h, m, mx):
        """Ratilorn's softmax attention: biased projections, normed heads."""
        q, k, v = (self.heads(h, m + n, x) for n, x in (("q", mx["heads"]), ("k", mx["kv_heads"]), ("v", mx["kv_heads"])))
        q, k = _unit(q, self.eps) * self.w(m + "q.norm"), _unit(k, self.eps) * self.w(m + "k.norm")
        return self.lin(_attend(q, k, v, lambda s, dist: s * mx["scale"]).flatten(-2), m + "o")

    def mixer(self, h, L, p, i):
        m, mx = p + "mix.", L["mixer"]
        if L["type"] == "attention":
            return self.differential(h, m, mx) if self.design == "rosilix" else self.attention(h, m, mx, i)
        if L["type"] == "mamba2":
            return self.state_space(h, m, mx)
        return {"latent_attention": self.latent, "mingru": self.min_gru, "delta": self.delta, "parallel": self.parallel,
                "parallel_2": self.parallel}[L["type"]](h, m, mx, i)

    # -- feed-forwards
    def unit(self, h, f, lim=0.0):
        if f + "gate" not in self.W:
            return self.lin(torch.relu(self.lin(h, f + "up")) ** 2, f + "down")
        g, u = self.lin(h, f + "gate"), self.lin(h, f + "up")
        if lim:
            g, u = g.clamp(max=lim), u.clamp(-lim, lim)
            return self.lin(g * torch.sigmoid(1.702 * g) * (u + 1), f + "down")
        return self.lin(_silu(g) * u, f + "down")

    def feed_forward(self, h, mlp, f):
        D = self.design
        if mlp["kind"] == "dense":
            if D == "kekapel":
                z, a = self.lin(h, f + "up"), self.w(f + "act")
                return self.lin(a[0] * _unit(z, self.eps) + a[1] * _unit(z ** 2, self.eps) + a[2] * _unit(z ** 3, self.eps) + a[3],
                                f + "down")
            return self.unit(h, f, mlp.get("limit", 0.0))
        r = mlp["router"]
        z = self.lin(h, f + "router")
        if D == "kekapel":
            val, idx = z.topk(r["top"], -1)
            wt = torch.softmax(val, -1)
        elif D == "lorulix":
            wt, idx = torch.softmax(z, -1).topk(r["top"], -1)
            wt = wt * r["scale"]
        elif D == "ratilorn":
            s = torch.sigmoid(z)
            c = s + self.w(f + "correction")
            groups = c.unflatten(-1, (r["groups"]["count"], -1))
            kept = groups.topk(min(2, groups.shape[-1]), -1).values.sum(-1).topk(r["groups"]["keep"], -1).indices
            keep = torch.zeros(groups.shape[:-1], dtype=torch.bool, device=h.device).scatter_(-1, kept, True)
            idx = c.masked_fill(~keep.repeat_interleave(groups.shape[-1], -1), -math.inf).topk(r["top"], -1).indices
            wt = s.gather(-1, idx)
            wt = wt / (wt.sum(-1, keepdim=True) + 1e-20)
        else:
            idx = torch.sigmoid(z).topk(r["top"], -1).indices
            wt = torch.sigmoid(z).gather(-1, idx)
        out = torch.zeros_like(h)
        for x in range(r["experts"]):
            share = (wt * (idx == x)).sum(-1, keepdim=True)
            rows = share[..., 0] != 0
            hx, sx = h[rows], share[rows]
            y = self.unit(sx * hx, f"{f}e{x}.") if D == "rokevik" else sx * self.unit(hx, f"{f}e{x}.", mlp["expert"].get("limit", 0.0))
            out[rows] += y
        if "shared" in mlp:
            sh = self.unit(h, f + "shared.")
            out = out + (torch.sigmoid(self.lin(h, f + "shared.sg")) * sh if D == "lorulix" else sh)
        return out

    # -- stacks
    def llama(self, x):
        c, eps = self.c, self.eps
        H, G = c["num_attention_heads"], c["num_key_value_heads"]
        d = c["hidden_size"] // H
        rot = dict(base=c["rope_theta"], dims=d)
        for i in range(DEPTH):
            p = f"model.layers.{i}."
            h = _unit(x, eps) * self.w(p + "input_layernorm.weight")
            q, k, v = (self.heads(h, f"{p}self_attn.{n}_proj.weight", y) for n, y in (("q", H), ("k", G), ("v", G)))
            o = _attend(_rotate(q, rot), _rotate(k, rot), v, lambda s, dist: s * d ** -0.5)
            x = x + self.lin(o.flatten(-2), p + "self_attn.o_proj.weight")
            h = _unit(x, eps) * self.w(p + "post_attention_layernorm.weight")
            x = x + self.lin(_silu(self.lin(h, p + "mlp.gate_proj.weight")) * self.lin(h, p + "mlp.up_proj.weight"), p + "mlp.down_proj.weight")
        return _unit(x, eps) * self.w("model.norm.weight")

    def norm(self, x, name):
        if self.design == "kekapel":
            mu = x.mean(-1, keepdim=True)
            return (x - mu) / torch.sqrt(((x - mu) ** 2).mean(-1, keepdim=True) + self.eps) * self.w(name) + self.w(name + ".b")
        g = self.c["norm"].get("groups", 1)
        y = _unit(x.unflatten(-1, (g, -1)), self.eps).flatten(-2)
        return y * ((1.0 if self.design in ("lorulix", "ratilorn", "vafozen") else 0.0) + self.w(name))

    def sublayer(self, x, p, q, f):
        """The stream after one sublayer f of layer p (q: "1" the mixer, "2" the feed-forward)."""
        D = self.design
        if D == "ratilorn":
            return x + self.norm(f(x), f"{p}norm{q}")
        if D == "rokevik":
            h = self.norm((self.w(f"{p}hc{q}.in")[:, None, None, None] * x).sum(0), f"{p}norm{q}")
            y, mix, out = f(h), self.w(f"{p}hc{q}.mix"), self.w(f"{p}hc{q}.out")
            return torch.stack([sum(mix[s, t] * x[s] for s in range(2)) + out[t] * y for t in range(2)])
        h = self.norm(x, f"{p}norm{q}")
        if D == "lorulix":
            gate = torch.sigmoid(self.lin(h, f"{p}rg{q}"))
            return x + self.norm(f(h + _conv(h, self.w(f"{p}canon{q}"))) * gate, f"{p}norm{q}b")
        return x + (self.c["residual_mult"] if D == "kekapel" else 1.0) * self.norm(f(h), f"{p}norm{q}b")

    def logits(self, tokens, at):
        """tokens [B, T] (rows padded at their ends), at: (rows, positions) whose logits are wanted."""
        self.cache, self.v_first = {}, None
        D = self.design
        x = self.w("model.embed_tokens.weight" if D == "llama" else "embed")[tokens]
        if "pos" in self.W:
            x = x + self.w("pos")[:tokens.shape[1]]
        if D == "llama":
            return self.llama(x)[at] @ self.w("lm_head.weight").T
        x = torch.stack((x, x)) if D == "rokevik" else x
        for i, L in enumerate(self.c["layers"]):
            p = f"l{i}."
            if D == "vafozen":
                h = self.norm(x, p + "norm1")
                x = x + self.mixer(h, L, p, i) + self.feed_forward(h, L["mlp"], p + "mlp.")
                continue
            x = self.sublayer(x, p, "1", lambda h: self.mixer(h, L, p, i))
            x = self.sublayer(x, p, "2", lambda h: self.feed_forward(h, L["mlp"], p + "mlp."))
        x = self.norm(x.sum(0) if D == "rokevik" else x, "final.norm")[at]
        if D == "ratilorn":
            return x @ self.w("embed").T * self.c["logit_scale"]
        return _cap(x @ self.w("head").T, self.c.get("logit_softcap", 0.0))


@torch.no_grad()
def exact(case, seed):
    new, contexts = inputs_of(case, seed)
    model = _Exact(case["design"], case["size"], case["dtype"])
    follow = (lambda t: t) if case["design"] == "ratilorn" else successor
    steps = case["steps"]
    rows = [list(p) for p in new] + [list(c) for c in contexts]
    ends = [len(r) - 1 for r in rows]
    sampled = []
    for i in range(steps):
        sampled.append(torch.tensor([follow(r[-1]) for r in rows]))
        for r, t in zip(rows, sampled[-1].tolist()):
            r.append(t)
    group, got = max(1, 12000 // max(len(r) for r in rows)), []
    for a in range(0, len(rows), group):        # (a few rows at a time: the score matrices of a whole batch are large)
        part = rows[a:a + group]
        tokens = torch.zeros(len(part), max(len(r) for r in part), dtype=torch.long, device="cuda")
        for n, r in enumerate(part):
            tokens[n, :len(r)] = torch.tensor(r)
        n = torch.arange(len(part), device="cuda")[:, None].expand(-1, max(1, steps))
        at = torch.tensor(ends[a:a + group], device="cuda")[:, None] + torch.arange(max(1, steps), device="cuda")
        got.append(model.logits(tokens, (n.flatten(), at.flatten())).unflatten(0, (len(part), -1)))
    logits = torch.cat(got)
    if not steps:
        return {"logits": logits[:, 0]}
    return {"logits": [logits[:, i].contiguous() for i in range(steps)], "tokens": sampled}
