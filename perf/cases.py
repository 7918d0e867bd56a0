"""The work whose speed counts: what users of this package have it do, through its public entry points.

A case is a ``kind`` with its sizes:

  mlp           the sparse MLP module alone: neuron selection, fc1, fc2, the predictor for the next layer
  layers        sixteen decode steps (one back-fill window) of consecutive sparse blocks, from a HIP graph
  opt_generate  greedy generation of an OPT-shaped model with sparse blocks: prompt, then HIP graphs
  opt_prompt    the prompt of such a model
  generate      greedy generation of a Vimulorn or Varolorn model
  prompt        the prompt of one, whole or in portions

Weights are random.  Where a token is chosen, embeddings are large against what the layers add, and where a whole model
selects neurons and heads, the predictors are decisive: a trained model's choices stand well apart too, and results then
differ by rounding only.  ``exact`` restates every kind in 64 bits.
"""
from __future__ import annotations

import math
import zlib

import torch
import torch.nn.functional as F

DEV = "cuda"
WINDOW = 16
VOCAB = 50272  # of the OPT models
RANK = 1000    # of their predictors

# width, feed-forward, heads, head size, selected neurons and heads
OPT = {
    "opt-125m": (768, 3072, 12, 64, 1024, 4),
    "opt-6.7b": (4096, 16384, 32, 128, 4096, 16),
    "opt-13b": (5120, 20480, 40, 128, 2048, 16),
    "opt-66b": (9216, 36864, 72, 128, 4096, 24),
    "opt-175b": (12288, 49152, 96, 128, 4096, 32),
}


def listed():
    return [
        # one decode step of the smallest model's MLP: launches and latency
        dict(name="mlp 125m", kind="mlp", size="opt-125m", batch=1),
        # the headline: decode of three OPT-175B blocks, one sequence, 2048 cached tokens
        dict(name="layers 175b", kind="layers", size="opt-175b", batch=1, blocks=3, cached=2048),
        # decode in lockstep: sixteen sequences share the selection
        dict(name="layers 66b x16", kind="layers", size="opt-66b", batch=16, blocks=2, cached=1024),
        # a chat turn of the 13B shape: short prompt, sparse decode from graphs
        dict(name="generate 13b", kind="opt_generate", size="opt-13b", blocks=24, prompt=100, new=50),
        # prompts of the dense phase: one that the weights bound, and an ordinary ragged one
        dict(name="prompt 13b 128", kind="opt_prompt", size="opt-13b", blocks=8, prompt=128),
        dict(name="prompt 6.7b 777", kind="opt_prompt", size="opt-6.7b", blocks=8, prompt=777),
        # a long document into a Vimulorn model, and a conversation that arrives in short portions
        dict(name="vimulorn-4k 2048", kind="prompt", model="vimulorn-4k", dtype="bf16", tokens=2048, portion=2048),
        dict(name="vimulorn-4k portions", kind="prompt", model="vimulorn-4k", dtype="bf16", tokens=189, portion=47),
        dict(name="vimulorn-2k generate", kind="generate", model="vimulorn-2k", dtype="bf16", prompt=300, new=66),
        # the same for Varolorn, at an odd length
        dict(name="varolorn-4k 1999", kind="prompt", model="varolorn-4k", dtype="bf16", tokens=1999, portion=1999),
        dict(name="varolorn-4k generate", kind="generate", model="varolorn-4k", dtype="bf16", prompt=33, new=48),
        # full precision, as logits are compared and models are checked
        dict(name="vimulorn-2k fp32 500", kind="prompt", model="vimulorn-2k", dtype="fp32", tokens=500, portion=500),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["mlp", "layers", "opt_generate", "opt_prompt", "generate", "generate", "prompt", "prompt", "prompt"])
    if kind == "mlp":
        return dict(kind=kind, size=rng.choice(["opt-125m", "opt-6.7b", "opt-13b"]), batch=_log(rng, 1, 32))
    if kind == "layers":
        size = rng.choice(["opt-6.7b", "opt-13b", "opt-66b", "opt-175b"])
        return dict(kind=kind, size=size, batch=rng.choice([1, _log(rng, 2, 32)]), blocks=rng.randint(1, 2),
                    cached=_log(rng, 128, 2048))
    if kind == "opt_generate":
        return dict(kind=kind, size=rng.choice(["opt-6.7b", "opt-13b"]), blocks=rng.randint(6, 16), prompt=_log(rng, 4, 600),
                    new=rng.randint(20, 60))
    if kind == "opt_prompt":
        return dict(kind=kind, size=rng.choice(["opt-6.7b", "opt-13b"]), blocks=rng.randint(4, 8), prompt=_log(rng, 8, 2000))
    if kind == "generate":
        return dict(kind=kind, model=rng.choice(_MODELS), dtype="bf16", prompt=_log(rng, 2, 1500), new=rng.randint(20, 70))
    tokens = _log(rng, 2, 2048)
    portion = rng.choice([tokens, tokens, max(1, tokens // rng.randint(2, 5))])
    dtype = rng.choice(["bf16"] * 5 + ["fp32"])
    model = rng.choice(_MODELS)
    if dtype == "fp32":  # short ones of the smaller sizes
        model, tokens = model.replace("4k", "2k"), min(tokens, 600)
        portion = min(tokens, portion)
    return dict(kind=kind, model=model, dtype=dtype, tokens=tokens, portion=portion)


# ---- inputs -----------------------------------------------------------------------------------------------------------
class _Rand:
    """Tensors by name, each from the seed and its name alone."""

    def __init__(self, seed, dtype):
        self.seed, self.dtype = int(seed), dtype

    def _gen(self, name):
        g = torch.Generator(device=DEV)
        g.manual_seed((self.seed * 1000003 + zlib.crc32(name.encode())) % (1 << 62))
        return g

    def normal(self, name, *shape, std=1.0, mean=0.0, dtype=None):
        t = torch.empty(*shape, dtype=torch.float32, device=DEV)
        return t.normal_(mean, std, generator=self._gen(name)).to(dtype or self.dtype)

    def linear(self, name, out, inp, gain=1.0):
        return self.normal(name, out, inp, std=gain * inp ** -0.5)

    def ids(self, name, count, high):
        return torch.randint(0, high, (count,), generator=self._gen(name), device=DEV)

    def subset(self, name, count, high):
        return torch.randperm(high, generator=self._gen(name), device=DEV)[:count].sort().values


def _rank(size):
    return 128 if size == "opt-125m" else RANK


def _opt_block(r, size, l, decisive=None):
    """State dict of block l.  decisive: a direction of the residual stream that every token has; the selections of the
    next block then are a set of hot neurons and heads."""
    d, ffn, H, _, K, Hk = OPT[size]
    p, rank = f"b{l}.", _rank(size)
    t = {
        "mixer.Wqkv.weight": r.normal(p + "wqkv", 3 * d, d, std=0.02), "mixer.Wqkv.bias": r.normal(p + "bqkv", 3 * d, std=0.02),
        "mixer.out_proj.weight": r.normal(p + "wo", d, d, std=0.02), "mixer.out_proj.bias": r.normal(p + "bo", d, std=0.02),
        "mixer.sp.fc0.weight": r.normal(p + "sa", rank, d, std=0.05), "mixer.sp.fc1.weight": r.normal(p + "sb", H, rank, std=0.05),
        "mlp.fc1.weight": r.normal(p + "w1", ffn, d, std=0.02), "mlp.fc1.bias": r.normal(p + "b1", ffn, std=0.02, mean=-0.1),
        "mlp.fc2.weight": r.normal(p + "w2", d, ffn, std=0.02), "mlp.fc2.bias": r.normal(p + "b2", d, std=0.02),
        "mlp.sp.fc0.weight": r.normal(p + "ma", rank, d, std=0.05), "mlp.sp.fc1.weight": r.normal(p + "mb", ffn, rank, std=0.05),
    }
    for n in ("norm1", "norm2"):
        t[n + ".weight"], t[n + ".bias"] = r.normal(p + n, d, std=0.1, mean=1.0), r.normal(p + n + "b", d, std=0.1)
    if decisive is not None:
        for n, out, k in (("mixer", H, Hk), ("mlp", ffn, K)):
            t[n + ".sp.fc0.weight"][0] = decisive
            column = torch.full((out,), -8.0, device=DEV)
            column[r.subset(p + n + "hot", k, out)] = 8.0
            t[n + ".sp.fc1.weight"][:, 0] = column
    return t


def _opt_ends(r, size, positions):
    """Embeddings and final norm.  The direction that every position has is what decisive predictors read."""
    d = OPT[size][0]
    u = r.normal("u", d, dtype=torch.float32)
    u = u / u.norm()
    pos = r.normal("pos", positions, d, std=0.5, dtype=torch.float32) + 120.0 * u
    t = {"embeddings.word_embeddings.weight": r.normal("embed", VOCAB, d, std=3.0), "embeddings.position_embeddings.weight": pos.half(),
         "ln_f.weight": r.normal("lnf", d, std=0.1, mean=1.0), "ln_f.bias": r.normal("lnfb", d, std=0.1)}
    return t, u.half()


def _layer_inputs(r, c):
    """Cached keys and values per block, and per position the stream, the selected heads and the predictor's logits."""
    d, ffn, H, hd, _, Hk = OPT[c["size"]]
    B, S = c["batch"], c["cached"]
    kv = [(r.normal(f"k{l}", B, H, S, hd), r.normal(f"v{l}", B, H, S, hd)) for l in range(c["blocks"])]
    steps = []
    for s in range(WINDOW):
        heads = [r.subset(f"h{s}.{l}", Hk, H).int() for l in range(c["blocks"])]
        logits = [r.normal(f"m{s}.{l}", *((ffn,) if B == 1 else (B, ffn)), std=4.0) for l in range(c["blocks"])]
        steps.append((r.normal(f"x{s}", B, 1, d), r.normal(f"r{s}", B, 1, d), heads, logits))
    return kv, steps


_MODELS = ["vimulorn-4k", "vimulorn-2k", "varolorn-4k", "varolorn-2k"]


def _model_config(name):
    from dejavu_amd.workloads import VAROLORN_CONFIGS, VIMULORN_CONFIGS

    return {**VIMULORN_CONFIGS, **VAROLORN_CONFIGS}[name]


def _conv(r, name, channels, taps):
    w = r.normal(name, channels, taps, std=0.4, dtype=torch.float32)
    w[:, -1] += 1.0
    return w.to(r.dtype)


def _vimulorn(r, cfg):
    t, w = {}, cfg["width"]

    def norm(name, mean=1.0):
        t[name], t[name + ".b"] = r.normal(name, w, std=0.2 * mean, mean=mean), r.normal(name + ".b", w, std=0.1 * mean)
        t[name + ".alpha"] = r.normal(name + ".alpha", 1, std=0.1, mean=0.6).reshape(())

    t["embed"] = r.normal("embed", cfg["vocab"], w)
    # the next token stands where the head's row is this token's embedding
    t["head"] = (t["embed"].float() * w ** -0.5).to(r.dtype).roll(1, 0)
    norm("final.norm")
    for i, layer in enumerate(cfg["layers"]):
        m, p = layer["mixer"], f"l{i}.mix."
        H, dim, vdim = m["heads"], m["dim"], m["vdim"]

        def lin(name, out, inp, gain=1.0):
            t[p + name] = r.linear(p + name, out, inp, gain)

        for k in ("norm1", "norm2"):
            norm(f"l{i}.{k}")
            norm(f"l{i}.{k}b", 0.4)
        if layer["type"] == "latent_attention":
            qr, kr = m["q_rank"], m["kv_rank"]
            for k, out, inp in (("dq", qr, w), ("dkv", kr, w), ("g", H, w), ("uq", H * dim, qr), ("uk", H * dim, kr),
                                ("uv", H * vdim, kr)):
                lin(k, out, inp, 1.5 if k in ("uq", "uk") else 1.0)
            for k, n in (("dq", qr), ("dkv", kr)):
                t[p + k + ".norm"] = r.normal(p + k + ".norm", n, std=0.2, mean=1.0)
        else:
            G, delta = m["kv_heads"], layer["type"] == "channel_delta"
            for k, rows in (("q", (G if delta else H) * dim), ("k", G * dim), ("v", (H if delta else G) * vdim)):
                lin(k, rows, w)
                t[p + k + ".conv"] = _conv(r, p + k + ".conv", rows, m["conv"])
            if delta:
                for k, out, inp in (("b", H, w), ("a1", m["decay_rank"], w), ("g1", m["gate_rank"], w),
                                    ("a2", H * dim, m["decay_rank"]), ("g2", H * vdim, m["gate_rank"])):
                    lin(k, out, inp)
                t[p + "A_log"], t[p + "dt_bias"] = r.normal(p + "A_log", H, mean=-2.0), r.normal(p + "dt_bias", H * dim)
                t[p + "norm"] = r.normal(p + "norm", vdim, std=0.2, mean=1.0)
            else:
                t[p + "sink"] = r.normal(p + "sink", H, mean=1.0)
        lin("o", w, H * vdim, 1.5)
        p, ff = f"l{i}.mlp.", layer["mlp"]["ff"]
        lin("gate", ff, w, 1.5), lin("up", ff, w, 1.5), lin("down", w, ff)
    return t


def _varolorn(r, cfg):
    t, w, S = {}, cfg["width"], cfg["streams"]

    def hyper(p):
        t[p + ".in"], t[p + ".out"] = r.normal(p + ".in", S, std=0.05, mean=1.0 / S), r.normal(p + ".out", S, std=0.05, mean=0.3)
        t[p + ".mix"] = (torch.eye(S, device=DEV) * 0.9 + r.normal(p + ".mix", S, S, std=0.03, mean=0.025).float()).to(r.dtype)

    t["embed"] = r.linear("embed", cfg["vocab"], w)
    t["bigram"] = r.normal("bigram", cfg["embedding"]["bigram"]["buckets"] + 1, w, std=0.5)
    t["final.norm"] = r.normal("final.norm", w, std=0.2)
    for i, layer in enumerate(cfg["layers"]):
        m, p = layer["mixer"], f"l{i}.mix."
        H, vdim = m["heads"], m["vdim"]

        def vec(name, n, std, mean=0.0):
            t[p + name] = r.normal(p + name, n, std=std, mean=mean)

        for k in ("1", "2"):
            t[f"l{i}.norm{k}"] = r.normal(f"l{i}.norm{k}", w, std=0.2)
            hyper(f"l{i}.hc{k}")
        if layer["type"] == "attention":
            G, dim = m["kv_heads"], m["dim"]
            for k, rows in (("q", H * dim), ("k", G * dim), ("v", G * vdim)):
                t[p + k] = r.linear(p + k, rows, w)
                vec(k + ".b", rows, 0.3)
            vec("q.norm", dim, 0.3, 1.0), vec("k.norm", dim, 0.3, 1.0), vec("o.b", w, 0.1)
            t[p + "rel"], t[p + "g"] = r.normal(p + "rel", m["bias_rows"], H), r.linear(p + "g", H, w)
            if m["v_mix"]:
                t[p + "vmix"] = r.normal(p + "vmix", 1, std=0.1, mean=0.4).reshape(())
        else:
            inner, bc = H * vdim, m["groups"] * m["state"]
            t[p + "in"] = r.linear(p + "in", 2 * inner + 2 * bc + H, w)
            t[p + "conv"] = _conv(r, p + "conv", inner + 2 * bc, m["conv"])
            vec("conv.b", inner + 2 * bc, 0.2), vec("A_log", H, 1.0, -0.5), vec("dt_bias", H, 1.0, -2.0), vec("D", H, 1.0, 1.0)
            vec("norm", inner, 0.2, 1.0)
        t[p + "o"] = r.linear(p + "o", w, H * vdim)
        ff = layer["mlp"]["ff"]
        for k, out, inp in (("gate", ff, w), ("up", ff, w), ("down", w, ff)):
            t[f"l{i}.mlp.{k}"] = r.linear(f"l{i}.mlp.{k}", out, inp, 1.0 if k == "down" else 1.5)
    return t


def _model_tensors(c, seed):
    cfg = _model_config(c["model"])
    r = _Rand(seed, torch.float32 if c["dtype"] == "fp32" else torch.bfloat16)
    return r, cfg, (_vimulorn if c["model"].startswith("vimulorn") else _varolorn)(r, cfg)


# ---- what a program holds, and one pass ---------------------------------------------------------------------------------
def _load_block(block, tensors):
    block.load_state_dict(tensors)
    block.mlp.transposed_fc2()
    if hasattr(block.mixer, "transposed_out_proj"):
        block.mixer.transposed_out_proj()


@torch.no_grad()
def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


@torch.no_grad()
def run(state):
    return state["run"](state)


def _prepare_mlp(c, seed):
    from dejavu_amd.modules import ParallelFusedMLPDejavu

    d, ffn, _, _, K, _ = OPT[c["size"]]
    r, B = _Rand(seed, torch.float16), c["batch"]
    mlp = ParallelFusedMLPDejavu(d, ffn, {"embed_dim": d, "low_rank_dim": _rank(c["size"]), "out_dim": ffn, "K": K}, activation="relu",
                                 layer_idx=0, sequence_parallel=False, device=DEV, dtype=torch.float16)
    mlp.load_state_dict({k[4:]: v for k, v in _opt_block(r, c["size"], 0).items() if k.startswith("mlp.")})
    mlp.transposed_fc2()
    return dict(run=_run_mlp, mlp=mlp, x=r.normal("x", B, 1, d), residual=r.normal("r", B, 1, d),
                logits=r.normal("m", *((ffn,) if B == 1 else (B, ffn)), std=4.0))


def _run_mlp(s):
    idx = s["mlp"].sp.topk(s["logits"])
    out, logits = s["mlp"](s["x"], s["residual"], idx)
    return out, logits, idx


def _prepare_layers(c, seed):
    from dejavu_amd.block import create_sparse_block
    from dejavu_amd.fused_layer import LayerChain
    from dejavu_amd.modules import InferenceParams, join_side_stream
    from dejavu_amd.workloads import pack_k_cache

    d, ffn, H, hd, K, Hk = OPT[c["size"]]
    r, B, S, n = _Rand(seed, torch.float16), c["batch"], c["cached"], c["blocks"]
    ip = InferenceParams(max_sequence_len=S, max_batch_size=B)
    blocks = []
    kv, steps = _layer_inputs(r, c)
    for l in range(n):
        block = create_sparse_block(d, ffn, H, _rank(c["size"]), K, _rank(c["size"]), Hk, layer_idx=l, device=DEV).eval()
        _load_block(block, _opt_block(r, c["size"], l))
        block.mixer.cache_offset = torch.tensor([S - WINDOW], dtype=torch.int32, device=DEV)
        block.mixer.hold_window = True  # a pass is the window at the end of the cache
        block.defer_mlp_reduce = B > 1 and l + 1 < n
        ip.key_value_memory_dict[l] = (pack_k_cache(kv[l][0]), kv[l][1])
        blocks.append(block)

    def window():
        out = []
        for s, (hidden, residual, heads, logits) in enumerate(steps):
            ip.sequence_len_offset = S - WINDOW + s
            if B == 1:
                chain = LayerChain()
                for l, block in enumerate(blocks):
                    chain.add(block, heads[l], logits[l], ip, *((hidden, residual) if l == 0 else ()))
                hidden, residual, last, _, _ = chain.run()
                first = (chain.outputs[0][3], chain.outputs[0][4])
            else:
                for l, block in enumerate(blocks):
                    hidden, residual, last, att = block(hidden, residual, mixer_kwargs={"inference_params": ip},
                                                        head_idx=heads[l], mlp_sp_logit=logits[l])
                    first = (att,) if l == 0 else first
                join_side_stream()
            out.append((hidden, residual) + ((last, first) if s == WINDOW - 1 else ()))
        return out

    window()  # what later steps reuse is made here
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = window()
    return dict(run=_run_layers, graph=graph, out=out, caches=ip.key_value_memory_dict[n - 1], keep=(blocks, ip, steps))


def _run_layers(s):
    s["graph"].replay()
    return s["out"], s["caches"]


def _opt_model(c, seed, positions, decisive):
    from dejavu_amd.gpt import GPTLMHeadModel, SparseGPTConfig

    d, ffn, H, _, K, Hk = OPT[c["size"]]
    conf = SparseGPTConfig(hidden_size=d, num_attention_heads=H, num_hidden_layers=c["blocks"], vocab_size=VOCAB, n_inner=ffn,
                           max_position_embeddings=positions, mlp_K=K, mlp_sp_dim=RANK, att_K=[Hk, Hk], att_sp_dim=RANK,
                           pad_vocab_size_multiple=8)
    model = GPTLMHeadModel(conf, device=DEV, dtype=torch.float16).eval()
    r = _Rand(seed, torch.float16)
    ends, u = _opt_ends(r, c["size"], positions)
    model.transformer.load_state_dict(ends, strict=False)
    model.tie_weights()
    for l, block in enumerate(model.transformer.layers):
        _load_block(block, _opt_block(r, c["size"], l, u if decisive else None))
    return model, r.ids("ids", c["prompt"], VOCAB)[None]


def _prepare_opt_generate(c, seed):
    model, ids = _opt_model(c, seed, c["prompt"] + c["new"], True)
    s = dict(run=_run_generate, model=model, ids=ids, length=c["prompt"] + c["new"])
    _run_generate(s)  # a program's first turn captures its graphs
    return s


def _run_generate(s):
    out = s["model"].generate(s["ids"], max_length=s["length"], cg=True, return_dict_in_generate=True, output_scores=True)
    return out.sequences, out.scores


def _prepare_opt_prompt(c, seed):
    from dejavu_amd.modules import InferenceParams

    model, ids = _opt_model(c, seed, c["prompt"], False)
    return dict(run=_run_opt_prompt, model=model, ids=ids, ip=InferenceParams(max_sequence_len=c["prompt"] + WINDOW, max_batch_size=1))


def _run_opt_prompt(s):
    s["ip"].restart()
    logits = s["model"](s["ids"], inference_params=s["ip"], last_token_only=True).logits
    return logits, s["ip"].key_value_memory_dict


def _prepare_generate(c, seed):
    from dejavu_amd.registry import build_model

    r, cfg, t = _model_tensors(c, seed)
    s = dict(run=_run_generate, model=build_model(cfg, t, dtype=r.dtype), ids=r.ids("ids", c["prompt"], cfg["vocab"])[None],
             length=c["prompt"] + c["new"])
    del t
    _run_generate(s)
    return s


def _prepare_prompt(c, seed):
    from dejavu_amd.inference import InferenceParams
    from dejavu_amd.registry import build_model

    r, cfg, t = _model_tensors(c, seed)
    return dict(run=_run_prompt, model=build_model(cfg, t, dtype=r.dtype), ids=r.ids("ids", c["tokens"], cfg["vocab"])[None],
                portion=c["portion"], ip=InferenceParams(max_sequence_len=c["tokens"] + 64, max_batch_size=1))


def _run_prompt(s):
    ip, n = s["ip"], s["ids"].shape[1]
    ip.restart()
    for at in range(0, n, s["portion"]):
        ids = s["ids"][:, at:at + s["portion"]]
        logits = s["model"](ids, inference_params=ip, last_token_only=True).logits
        ip.sequence_len_offset += ids.shape[1]
    return logits, ip.key_value_memory_dict


_PREPARE = {"mlp": _prepare_mlp, "layers": _prepare_layers, "opt_generate": _prepare_opt_generate,
            "opt_prompt": _prepare_opt_prompt, "generate": _prepare_generate, "prompt": _prepare_prompt}


# ---- what a pass cannot do without ----------------------------------------------------------------------------------------
def _opt_step(size, batch, cached, flush=False):
    """(bytes, flops) of one sparse block at a decode step."""
    d, ffn, H, hd, K, Hk = OPT[size]
    Hk, rank = H if flush else Hk, _rank(size)
    weights = 4 * Hk * hd * d + 2 * K * d + 2 * d * rank + rank * (ffn + H)
    return 2 * weights + 4 * batch * Hk * hd * cached, 2 * batch * (weights + 2 * Hk * hd * cached)


def _model_sizes(name):
    """(weights that every token meets, of them the head's, per-layer-run attention (heads * sizes, reach))."""
    cfg = _model_config(name)
    layers, w, vocab = cfg["layers"], cfg["width"], cfg["vocab"]
    loop = cfg.get("loop")
    order = list(range(len(layers)))
    if loop:
        order = order[:loop["start"]] + order[loop["start"]:loop["stop"]] * loop["times"] + order[loop["stop"]:]
    weights, attention = 0, []
    for i in order:
        m, kind = layers[i]["mixer"], layers[i]["type"]
        H, vdim = m["heads"], m["vdim"]
        weights += 3 * w * layers[i]["mlp"]["ff"] + w * H * vdim
        if kind == "mamba2":
            weights += w * (2 * H * vdim + 2 * m["groups"] * m["state"] + H)
            attention.append((2 * H * vdim * m["state"], 1, 0))
            continue
        dim = m["dim"]
        if kind == "latent_attention":
            weights += (m["q_rank"] + m["kv_rank"] + H) * w + H * dim * m["q_rank"] + H * (dim + vdim) * m["kv_rank"]
            attention.append((H * (dim + vdim), 1 << 30, 2 * m["kv_rank"]))
        elif kind == "channel_delta":
            weights += (2 * m["kv_heads"] * dim + H * vdim + H + m["decay_rank"] + m["gate_rank"]) * w
            weights += H * dim * m["decay_rank"] + H * vdim * m["gate_rank"]
            attention.append((3 * H * vdim * dim, 1, 0))
        else:
            weights += (H * dim + m["kv_heads"] * (dim + vdim)) * w
            attention.append((H * (dim + vdim), (m.get("mask") or {}).get("size") or 1 << 30, 2 * m["kv_heads"] * (dim + vdim)))
    return weights, vocab * w, attention


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        d, ffn, _, _, K, _ = OPT[case["size"]]
        n = 2 * K * d + _rank(case["size"]) * (d + ffn)
        return {"bytes": 2 * n, "flops": 2 * case["batch"] * n}
    if kind == "layers":
        steps = [_opt_step(case["size"], case["batch"], case["cached"] - WINDOW + s + 1, s == WINDOW - 1) for s in range(WINDOW)]
        return {"bytes": case["blocks"] * sum(b for b, _ in steps), "flops": case["blocks"] * sum(f for _, f in steps)}
    if kind in ("opt_generate", "opt_prompt"):
        d, ffn, _, _, _, _ = OPT[case["size"]]
        n, blocks, dense = case["prompt"], case["blocks"], 4 * d * d + 2 * d * ffn
        total_b = 2 * (blocks * (dense + 2 * n * d) + VOCAB * d)
        total_f = 2 * (blocks * (n * dense + n * n * d) + VOCAB * d)
        for s in range(case.get("new", 1) - 1):
            b, f = _opt_step(case["size"], 1, n + s + 1, s % WINDOW == WINDOW - 1)
            extra = dense + VOCAB * d  # the first block is dense
            total_b, total_f = total_b + (blocks - 1) * b + 2 * extra, total_f + (blocks - 1) * f + 2 * extra
        return {"bytes": total_b, "flops": total_f}
    weights, head, attention = _model_sizes(case["model"])
    size = 4 if case["dtype"] == "fp32" else 2
    if kind == "generate":
        portions = [case["prompt"]] + [1] * (case["new"] - 1)
    else:
        n, p = case["tokens"], case["portion"]
        portions = [p] * (n // p) + ([n % p] if n % p else [])
    total_b = total_f = at = 0
    for p in portions:
        total_b += size * (weights + head)
        total_f += 2 * (p * weights + head)
        for wide, reach, row in attention:
            mean = min(reach, at + (p + 1) / 2)  # keys that a token sees
            total_f += 2 * p * wide * mean
            total_b += size // 2 * row * min(reach, at + p)
        at += p
    return {"bytes": int(total_b), "flops": int(total_f)}


def tolerance(case):
    """About four times the distance from ``exact``: 3e-4 (mlp), 2e-3 (other OPT kinds), 6e-3 (bf16 models), 5e-7 (fp32; the
    states beside the logits are a few times further off)."""
    kind = case["kind"]
    if kind == "mlp":
        return {"rel": 1.2e-3, "max": 1e-2}
    if kind in ("layers", "opt_prompt", "opt_generate"):  # fp16 between the launches, up to 24 blocks
        return {"rel": 1e-2, "max": 0.2}
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 2e-2, "max": 0.5}


# ---- the same in 64 bits -----------------------------------------------------------------------------------------------
@torch.no_grad()
def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def _d(t):
    return t.double()


def _layer_norm(x, t, name):
    return F.layer_norm(x, x.shape[-1:], _d(t[name + ".weight"]), _d(t[name + ".bias"]), 1e-5)


def _linear(x, t, name):
    return x @ _d(t[name + ".weight"]).t() + _d(t[name + ".bias"])


def _predict(x, t, name):
    return x @ _d(t[name + ".sp.fc0.weight"]).t() @ _d(t[name + ".sp.fc1.weight"]).t()


def _top(logits, k):
    """The k largest of a vector, ties to the lower index, ascending."""
    return logits.sort(descending=True, stable=True).indices[:k].sort().values


def _scores(logits):
    return logits if logits.dim() == 1 else logits.amax(0)


def _exact_mlp(c, seed):
    d, ffn, _, _, K, _ = OPT[c["size"]]
    r, B = _Rand(seed, torch.float16), c["batch"]
    t = _opt_block(r, c["size"], 0)
    idx = _top(_scores(r.normal("m", *((ffn,) if B == 1 else (B, ffn)), std=4.0)), K)
    h = (r.normal("x", B, 1, d).double() @ _d(t["mlp.fc1.weight"][idx]).t() + _d(t["mlp.fc1.bias"][idx])).relu()
    out = h @ _d(t["mlp.fc2.weight"][:, idx]).t() + _d(t["mlp.fc2.bias"])
    logits = _predict(r.normal("r", B, d).double(), t, "mlp")
    return out, logits.view(-1) if B == 1 else logits, idx


def _exact_layers(c, seed):
    d, ffn, H, hd, K, Hk = OPT[c["size"]]
    r, B, S, n = _Rand(seed, torch.float16), c["batch"], c["cached"], c["blocks"]
    kv, steps = _layer_inputs(r, c)
    out, weights = [None] * WINDOW, None
    hidden = [_d(s[0][:, 0]) for s in steps]
    residual = [_d(s[1][:, 0]) for s in steps]
    for l in range(n):
        t = _opt_block(r, c["size"], l)
        wqkv, wo = _d(t["mixer.Wqkv.weight"]), _d(t["mixer.out_proj.weight"])
        k, v = (x.double() for x in kv[l])
        for s in range(WINDOW):
            heads = torch.arange(H, device=DEV) if s == WINDOW - 1 else steps[s][2][l].long()
            residual[s] = hidden[s] + residual[s]
            x = _layer_norm(residual[s], t, "norm1")
            if l == 0 and s == WINDOW - 1:
                att = _top(_scores(_predict(residual[s], t, "mixer").half().squeeze(0)), Hk)
            qkv = (x @ wqkv.t() + _d(t["mixer.Wqkv.bias"])).view(B, 3, H, hd)
            at = S - WINDOW + s
            k[:, :, at], v[:, :, at] = qkv[:, 1], qkv[:, 2]
            p = torch.einsum("bhd,bhsd->bhs", qkv[:, 0, heads], k[:, heads, :at + 1]) * hd ** -0.5
            ctx = torch.zeros(B, H, hd, dtype=torch.float64, device=DEV)
            ctx[:, heads] = torch.einsum("bhs,bhsd->bhd", p.softmax(-1), v[:, heads, :at + 1])
            residual[s] = residual[s] + ctx.view(B, d) @ wo.t() + _d(t["mixer.out_proj.bias"])
            x = _layer_norm(residual[s], t, "norm2")
            idx = _top(_scores(steps[s][3][l]), K)
            h = (x @ _d(t["mlp.fc1.weight"][idx]).t() + _d(t["mlp.fc1.bias"][idx])).relu()
            hidden[s] = h @ _d(t["mlp.fc2.weight"][:, idx]).t() + _d(t["mlp.fc2.bias"])
            if l == 0 and s == WINDOW - 1:
                first = (att, idx) if B == 1 else (att,)
        del wqkv, wo
    out = [(h.unsqueeze(1), x.unsqueeze(1)) for h, x in zip(hidden, residual)]
    last = _predict(residual[-1], t, "mlp")
    out[-1] += (last.view(-1) if B == 1 else last, first)
    packed = k.view(B, H, S, hd // 8, 8).permute(0, 1, 3, 2, 4)
    return out, (packed, v)


def _exact_opt(c, seed, positions, tokens, decisive, caches=None):
    """Logits after every token; tokens from ``c["prompt"]`` on are decode steps, which select."""
    d, ffn, H, hd, K, Hk = OPT[c["size"]]
    r, n, T = _Rand(seed, torch.float16), c["prompt"], tokens.numel()
    ends, u = _opt_ends(r, c["size"], positions)
    x = _d(ends["embeddings.word_embeddings.weight"][tokens]) + _d(ends["embeddings.position_embeddings.weight"][:T])
    see = torch.ones(T, T, dtype=torch.bool, device=DEV).tril()
    heads = neurons = None
    for l in range(c["blocks"]):
        t = _opt_block(r, c["size"], l, u if decisive else None)
        next_heads = [_top(row.half(), Hk) for row in _predict(x[n:], t, "mixer")]
        q, k, v = _linear(_layer_norm(x, t, "norm1"), t, "mixer.Wqkv").view(T, 3, H, hd).permute(1, 2, 0, 3)
        if caches is not None:
            caches.append((k, v))
        ctx = torch.empty(T, H, hd, dtype=torch.float64, device=DEV)
        for h in range(H):
            ctx[:, h] = ((q[h] @ k[h].t()) * hd ** -0.5).masked_fill(~see, -math.inf).softmax(-1) @ v[h]
        if heads is not None:
            for s, chosen in enumerate(heads):
                if s % WINDOW != WINDOW - 1:
                    ctx[n + s] *= torch.zeros(H, 1, dtype=torch.float64, device=DEV).index_fill_(0, chosen, 1.0)
        x = x + _linear(ctx.view(T, d), t, "mixer.out_proj")
        h = _linear(_layer_norm(x, t, "norm2"), t, "mlp.fc1").relu()
        if neurons is not None:
            for s, chosen in enumerate(neurons):
                h[n + s] *= torch.zeros(ffn, dtype=torch.float64, device=DEV).index_fill_(0, chosen, 1.0)
        heads, neurons = next_heads, [_top(row.half(), K) for row in _predict(x[n:], t, "mlp")]
        x = x + _linear(h, t, "mlp.fc2")
    return _layer_norm(x[n - 1:], ends, "ln_f") @ _d(ends["embeddings.word_embeddings.weight"]).t()


def _exact_opt_generate(c, seed):
    n, new = c["prompt"], c["new"]
    ids = _Rand(seed, torch.float16).ids("ids", n, VOCAB)
    tokens = torch.cat([ids, ids[-1:].repeat(new - 1)])  # a token's own row of the tied head stands out
    logits = _exact_opt(c, seed, n + new, tokens, True)
    return torch.cat([ids, logits.argmax(-1)])[None], logits


def _exact_opt_prompt(c, seed):
    n = c["prompt"]
    d, _, H, hd, _, _ = OPT[c["size"]]
    caches = []
    logits = _exact_opt(c, seed, n, _Rand(seed, torch.float16).ids("ids", n, VOCAB), False, caches)
    memory = {}
    for l, (k, v) in enumerate(caches):
        kc, vc = (torch.zeros(1, H, n + WINDOW, hd, dtype=torch.float64, device=DEV) for _ in range(2))
        kc[0, :, :n], vc[0, :, :n] = k, v
        memory[l] = (kc.view(1, H, n + WINDOW, hd // 8, 8).permute(0, 1, 3, 2, 4), vc)
    return logits[-1:][None], memory


def _rms(x, eps):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt()


def _taps(x, w, b=None):
    """Causal depthwise convolution of (T, channels) with (channels, taps), the last tap the newest token's."""
    y = F.conv1d(x.t()[None], _d(w)[:, None], None if b is None else _d(b), padding=w.shape[1] - 1, groups=w.shape[0])
    return y[0, :, :x.shape[0]].t()


def _attend(q, k, v, scale, see, sink=None, bias=None):
    """q (T, H, dim), k and v (T, G, ..): every head in turn."""
    T, H, rep = q.shape[0], q.shape[1], q.shape[1] // k.shape[1]
    out = torch.empty(T, H, v.shape[2], dtype=torch.float64, device=DEV)
    for h in range(H):
        s = (q[:, h] @ k[:, h // rep].t()) * scale
        if bias is not None:
            s = s + bias(h)
        s = s.masked_fill(~see, -math.inf)
        if sink is not None:
            s = torch.cat([s, _d(sink[h]).expand(T, 1)], 1)
        out[:, h] = s.softmax(-1)[:, :T] @ v[:, h // rep]
    return out


def _vimulorn_mixer(kind, h, p, m, eps):
    T, H, dim, vdim = h.shape[0], m["heads"], m["dim"], m["vdim"]
    lin = lambda x, name: x @ _d(p[name]).t()  # noqa: E731
    ages = torch.arange(T, device=DEV)[:, None] - torch.arange(T, device=DEV)
    if kind == "latent_attention":
        q = lin(_rms(lin(h, "dq"), eps) * _d(p["dq.norm"]), "uq").view(T, H, dim)
        c = _rms(lin(h, "dkv"), eps) * _d(p["dkv.norm"])
        o = _attend(q, lin(c, "uk").view(T, H, dim), lin(c, "uv").view(T, H, vdim), m["scale"], ages >= 0)
        o = o * lin(h, "g").sigmoid()[..., None]
    elif kind == "attention":
        G = m["kv_heads"]
        q, k, v = (_taps(lin(h, n), p[n + ".conv"]) for n in "qkv")
        o = _attend(_rms(q.view(T, H, dim), eps), _rms(k.view(T, G, dim), eps), v.view(T, G, vdim), m["scale"],
                    (ages >= 0) & (ages < m["mask"]["size"]), p["sink"])
    else:
        G = m["kv_heads"]
        q, k, v = (F.silu(_taps(lin(h, n), p[n + ".conv"])) for n in "qkv")
        q, k = (x.view(T, G, dim) / (x.view(T, G, dim).square().sum(-1, keepdim=True) + 1e-6).sqrt() for x in (q, k))
        q, k, v = (q * dim ** -0.5).repeat_interleave(H // G, 1), k.repeat_interleave(H // G, 1), v.view(T, H, vdim)
        beta = lin(h, "b").sigmoid()
        z = (lin(lin(h, "a1"), "a2") + _d(p["dt_bias"])).view(T, H, dim)
        g = torch.exp(-_d(p["A_log"]).exp()[:, None] * F.softplus(z, threshold=50))
        S, rows = torch.zeros(H, dim, vdim, dtype=torch.float64, device=DEV), []
        for i in range(T):
            S = S * g[i, :, :, None]
            u = beta[i, :, None] * (v[i] - torch.bmm(k[i, :, None], S)[:, 0])
            S = torch.baddbmm(S, k[i, :, :, None], u[:, None])
            rows.append(torch.bmm(q[i, :, None], S)[:, 0])
        o = _rms(torch.stack(rows), eps) * _d(p["norm"])
        o = o * lin(lin(h, "g1"), "g2").sigmoid().view(T, H, vdim)
    return lin(o.reshape(T, -1), "o")


def _under(t, prefix):
    return {k[len(prefix):]: v for k, v in t.items() if k.startswith(prefix)}


def _exact_vimulorn(cfg, t, tokens, first):
    eps, loop = cfg["norm"]["eps"], cfg.get("loop")

    def norm(x, name):
        return torch.tanh(_d(t[name + ".alpha"]) * x) * _d(t[name]) + _d(t[name + ".b"])

    order = [(i, False) for i in range(len(cfg["layers"]))]
    if loop:
        a, b = loop["start"], loop["stop"]
        order = order[:a] + [(i, n > 0 and i == a) for n in range(loop["times"]) for i in range(a, b)] + order[b:]
    start = _d(t["embed"][tokens])
    x = start.clone()
    for i, again in order:
        layer = cfg["layers"][i]
        x = x + start if again else x
        x = x + norm(_vimulorn_mixer(layer["type"], norm(x, f"l{i}.norm1"), _under(t, f"l{i}.mix."), layer["mixer"], eps), f"l{i}.norm1b")
        h, limit, p = norm(x, f"l{i}.norm2"), layer["mlp"]["limit"], _under(t, f"l{i}.mlp.")
        gate, up = (h @ _d(p["gate"]).t()).clamp(max=limit), (h @ _d(p["up"]).t()).clamp(-limit, limit)
        x = x + norm((gate * (1.702 * gate).sigmoid() * (up + 1.0)) @ _d(p["down"]).t(), f"l{i}.norm2b")
    return norm(x[first:], "final.norm") @ _d(t["head"]).t()


def _bucket(n, rows, far):
    half = rows // 2
    if n < half:
        return n
    k, rest = 0, rows - half
    while k < rest and far ** (k + 1) * half ** rest <= n ** rest * half ** (k + 1):
        k += 1
    return min(rows - 1, half + k)


def _varolorn_mixer(kind, h, p, m, eps, state):
    T, H, vdim = h.shape[0], m["heads"], m["vdim"]
    if kind == "attention":
        G, dim, chunk = m["kv_heads"], m["dim"], (m.get("mask") or {}).get("size") or T
        q, k, v = ((h @ _d(p[n]).t() + _d(p[n + ".b"])).view(T, heads, -1) for n, heads in (("q", H), ("k", G), ("v", G)))
        if m["v_mix"]:
            lam = _d(p["vmix"])
            v, state["v"] = (v if "v" not in state else (1.0 - lam) * v + lam * state["v"]), state.get("v", v)
        at = torch.arange(T, device=DEV)
        ages = at[:, None] - at
        rel = _d(p["rel"])[torch.tensor([_bucket(n, p["rel"].shape[0], m["bias_max"]) for n in range(T)], device=DEV)]
        o = _attend(_rms(q, eps) * _d(p["q.norm"]), _rms(k, eps) * _d(p["k.norm"]), v, m["scale"],
                    (ages >= 0) & (at[:, None] // chunk == at // chunk), bias=lambda i: rel[ages.clamp(min=0), i])
        o = (o * (h @ _d(p["g"]).t()).sigmoid()[..., None]).reshape(T, -1)
        return o @ _d(p["o"]).t() + _d(p["o.b"])
    N, G = m["state"], m["groups"]
    inner, bc = H * vdim, N * G
    z, xbc, dt = (h @ _d(p["in"]).t()).split([inner, inner + 2 * bc, H], 1)
    x, B, C = F.silu(_taps(xbc, p["conv"], p["conv.b"])).split([inner, bc, bc], 1)
    B, C = (a.reshape(T, G, N).repeat_interleave(H // G, 1) for a in (B, C))
    x, dt = x.reshape(T, H, vdim), F.softplus(dt + _d(p["dt_bias"]), threshold=50)
    keep = torch.exp(-_d(p["A_log"]).exp() * dt)
    S, rows = torch.zeros(H, N, vdim, dtype=torch.float64, device=DEV), []
    for i in range(T):
        S = torch.baddbmm(S * keep[i, :, None, None], (dt[i, :, None] * B[i])[:, :, None], x[i][:, None])
        rows.append(torch.bmm(C[i, :, None], S)[:, 0])
    y = (torch.stack(rows) + _d(p["D"])[:, None] * x).view(T, inner) * F.silu(z)
    y = _rms(y.view(T, m["norm_groups"], -1), eps).view(T, inner) * _d(p["norm"])
    return y @ _d(p["o"]).t()


def _exact_varolorn(cfg, t, tokens, first):
    eps, emb, state = cfg["norm"]["eps"], cfg["embedding"], {}
    big = emb["bigram"]
    rows = torch.cat([tokens.new_tensor([big["buckets"]]),
                      (tokens[:-1] * big["mul_prev"] + tokens[1:] * big["mul_cur"]) % big["buckets"]])
    x = _d(t["embed"][tokens]) * emb["scale"] + _d(t["bigram"][rows])
    streams = x[None].repeat(cfg["streams"], 1, 1)

    def norm(x, name):
        return _rms(x, eps) * (1.0 + _d(t[name]))

    for i, layer in enumerate(cfg["layers"]):
        for k in "12":
            hc = _under(t, f"l{i}.hc{k}.")
            h = norm(torch.einsum("s,stw->tw", _d(hc["in"]), streams), f"l{i}.norm{k}")
            if k == "1":
                y = _varolorn_mixer(layer["type"], h, _under(t, f"l{i}.mix."), layer["mixer"], eps, state)
            else:
                p = _under(t, f"l{i}.mlp.")
                y = ((h @ _d(p["gate"]).t()).relu() * (h @ _d(p["up"]).t())) @ _d(p["down"]).t()
            streams = torch.einsum("st,snw->tnw", _d(hc["mix"]), streams) + _d(hc["out"])[:, None, None] * y
    return norm(streams.sum(0)[first:], "final.norm") @ _d(t["embed"]).t()


def _exact_model(c, seed, extra):
    """Logits from the prompt's last token on; every further token is the one whose logit stands out."""
    r, cfg, t = _model_tensors(c, seed)
    tokens = r.ids("ids", c.get("prompt") or c["tokens"], cfg["vocab"])
    first = tokens.numel() - 1
    vimulorn = c["model"].startswith("vimulorn")
    if extra:
        step = (lambda token: (token + 1) % cfg["vocab"]) if vimulorn else (lambda token: token)
        for _ in range(extra):
            tokens = torch.cat([tokens, step(tokens[-1:])])
    return tokens[:first + 1], (_exact_vimulorn if vimulorn else _exact_varolorn)(cfg, t, tokens, first)


def _exact_generate(c, seed):
    ids, logits = _exact_model(c, seed, c["new"] - 1)
    return torch.cat([ids, logits.argmax(-1)])[None], logits


def _exact_prompt(c, seed):
    return _exact_model(c, seed, 0)[1][None], None  # the state's layout is the package's own


_EXACT = {"mlp": _exact_mlp, "layers": _exact_layers, "opt_generate": _exact_opt_generate, "opt_prompt": _exact_opt_prompt,
          "generate": _exact_generate, "prompt": _exact_prompt}
