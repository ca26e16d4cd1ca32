"""The work that is timed: prompts, decode steps and images through the models' public entry points.

Every case is one call pattern of a serving program.  `decode` feeds given tokens to sequences that already hold a context (one sequence through `step`, several
through `step_batch`), `prompt` reads a prompt into an empty cache or behind a cached prefix, `image` runs the vision tower.  Models have random weights of the
widths that the benchmarks use and four layers, as the design benchmark's have: a step's cost is the layers' and the head's, and the outputs stay comparable
with 64-bit arithmetic (bfloat16 through 32 random layers does not).  Tokens are given, not fed back, so that one rounded logit cannot turn a pass into another text."""
from __future__ import annotations

import math

import numpy as np
import torch

LAYERS = 4
VOCAB = 32768

# Widths of Llama-shaped models: TinyLlama-1.1B, Llama-3.2-3B, Llama-3-8B.
LLAMA = {
    "1b": {"hidden_size": 2048, "intermediate_size": 5632, "num_attention_heads": 32, "num_key_value_heads": 4, "rope_theta": 10000.0},
    "3b": {"hidden_size": 3072, "intermediate_size": 8192, "num_attention_heads": 24, "num_key_value_heads": 8, "rope_theta": 500000.0},
    "8b": {"hidden_size": 4096, "intermediate_size": 14336, "num_attention_heads": 32, "num_key_value_heads": 8, "rope_theta": 500000.0},
}
# Layer-stack designs at the sizes of the design benchmark.
TADUZEN = {
    "dense4096": {"width": 4096, "heads": 32, "ff": 14336},
    "moe2048": {"width": 2048, "heads": 16, "experts": 64, "top": 6, "ff": 1408, "shared": 2816},
}
LAGELORN = {
    "wide4096": {"width": 4096, "heads": 32, "kv_heads": 8, "delta": {"heads": 32, "kv_heads": 16, "dim": 128, "vdim": 128, "conv": 4}, "rank": 128, "side": 256, "ff": 14336},
    "slim2048": {"width": 2048, "heads": 16, "kv_heads": 4, "delta": {"heads": 16, "kv_heads": 16, "dim": 128, "vdim": 256, "conv": 4}, "rank": 64, "side": 128, "ff": 8448},
}
DIM = 128          # of every head of the layer-stack designs
LATENT = 512
POSITIONS = 8192
VISION = {"depth": 8, "hidden_size": 1280, "intermediate_size": 3420, "out_hidden_size": 3584, "num_heads": 16}   # the 7B tower's widths, a quarter of its blocks


def listed():
    return [
        # a small dense float16 model answers one user: the smallest launches there are
        {"name": "decode f16 1b x1", "kind": "decode", "model": "llama", "size": "1b", "weights": "f16", "batch": 1, "context": 128, "steps": 16},
        # the benchmark's own workload: one int4 sequence behind a short prompt
        {"name": "decode int4 8b x1", "kind": "decode", "model": "llama", "size": "8b", "weights": "int4", "batch": 1, "context": 128, "steps": 16},
        # the same model serves a few users, and a full batch at a thousand tokens each
        {"name": "decode int4 8b x8", "kind": "decode", "model": "llama", "size": "8b", "weights": "int4", "batch": 8, "context": 200, "steps": 16},
        {"name": "decode int4 8b x32", "kind": "decode", "model": "llama", "size": "8b", "weights": "int4", "batch": 32, "context": 1000, "steps": 16},
        # unquantised weights under an ordinary load
        {"name": "decode bf16 8b x8", "kind": "decode", "model": "llama", "size": "8b", "weights": "bf16", "batch": 8, "context": 1000, "steps": 16},
        # a long document, and an ordinary question of an odd length
        {"name": "prompt int4 8b 4096", "kind": "prompt", "model": "llama", "size": "8b", "weights": "int4", "cached": 0, "tokens": 4096},
        {"name": "prompt bf16 8b 509", "kind": "prompt", "model": "llama", "size": "8b", "weights": "bf16", "cached": 0, "tokens": 509},
        # the next turn of a chat: a few words behind a cached conversation
        {"name": "prompt int4 8b 37 behind 900", "kind": "prompt", "model": "llama", "size": "8b", "weights": "int4", "cached": 900, "tokens": 37},
        # layer-stack designs: a mixture under a full batch, recurrent states under an ordinary one, a long prompt
        {"name": "decode taduzen moe2048 x32", "kind": "decode", "model": "taduzen", "size": "moe2048", "weights": "bf16", "batch": 32, "context": 600, "steps": 16},
        {"name": "decode lagelorn wide4096 x8", "kind": "decode", "model": "lagelorn", "size": "wide4096", "weights": "bf16", "batch": 8, "context": 300, "steps": 24},
        {"name": "prompt lagelorn wide4096 2000", "kind": "prompt", "model": "lagelorn", "size": "wide4096", "weights": "bf16", "cached": 0, "tokens": 2000},
        # an image of 448 x 448 pixels
        {"name": "image 32x32", "kind": "image", "height": 32, "width": 32},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["decode"] * 5 + ["prompt"] * 4 + ["image"])
    if kind == "image":
        return {"kind": kind, "height": 2 * rng.randint(4, 24), "width": 2 * rng.randint(4, 24)}
    model = rng.choice(["llama"] * 5 + ["taduzen"] * 2 + ["lagelorn"])
    size = rng.choice(sorted({"llama": LLAMA, "taduzen": TADUZEN, "lagelorn": LAGELORN}[model]))
    weights = "bf16" if model != "llama" else rng.choice(["f16", "bf16"] if size == "1b" else ["int4", "int4", "int8", "bf16"])
    case = {"kind": kind, "model": model, "size": size, "weights": weights}
    if kind == "decode":
        return dict(case, batch=log(1, 32), context=log(40, 1000), steps=rng.randint(10, 16))
    return dict(case, cached=rng.choice([0, 0, log(40, 1000)]) if model == "llama" else 0, tokens=log(8, 3000 if model == "llama" else 2000))


# ------------------------------------------------------------------ weights
def _quantise(w, bits):
    """Groups of 64 along a row: w = scale * code + bias, the codes packed from a word's low bits up, scale and bias in bfloat16."""
    n, k = w.shape
    g = w.float().view(n, k // 64, 64)
    lo, hi = g.amin(-1, keepdim=True), g.amax(-1, keepdim=True)
    scale, bias = ((hi - lo) / (2 ** bits - 1)).to(torch.bfloat16), lo.to(torch.bfloat16)
    q = ((g - bias.float()) / scale.float()).round_().clamp_(0, 2 ** bits - 1).to(torch.uint8).view(n, k)
    if bits == 4:
        q = q[:, 0::2] | (q[:, 1::2] << 4)
    return q.contiguous().view(torch.int32), scale.squeeze(-1), bias.squeeze(-1)


class _Weights(dict):
    """A random checkpoint, drawn on the GPU."""

    def __init__(self, seed, dtype):
        super().__init__()
        self.gen, self.dtype = torch.Generator(device="cuda").manual_seed(seed), dtype

    def put(self, name, *shape, std=None, mean=0.0):
        w = torch.randn(shape, generator=self.gen, device="cuda").mul_(shape[-1] ** -0.5 if std is None else std).add_(mean)
        self[name] = w.to(self.dtype)

    def lean(self, a, b):
        """A token's query leans on its own key, as trained ones do: otherwise the first outputs of a recurrent head are next to nothing, and its norm blows up their rounding."""
        self[a] = (self[a].float() * 0.4 + self[b].float() * 0.92).to(self.dtype)


def _llama(case, seed):
    """(config, checkpoint) in the layout of a Hugging Face directory."""
    size = LLAMA[case["size"]]
    H, I, D = size["hidden_size"], size["intermediate_size"], size["hidden_size"] // size["num_attention_heads"]
    bits = {"int4": 4, "int8": 8}.get(case["weights"])
    cfg = dict(size, model_type="llama", num_hidden_layers=LAYERS, vocab_size=VOCAB, rms_norm_eps=1e-5, max_position_embeddings=POSITIONS, tie_word_embeddings=False,
               quantization={"group_size": 64, "bits": bits} if bits else None)
    w = _Weights(seed, torch.float16 if case["weights"] == "f16" else torch.bfloat16)

    def linear(name, n, k, std=None):
        w.put(name + ".weight", n, k, std=std)
        if bits:
            w[name + ".weight"], w[name + ".scales"], w[name + ".biases"] = _quantise(w[name + ".weight"], bits)

    linear("model.embed_tokens", VOCAB, H, std=1.0), linear("lm_head", VOCAB, H)
    w.put("model.norm.weight", H, std=0.02, mean=1.0)
    for i in range(LAYERS):
        p = f"model.layers.{i}."
        w.put(p + "input_layernorm.weight", H, std=0.02, mean=1.0), w.put(p + "post_attention_layernorm.weight", H, std=0.02, mean=1.0)
        linear(p + "self_attn.q_proj", H, H), linear(p + "self_attn.o_proj", H, H)
        linear(p + "self_attn.k_proj", size["num_key_value_heads"] * D, H), linear(p + "self_attn.v_proj", size["num_key_value_heads"] * D, H)
        linear(p + "mlp.gate_proj", I, H), linear(p + "mlp.up_proj", I, H), linear(p + "mlp.down_proj", H, I)
    return cfg, w


def _taduzen(case, seed):
    size = TADUZEN[case["size"]]
    W, H, F = size["width"], size["heads"], size["ff"]
    mixer = {"heads": H, "dim": DIM, "vdim": DIM, "kv_rank": LATENT, "scale": DIM ** -0.5, "mask": {"size": 4096}}
    mlp = {"kind": "dense", "ff": F} if "experts" not in size else \
        {"kind": "moe", "expert": {"ff": F}, "router": {"experts": size["experts"], "top": size["top"]}, "shared": {"ff": size["shared"]}}
    cfg = {"architecture": "Taduzen", "vocab": VOCAB, "width": W, "logit_scale": 1.0, "norm": {"eps": 1e-6}, "layers": [{"type": "latent_attention", "mixer": mixer, "mlp": mlp}] * LAYERS}
    w = _Weights(seed, torch.bfloat16)

    def norm(name):
        w.put(name, W, std=0.02, mean=1.0), w.put(name + ".b", W, std=0.02)
        w[name + ".alpha"] = torch.tensor(0.5, dtype=torch.bfloat16, device="cuda")

    w.put("embed", VOCAB, W, std=1.0), w.put("head", VOCAB, W), norm("final.norm")
    for i in range(LAYERS):
        p = f"l{i}."
        for n in ("norm1", "norm1b", "norm2", "norm2b"):
            norm(p + n)
        w.put(p + "mix.q", H * DIM, W), w.put(p + "mix.dkv", LATENT, W), w.put(p + "mix.dkv.norm", LATENT, std=0.02, mean=1.0)
        w.put(p + "mix.uk", H * DIM, LATENT), w.put(p + "mix.uv", H * DIM, LATENT), w.put(p + "mix.o", W, H * DIM)
        if "experts" not in size:
            w.put(p + "mlp.up", F, W), w.put(p + "mlp.down", W, F)
            continue
        for e in [f"e{e}" for e in range(size["experts"])] + ["shared"]:
            f = size["shared"] if e == "shared" else F
            w.put(f"{p}mlp.{e}.gate", f, W), w.put(f"{p}mlp.{e}.up", f, W), w.put(f"{p}mlp.{e}.down", W, f)
        w.put(p + "mlp.shared.sg", 1, W)
        w[p + "mlp.table"] = torch.rand(VOCAB, size["experts"], generator=w.gen, device="cuda").topk(size["top"], dim=1).indices.to(torch.int32)
    return cfg, w


def _lagelorn(case, seed):
    size = LAGELORN[case["size"]]
    W, H, G, d, R, S, F = (size[k] for k in ("width", "heads", "kv_heads", "delta", "rank", "side", "ff"))
    left = {"heads": H, "kv_heads": G, "dim": DIM, "vdim": DIM, "scale": DIM ** -0.5, "bias_max": 128, "mask": {"size": 4096}}
    kinds = [("delta", d), ("parallel", {"left": left, "right": {"heads": H, "dim": DIM}, "left_scale": 0.7, "right_scale": 0.7})]
    layers = [{"type": kinds[i % 2][0], "mixer": kinds[i % 2][1], "mlp": {"kind": "dense", "ff": F}} for i in range(LAYERS)]
    cfg = {"architecture": "Lagelorn", "vocab": VOCAB, "width": W, "max_positions": POSITIONS, "token_side": {"dim": S}, "norm": {"eps": 1e-6}, "postln_alpha": 2.0, "logit_softcap": 30.0,
           "layers": layers}
    w = _Weights(seed, torch.bfloat16)
    w.put("embed", VOCAB, W, std=1.0), w.put("pos", POSITIONS, W, std=0.2), w.put("side.embed", VOCAB, LAYERS * S, std=1.0)
    w.put("final.norm", W, std=0.02, mean=1.0), w.put("head", VOCAB, W)
    for i, lay in enumerate(layers):
        p = f"l{i}."
        w.put(p + "norm1", W, std=0.02, mean=1.0), w.put(p + "norm2", W, std=0.02, mean=1.0)
        w.put(p + "side.gate", S, W), w.put(p + "side.proj", W, S), w.put(p + "side.norm", W, std=0.02, mean=0.2)
        if lay["type"] == "delta":
            q = p + "mix."
            for n, c in (("q", d["kv_heads"] * DIM), ("k", d["kv_heads"] * DIM), ("v", d["heads"] * d["vdim"])):
                w.put(q + n, c, W), w.put(q + n + ".conv", c, d["conv"], std=0.4)
                w[q + n + ".conv"][:, -1] += 0.8
            w.lean(q + "q", q + "k"), w.lean(q + "q.conv", q + "k.conv")
            w.put(q + "g", d["heads"] * d["vdim"], W), w.put(q + "a", d["heads"], W), w.put(q + "b", d["heads"], W), w.put(q + "A_log", d["heads"], std=0.5)
            w.put(q + "dt_bias", d["heads"], std=1.0, mean=-3.0), w.put(q + "norm", d["vdim"], std=0.02, mean=1.0), w.put(q + "o", W, d["heads"] * d["vdim"])
        else:
            q = p + "mix.left."
            w.put(q + "q", H * DIM, W), w.put(q + "q.b", H * DIM, std=0.02), w.put(q + "k", G * DIM, W), w.put(q + "k.b", G * DIM, std=0.02), w.put(q + "o", W, H * DIM)
            w.put(q + "q.norm", H * DIM, std=0.02, mean=1.0), w.put(q + "k.norm", G * DIM, std=0.02, mean=1.0), w.put(q + "rel", 32, H, std=0.5), w.put(q + "sink", H, std=1.0)
            q = p + "mix.right."
            for n in "rkvgw":
                w.put(q + "mu." + n, W, std=0.2, mean=0.5)
            for n in "rkvg":
                w.put(q + n, H * DIM, W)
            w.lean(q + "r", q + "k")
            w.put(q + "w1", R, W), w.put(q + "w2", H * DIM, R), w.put(q + "w0", H * DIM, std=1.0, mean=-3.0), w.put(q + "u", H, DIM, std=0.3)
            w.put(q + "norm", H * DIM, std=0.02, mean=1.0), w.put(q + "o", W, H * DIM)
        for n in ("gate", "up"):
            w.put(p + f"mlp.{n}", F, W), w.put(p + f"mlp.{n}.b", F, std=0.02)
        w.put(p + "mlp.down", W, F), w.put(p + "mlp.down.b", W, std=0.02)
    return cfg, w


def _vision(seed):
    c = VISION
    H, I, O = c["hidden_size"], c["intermediate_size"], c["out_hidden_size"]
    w = _Weights(seed, torch.bfloat16)

    def linear(name, n, k):
        w.put(name + ".weight", n, k), w.put(name + ".bias", n, std=0.1)

    t = "vision_tower."
    w.put(t + "patch_embed.proj.weight", H, 1176)
    w[t + "patch_embed.proj.weight"] = w[t + "patch_embed.proj.weight"].view(H, 3, 2, 14, 14)
    for i in range(c["depth"]):
        p = f"{t}blocks.{i}."
        w.put(p + "norm1.weight", H, std=0.02, mean=1.0), w.put(p + "norm2.weight", H, std=0.02, mean=1.0)
        linear(p + "attn.qkv", 3 * H, H), linear(p + "attn.proj", H, H), linear(p + "mlp.gate_proj", I, H), linear(p + "mlp.up_proj", I, H), linear(p + "mlp.down_proj", H, I)
    w.put(t + "merger.ln_q.weight", H, std=0.02, mean=1.0), linear(t + "merger.mlp.0", 4 * H, 4 * H), linear(t + "merger.mlp.2", O, 4 * H)
    return w


# ------------------------------------------------------------------ inputs
def _lengths(case):
    """Every sequence of a batch holds a context of its own length: 13 apart, around the case's."""
    return [max(8, case["context"] - 13 * (i % 8)) for i in range(case["batch"])]


def _tokens(case, seed):
    """int32 [sequences, tokens] on the CPU; a sequence uses the head of its row."""
    n, most = (case["batch"], case["context"] + case["steps"]) if case["kind"] == "decode" else (1, case["cached"] + case["tokens"])
    return torch.randint(0, VOCAB, (n, most), generator=torch.Generator().manual_seed(seed + 1), dtype=torch.int32)


def _pixels(case, seed):
    return torch.randn(case["height"] * case["width"], 1176, generator=torch.Generator(device="cuda").manual_seed(seed + 1), device="cuda").to(torch.bfloat16)


def _checkpoint(case, seed):
    return {"llama": _llama, "taduzen": _taduzen, "lagelorn": _lagelorn}[case["model"]](case, seed)


def prepare(case, seed):
    from proxy_inference_engine_amd.models import lagelorn, taduzen
    from proxy_inference_engine_amd.models.intern.vision import VisionConfig, VisionModel
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    if case["kind"] == "image":
        return {"case": case, "model": VisionModel(VisionConfig(**VISION), _vision(seed)), "pixels": _pixels(case, seed), "grid": [(1, case["height"], case["width"])]}
    cfg, w = _checkpoint(case, seed)
    design = {"taduzen": taduzen, "lagelorn": lagelorn}.get(case["model"])
    model = design.Model(design.ModelArgs(**cfg), w) if design else Model(ModelArgs(**cfg), w)
    del w
    tokens = _tokens(case, seed)
    state = {"case": case, "model": model}
    if case["kind"] == "prompt":
        if case["model"] == "lagelorn" or case["model"] == "taduzen":
            model.enable_paged_kv(num_pages=case["tokens"] // 64 + 2, max_blocks=case["tokens"] // 64 + 1)
        state["prompt"] = tokens[0, case["cached"]:].cuda()
        if case["cached"]:
            state["cache"] = model.make_cache()
            model.step(tokens[0, :case["cached"]].cuda(), state["cache"])
        return state
    lengths = _lengths(case)
    if case["batch"] > 1 or case["model"] != "llama":   # one Llama sequence keeps its keys and values in buffers of its own, several share a pool of pages
        blocks = (case["context"] + case["steps"]) // 64 + 1
        model.enable_paged_kv(num_pages=2 * blocks * case["batch"], max_blocks=blocks, **({"max_sequences": 2 * case["batch"]} if case["model"] != "llama" else {}))
    state["caches"] = [model.make_cache() for _ in lengths]
    if case["batch"] > 1:
        model.prefill_batch([tokens[i, :n].numpy() for i, n in enumerate(lengths)], state["caches"])
    else:
        model.step(tokens[0, :lengths[0]].cuda(), state["caches"][0])
    state["tokens"] = torch.stack([tokens[i, n:n + case["steps"]] for i, n in enumerate(lengths)], dim=1).contiguous().cuda()   # [steps, sequences]
    return state


# ------------------------------------------------------------------ one pass
def run(state):
    """decode: the logits of every step, [steps, sequences, vocabulary].  prompt: the logits of the last token, and for a fresh Llama prompt the keys and values that the cache now
    holds.  image: its features."""
    case, model = state["case"], state["model"]
    if case["kind"] == "image":
        return model(state["pixels"], state["grid"])
    if case["kind"] == "decode":
        return _decode(model, state["tokens"], state["caches"], recurrent=case["model"] == "lagelorn")
    cache = state.get("cache") or model.make_cache()
    logits = model.step(state["prompt"], cache)[2].clone()
    if case["model"] != "llama":
        cache[0].page_manager.release()
        return logits
    if case["cached"]:
        for layer in cache:
            layer.trim(case["tokens"])
        return logits
    return {"logits": logits, "keys": [c.keys[0, :, :c.offset] for c in cache], "values": [c.values[0, :, :c.offset] for c in cache]}


def _decode(model, tokens, caches, recurrent):
    steps, B = tokens.shape
    if recurrent:   # a recurrent state cannot go back: the steps run on forks of the sequences, as requests behind a shared prefix do
        forks = [c[0].page_manager.fork() for c in caches]
        caches = [[type(c)(seq, i) for i, c in enumerate(cache)] for cache, seq in zip(caches, forks)]
    out = None
    for t in range(steps):
        logits = model.step(tokens[t], caches[0])[2] if B == 1 else model.step_batch(tokens[t], caches)[2]
        if out is None:
            out = torch.empty((steps, B, logits.shape[-1]), dtype=logits.dtype, device=logits.device)
        out[t].copy_(logits.view(B, -1))
    for cache in caches:
        if recurrent:
            cache[0].page_manager.release()
        else:
            for layer in cache:
                layer.trim(steps)
    return out


# ------------------------------------------------------------------ what a pass cannot do without
def _layer_params(case):
    """(weights of one layer that every row multiplies, weights of its experts and how many one row uses, numbers cached per token and layer)."""
    if case["model"] == "llama":
        s = LLAMA[case["size"]]
        D = s["hidden_size"] // s["num_attention_heads"]
        kv = 2 * s["num_key_value_heads"] * D
        return s["hidden_size"] * (2 * s["hidden_size"] + kv + 3 * s["intermediate_size"]), None, kv
    if case["model"] == "taduzen":
        s = TADUZEN[case["size"]]
        W, HD = s["width"], s["heads"] * DIM
        mix = W * HD * 2 + W * LATENT + 2 * HD * LATENT
        if "experts" not in s:
            return mix + 2 * W * s["ff"], None, LATENT
        return mix + 3 * W * s["shared"], (3 * W * s["ff"], s["experts"], s["top"]), LATENT
    s = LAGELORN[case["size"]]
    W, HD, d = s["width"], s["heads"] * DIM, s["delta"]
    delta = W * (2 * d["kv_heads"] * DIM + 3 * d["heads"] * d["vdim"])
    parallel = W * (7 * HD + s["kv_heads"] * DIM) + s["rank"] * (W + HD)
    return (delta + parallel) // 2 + 3 * W * s["ff"] + 2 * W * s["side"], None, s["kv_heads"] * DIM   # the mean of the two kinds of layers; half of them cache keys and values


def work(case):
    """Bytes: the weights once per step (a step's rows share them; a mixture's as far as its rows choose them), the cached keys and values of every row's sequence, the logits.  Flops: a row's products and its
    scores.  Recurrent states are read and written once per step."""
    if case["kind"] == "image":
        n, H, I, L = case["height"] * case["width"], VISION["hidden_size"], VISION["intermediate_size"], VISION["depth"]
        params = 1176 * H + L * (4 * H * H + 3 * H * I)
        merger = 4 * H * (4 * H + VISION["out_hidden_size"])
        return {"bytes": 2 * (params + merger + n * 1176 + n // 4 * VISION["out_hidden_size"]), "flops": 2 * n * params + n // 2 * merger + 4 * n * H * (n + 7 * min(n, 64))}
    per, experts, cached = _layer_params(case)
    width = (LLAMA[case["size"]]["hidden_size"] if case["model"] == "llama" else {"taduzen": TADUZEN, "lagelorn": LAGELORN}[case["model"]][case["size"]]["width"])
    weight = {"int4": 0.5625, "int8": 1.0625}.get(case["weights"], 2.0)
    heads = DIM if case["model"] != "llama" else width // LLAMA[case["size"]]["num_attention_heads"]
    scores = 4 * heads * (LLAMA[case["size"]]["num_attention_heads"] if case["model"] == "llama" else {"taduzen": TADUZEN, "lagelorn": LAGELORN}[case["model"]][case["size"]]["heads"])
    if case["kind"] == "decode":
        steps, rows, seen = case["steps"], case["batch"], sum(_lengths(case)) + case["batch"] * case["steps"] // 2
        outputs = rows * VOCAB
    else:
        steps, rows, seen = 1, case["tokens"], case["cached"] + case["tokens"]
        outputs = VOCAB
    read, multiplied = LAYERS * per, LAYERS * per
    if experts:
        one, n, top = experts
        read += LAYERS * one * n * (1 - (1 - top / n) ** rows)
        multiplied += LAYERS * one * top
    state = 0
    if case["model"] == "lagelorn":
        s = LAGELORN[case["size"]]
        state = LAYERS // 2 * 4 * DIM * (s["delta"]["heads"] * s["delta"]["vdim"] + s["heads"] * DIM) * 2 * (case.get("batch", 1))
    pairs = seen if case["kind"] == "decode" else rows * (case["cached"] + (rows + 1) // 2)
    caching = LAYERS // 2 if case["model"] == "lagelorn" else LAYERS
    head_rows = rows if case["kind"] == "decode" else 1
    return {"bytes": steps * (weight * (read + width * VOCAB) + 2 * caching * cached * (seen + rows) + 2 * outputs + state),
            "flops": steps * (2 * rows * multiplied + 2 * head_rows * width * VOCAB + caching * scores * pairs)}


def tolerance(case):
    """Measured against `exact`: float16 Llama 0.0011, bfloat16 Llama 0.008 to 0.0095, Taduzen 0.0018 (its norms bound every number), Lagelorn 0.0042, the vision tower 0.013.  About four times that; rounding in
    another order moves two results apart by no more than twice each one's error, so the two largest stop at 0.03."""
    rel = 0.03 if case["kind"] == "image" else {"taduzen": 0.008, "lagelorn": 0.017}.get(case["model"], 0.0045 if case["weights"] == "f16" else 0.03)
    return {"rel": rel, "max": min(0.3, 20 * rel)}


# ------------------------------------------------------------------ the same in 64 bits
def _mm(x, w):
    return x @ w.double().t()


def _unit(x, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _attend(q, k, v, scale, window=None, chunk=None, bias=None, sink=None):
    """q [n, H, D], k [n, G, D], v [n, G, V] of one sequence -> [n, H, V], every query on the keys up to its own.  bias [H, distance]; sink [H]: one more score without a value."""
    n, H, _ = q.shape
    r = H // k.shape[1]
    out = torch.empty(n, H, v.shape[2], dtype=q.dtype, device=q.device)
    for lo in range(0, n, 512):
        i, j = torch.arange(lo, min(lo + 512, n), device=q.device)[:, None], torch.arange(min(lo + 512, n), device=q.device)[None]
        seen = j <= i
        if window is not None:
            seen &= i - j < window
        if chunk is not None:
            seen &= i // chunk == j // chunk
        for g in range(k.shape[1]):
            s = q[lo:lo + 512, g * r:(g + 1) * r].transpose(0, 1) @ k[:j.shape[1], g].t() * scale      # [r, rows, keys]
            if bias is not None:
                s = s + bias[g * r:(g + 1) * r][:, (i - j).clamp(min=0)]
            s = s.masked_fill(~seen, -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[g * r:(g + 1) * r, None, None].expand(r, s.shape[1], 1)], -1)
            out[lo:lo + 512, g * r:(g + 1) * r] = (torch.softmax(s, -1)[..., :j.shape[1]] @ v[:j.shape[1], g]).transpose(0, 1)
    return out


def _dequantised(w, name, bits):
    if not bits:
        return w[name + ".weight"]
    words, scale, bias = w[name + ".weight"], w[name + ".scales"].double(), w[name + ".biases"].double()
    codes = words.view(torch.uint8)
    if bits == 4:
        codes = torch.stack([codes & 15, codes >> 4], -1).view(words.shape[0], -1)
    g = codes.view(words.shape[0], -1, 64).double()
    return (g * scale[..., None] + bias[..., None]).view(words.shape[0], -1)


def _llama_exact(case, w, cfg, ids):
    """ids [S, n] -> (hidden [S, n, H] behind the last norm, keys, values per layer [S, G, n, D])."""
    bits, eps = (cfg["quantization"] or {}).get("bits"), cfg["rms_norm_eps"]
    nh, G = cfg["num_attention_heads"], cfg["num_key_value_heads"]
    D = cfg["hidden_size"] // nh
    S, n = ids.shape
    angle = torch.arange(n, device="cuda", dtype=torch.float64)[:, None] * cfg["rope_theta"] ** (-torch.arange(0, D, 2, device="cuda", dtype=torch.float64) / D)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def turn(x):
        a, b = x[..., :D // 2], x[..., D // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    def linear(x, name):
        return _mm(x, _dequantised(w, name, bits))

    x = _dequantised(w, "model.embed_tokens", bits)[ids].double()
    keys, values = [], []
    for i in range(LAYERS):
        p = f"model.layers.{i}."
        h = _unit(x, eps) * w[p + "input_layernorm.weight"].double()
        q, k, v = (linear(h, p + f"self_attn.{c}_proj").view(S, n, -1, D) for c in "qkv")
        q, k = turn(q), turn(k)
        keys.append(k.transpose(1, 2)), values.append(v.transpose(1, 2))
        y = torch.stack([_attend(q[s], k[s], v[s], D ** -0.5) for s in range(S)]).view(S, n, nh * D)
        x = x + linear(y, p + "self_attn.o_proj")
        h = _unit(x, eps) * w[p + "post_attention_layernorm.weight"].double()
        x = x + linear(_silu(linear(h, p + "mlp.gate_proj")) * linear(h, p + "mlp.up_proj"), p + "mlp.down_proj")
    return _unit(x, eps) * w["model.norm.weight"].double(), _dequantised(w, "lm_head", bits), keys, values


def _taduzen_exact(case, w, cfg, ids):
    size, eps = TADUZEN[case["size"]], cfg["norm"]["eps"]
    S, n = ids.shape
    H = size["heads"]

    def norm(x, name):
        return torch.tanh(w[name + ".alpha"].double() * x) * w[name].double() + w[name + ".b"].double()

    def gated(h, p):
        return _mm(_silu(_mm(h, w[p + "gate"])) * _mm(h, w[p + "up"]), w[p + "down"])

    x = w["embed"][ids].double()
    for i in range(LAYERS):
        p = f"l{i}."
        h = norm(x, p + "norm1")
        c = _unit(_mm(h, w[p + "mix.dkv"]), eps) * w[p + "mix.dkv.norm"].double()
        q, k, v = _mm(h, w[p + "mix.q"]).view(S, n, H, DIM), _mm(c, w[p + "mix.uk"]).view(S, n, H, DIM), _mm(c, w[p + "mix.uv"]).view(S, n, H, DIM)
        y = torch.stack([_attend(q[s], k[s], v[s], DIM ** -0.5, window=4096) for s in range(S)]).view(S, n, -1)
        x = x + norm(_mm(y, w[p + "mix.o"]), p + "norm1b")
        h = norm(x, p + "norm2")
        if "experts" not in size:
            y = _mm(torch.relu(_mm(h, w[p + "mlp.up"])).square(), w[p + "mlp.down"])
        else:
            y = gated(h, p + "mlp.shared.") * torch.sigmoid(_mm(h, w[p + "mlp.shared.sg"]))
            chosen, flat, out = w[p + "mlp.table"][ids].view(S * n, -1), h.reshape(S * n, -1), y.view(S * n, -1)
            for e in range(size["experts"]):
                rows = (chosen == e).any(1).nonzero().flatten()
                if len(rows):
                    out[rows] += gated(flat[rows], f"{p}mlp.e{e}.") / size["top"]
        x = x + norm(y, p + "norm2b")
    return norm(x, "final.norm"), w["head"], None, None


def _lagelorn_exact(case, w, cfg, ids):
    size, eps, alpha = LAGELORN[case["size"]], cfg["norm"]["eps"], cfg["postln_alpha"]
    S, n = ids.shape
    H, G, d, side = size["heads"], size["kv_heads"], size["delta"], size["side"]
    half, far = 16, 128   # the distance table: 32 rows, one per distance for the first half, then logarithmic up to `far`
    at = torch.tensor([k if k < half else min(31, half + math.floor(math.log(k / half) / math.log(far / half) * half)) for k in range(n)], device="cuda")

    def rms(x, name):
        return _unit(x, eps) * w[name].double()

    def back(x, by=1):
        return torch.cat([torch.zeros_like(x[:, :by]), x[:, :n - by]], 1) if by else x

    def delta(h, p):
        def conv(c):
            y, f = _mm(h, w[p + c]), w[p + c + ".conv"].double()
            return _silu(sum(back(y, f.shape[1] - 1 - j) * f[:, j] for j in range(f.shape[1]) if f.shape[1] - 1 - j < n))
        hd, gd, V = d["heads"], d["kv_heads"], d["vdim"]
        q, k, v = conv("q").view(S, n, gd, DIM), conv("k").view(S, n, gd, DIM), conv("v").view(S, n, hd, V)
        q, k = ((z * torch.rsqrt(z.square().sum(-1, keepdim=True) + 1e-6)).repeat_interleave(hd // gd, 2) for z in (q, k))
        decay = torch.exp(-torch.exp(w[p + "A_log"].double()) * torch.nn.functional.softplus(_mm(h, w[p + "a"]) + w[p + "dt_bias"].double()))
        beta = torch.sigmoid(_mm(h, w[p + "b"]))
        M, o = torch.zeros(S, hd, DIM, V, dtype=torch.float64, device="cuda"), torch.empty_like(v)
        for t in range(n):
            M = M * decay[:, t, :, None, None]
            u = beta[:, t, :, None] * (v[:, t] - (M * k[:, t, :, :, None]).sum(2))
            M = M + k[:, t, :, :, None] * u[:, :, None]
            o[:, t] = (M * q[:, t, :, :, None]).sum(2) * DIM ** -0.5
        o = (_unit(o, eps) * w[p + "norm"].double()).view(S, n, -1)
        return _mm(o * _silu(_mm(h, w[p + "g"])), w[p + "o"])

    def attention(h, p):
        raw = _mm(h, w[p + "k"]) + w[p + "k.b"].double()
        q, k = rms(_mm(h, w[p + "q"]) + w[p + "q.b"].double(), p + "q.norm").view(S, n, H, DIM), rms(raw, p + "k.norm").view(S, n, G, DIM)
        v, bias = raw.view(S, n, G, DIM), w[p + "rel"].double()[at].t().contiguous()
        y = torch.stack([_attend(q[s], k[s], v[s], DIM ** -0.5, chunk=4096, bias=bias, sink=w[p + "sink"].double()) for s in range(S)])
        return _mm(y.view(S, n, -1), w[p + "o"])

    def time_mix(h, p):
        mix = {c: h + (back(h) - h) * w[p + "mu." + c].double() for c in "rkvgw"}
        r, k, v = (_mm(mix[c], w[p + c]).view(S, n, H, DIM) for c in "rkv")
        decay = torch.exp(-torch.exp(_mm(torch.tanh(_mm(mix["w"], w[p + "w1"])), w[p + "w2"]) + w[p + "w0"].double())).view(S, n, H, DIM)
        u, M, o = w[p + "u"].double(), torch.zeros(S, H, DIM, DIM, dtype=torch.float64, device="cuda"), torch.empty_like(v)
        for t in range(n):
            o[:, t] = (M * r[:, t, :, :, None]).sum(2) + (r[:, t] * u * k[:, t]).sum(-1, keepdim=True) * v[:, t]
            M = M * decay[:, t, :, :, None] + k[:, t, :, :, None] * v[:, t, :, None]
        return _mm(_unit(o, eps).view(S, n, -1) * w[p + "norm"].double() * _silu(_mm(mix["g"], w[p + "g"])), w[p + "o"])

    x = w["embed"][ids].double() + w["pos"][:n].double()
    for i in range(LAYERS):
        p = f"l{i}."
        y = delta(x, p + "mix.") if i % 2 == 0 else 0.7 * (attention(x, p + "mix.left.") + time_mix(x, p + "mix.right."))
        x = rms(alpha * x + y, p + "norm1")
        y = _mm(_gelu(_mm(x, w[p + "mlp.gate"]) + w[p + "mlp.gate.b"].double()) * (_mm(x, w[p + "mlp.up"]) + w[p + "mlp.up.b"].double()), w[p + "mlp.down"]) + w[p + "mlp.down.b"].double()
        x = rms(alpha * x + y, p + "norm2")
        e = w["side.embed"][ids][..., i * side:(i + 1) * side].double()
        x = x + rms(_mm(_gelu(_mm(x, w[p + "side.gate"])) * e, w[p + "side.proj"]), p + "side.norm")
    return rms(x, "final.norm"), w["head"], None, None


def _vision_exact(case, w, pixels):
    c, h, wide, t = VISION, case["height"], case["width"], "vision_tower."
    H, D, n = c["num_heads"], c["hidden_size"] // c["num_heads"], h * wide
    row, col = (torch.from_numpy(np.ascontiguousarray(a.reshape(h // 2, 2, wide // 2, 2).transpose(0, 2, 1, 3).reshape(-1))).cuda() for a in np.mgrid[:h, :wide])   # 2 x 2 blocks, row by row
    f = 10000.0 ** (-torch.arange(0, D // 2, 2, device="cuda", dtype=torch.float64) / (D // 2))
    angle = torch.cat([row[:, None] * f, col[:, None] * f], 1)[:, None]
    window = row // 8 * (wide + 7) + col // 8

    def linear(x, name):
        return _mm(x, w[name + ".weight"]) + w[name + ".bias"].double()

    def norm(x, name):
        return _unit(x, 1e-6) * w[name + ".weight"].double()

    def turn(x):
        a, b = x[..., :D // 2], x[..., D // 2:]
        return torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin()], -1)

    x = _mm(pixels.double(), w[t + "patch_embed.proj.weight"].view(c["hidden_size"], -1))
    for i in range(c["depth"]):
        p = f"{t}blocks.{i}."
        q, k, v = linear(norm(x, p + "norm1"), p + "attn.qkv").view(n, 3, H, D).unbind(1)
        s = turn(q).transpose(0, 1) @ turn(k).permute(1, 2, 0) * D ** -0.5
        if i not in (7, 15, 23, 31):
            s = s.masked_fill(window[:, None] != window[None], -math.inf)
        x = x + linear((torch.softmax(s, -1) @ v.transpose(0, 1)).transpose(0, 1).reshape(n, -1), p + "attn.proj")
        y = norm(x, p + "norm2")
        x = x + linear(_silu(linear(y, p + "mlp.gate_proj")) * linear(y, p + "mlp.up_proj"), p + "mlp.down_proj")
    y = linear(norm(x, t + "merger.ln_q").view(n // 4, -1), t + "merger.mlp.0")
    return linear(y * 0.5 * (1 + torch.erf(y / math.sqrt(2))), t + "merger.mlp.2")


@torch.no_grad()
def exact(case, seed):
    if case["kind"] == "image":
        return _vision_exact(case, _vision(seed), _pixels(case, seed))
    cfg, w = _checkpoint(case, seed)
    ids = _tokens(case, seed).long().cuda()
    hidden, head, keys, values = {"llama": _llama_exact, "taduzen": _taduzen_exact, "lagelorn": _lagelorn_exact}[case["model"]](case, w, cfg, ids)

    def logits(x):
        z = _mm(x, head)
        return 30.0 * torch.tanh(z / 30.0) if case["model"] == "lagelorn" else z

    if case["kind"] == "decode":
        return logits(torch.stack([hidden[i, n:n + case["steps"]] for i, n in enumerate(_lengths(case))], dim=1))
    last = logits(hidden[0, -1])
    if case["model"] != "llama" or case["cached"]:
        return last
    return {"logits": last, "keys": [k[0] for k in keys], "values": [v[0] for v in values]}
