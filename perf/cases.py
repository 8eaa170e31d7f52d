"""Workloads of the library as a program sees them: prompts, decoding, batches, drafts and single products, through the public entry points
of espresso_amd, with seeded weights and tokens and a plain 64-bit statement of what each returns.

Kinds of case:
  product    one weight matrix against a few rows of activations held by the host (ops.Matrix.gemv)
  decode     a prompt that is already in the caches is continued greedily by `new` tokens, one at a time
  prefill    a prompt from an empty sequence up to the logits of the next token
  turn       the next turn of a conversation: more tokens behind a cached prefix, logits at the last few of them
  generate   a prompt and the greedy tokens behind it in one call
  batch      several sequences in lock step
  draft      the exact two-token loop: a one-layer draft proposes, the target verifies

Weights are normally distributed and quantised as GGUF files hold them.  Their output heads favour one successor for each token by a wide
margin, as those of a trained model do, so that greedy tokens do not hang on the last bits of a sum.
"""
import json
import math
import os
import tempfile

import numpy as np
import torch

import espresso_amd._lib as lib
import espresso_amd.engine as engine
import espresso_amd.llama as llama
import espresso_amd.ops as ops
import espresso_amd.synthetic as synthetic

# layers, heads, key/value heads, width, head size, feed-forward, vocabulary, rotary base (the registry's models and the benchmark's)
MODELS = {
    "stories": (6, 12, 12, 768, 64, 2048, 32000, 10000.0),
    "smolLM_135m": (30, 9, 3, 576, 64, 1536, 49152, 10000.0),
    "tinyLlama_1_1b": (22, 32, 4, 2048, 64, 5632, 32000, 10000.0),
    "llama3_2_1b": (16, 32, 8, 2048, 64, 8192, 128256, 500000.0),
    "llama3_2_3b": (28, 24, 8, 3072, 128, 8192, 128256, 500000.0),
    "llama3_8b": (32, 32, 8, 4096, 128, 14336, 128256, 500000.0),
}
FORMATS = {"f16": lib.FORMAT_F16, "q8_0": lib.FORMAT_Q8_0, "q4_0": lib.FORMAT_Q4_0, "q4_k": lib.FORMAT_Q4_K}
BLOCK = {"f16": (1, 2), "q8_0": (32, 34), "q4_0": (32, 18), "q4_k": (256, 144)}   # elements, bytes
STD = 0.02


def listed():
    return [
        # one call of the matrix handle a host program holds for a projection
        {"name": "product 4096x4096 q4_k", "kind": "product", "format": "q4_k", "rows": 4096, "cols": 4096, "batch": 2},
        # a small model answers a short prompt: every launch counts
        {"name": "decode stories q8_0", "kind": "decode", "model": "stories", "layers": 6, "format": "q8_0", "kv": "f32", "prompt": 16, "new": 64, "context": 256},
        # the headline workload: an 8B model decodes behind a 512-token prompt
        {"name": "decode 8b q4_k", "kind": "decode", "model": "llama3_8b", "layers": 32, "format": "q4_k", "kv": "f16", "prompt": 512, "new": 32, "context": 1024},
        # the end of a long conversation with a small model
        {"name": "decode 1b q4_0 long", "kind": "decode", "model": "llama3_2_1b", "layers": 16, "format": "q4_0", "kv": "f16", "prompt": 1900, "new": 32, "context": 2048},
        # the headline workload's prompt, on a quarter of its layers
        {"name": "prefill 8b q4_k", "kind": "prefill", "model": "llama3_8b", "layers": 8, "format": "q4_k", "kv": "f16", "prompt": 512, "context": 1024},
        # a document is read: several blocks and a ragged last one
        {"name": "prefill 3b q4_k long", "kind": "prefill", "model": "llama3_2_3b", "layers": 28, "format": "q4_k", "kv": "f16", "prompt": 1777, "context": 2048},
        # a chat message and its short answer with the smallest model, whose sizes fit no power of two
        {"name": "generate smol f16", "kind": "generate", "model": "smolLM_135m", "layers": 30, "format": "f16", "kv": "f32", "prompt": 77, "new": 24, "context": 512},
        # the next message of a conversation, with the logits of its last tokens
        {"name": "turn tinyllama q8_0", "kind": "turn", "model": "tinyLlama_1_1b", "layers": 22, "format": "q8_0", "kv": "f16", "prefix": 700, "count": 93, "want": 4, "context": 2048},
        # a server's batch, on a quarter of the model's layers
        {"name": "batch 8b q4_k", "kind": "batch", "model": "llama3_8b", "layers": 8, "format": "q4_k", "kv": "f16", "sequences": 16, "prompt": 60, "new": 24, "context": 512},
        # speculative decoding of the small model with a draft that is mostly right
        {"name": "draft stories f16", "kind": "draft", "model": "stories", "layers": 6, "format": "f16", "kv": "f32", "prompt": 16, "new": 64, "context": 256},
        # both layered designs: a prompt and an answer
        {"name": "generate ranavik d2048", "kind": "generate", "model": "d2048", "precision": "bf16", "window": 1024, "prompt": 600, "new": 24, "context": 1024},
        {"name": "generate forovik d2048", "kind": "generate", "model": "forovik-d2048", "precision": "bf16", "window": 256, "prompt": 1100, "new": 24, "context": 1536},
    ]


def draw(rng):
    """Another case of the same ranges; none costs more than the largest listed one."""
    most = max(_cost(c) for c in listed())
    while True:
        c = _draw(rng)
        if _cost(c) <= most:
            return c


def _spread(rng, low, high):
    """A whole number, spread evenly over the logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _draw(rng):
    kind = rng.choice(["product", "decode", "decode", "prefill", "prefill", "turn", "generate", "batch", "draft", "layered", "layered"])
    if kind == "product":
        m = MODELS[rng.choice(sorted(MODELS))]
        rows, cols = rng.choice([(m[3], m[3]), (m[2] * m[4], m[3]), (m[5], m[3]), (m[3], m[5])])
        fmt = rng.choice([f for f in FORMATS if cols % BLOCK[f][0] == 0])
        return {"kind": "product", "format": fmt, "rows": rows, "cols": cols, "batch": rng.choice([1, 1, 2, 3, 4, 7, 8, 16, 40])}
    if kind == "layered":
        sizes = sorted(synthetic.LAYERED_SIZES) + sorted(synthetic.SEQUENTIAL_SIZES)
        c = {"kind": rng.choice(["generate", "prefill", "batch"]), "model": rng.choice(sizes), "precision": rng.choice(["bf16", "bf16", "bf16", "f32"]),
             "window": rng.choice([256, 1024])}
        if c["precision"] == "f32":
            c["model"] = rng.choice(["d768", "forovik-d768"])
    else:
        name = rng.choice(["stories", "stories"] if kind == "draft" else sorted(MODELS))
        m = MODELS[name]
        layers = rng.randint(4, 8) if name == "llama3_8b" else m[0]
        c = {"kind": kind, "model": name, "layers": layers, "format": rng.choice([f for f in FORMATS if m[3] % BLOCK[f][0] == 0]), "kv": rng.choice(["f16", "f16", "f32"])}
    longest = 240 if c["model"] == "stories" else 1800
    if c["kind"] == "batch":
        c.update(sequences=rng.choice([2, 3, 4, 8, 13, 16]), prompt=_spread(rng, 4, min(longest // 2, 200)), new=rng.randint(8, 32))
    elif c["kind"] == "prefill":
        c.update(prompt=_spread(rng, 5, longest))
    elif c["kind"] == "turn":
        c.update(prefix=_spread(rng, 10, longest // 2), count=_spread(rng, 3, longest // 2), want=1)
        c["want"] = rng.randint(1, min(8, c["count"]))
    else:
        c.update(prompt=_spread(rng, 4, longest - 48), new=rng.randint(9, 48))
    c["context"] = min(256 if c["model"] == "stories" else 2048, c.get("prompt", 0) + c.get("prefix", 0) + c.get("count", 0) + c.get("new", 0) + rng.choice([1, 17, 200, 1024]))
    return c


# ---- what the work is --------------------------------------------------------------------------------------------------------------
def _bytes(fmt, n):
    return n // BLOCK[fmt][0] * BLOCK[fmt][1]


def _config(case):
    """The configuration of a layered case."""
    config = json.loads(json.dumps((synthetic.LAYERED_SIZES if case["model"] in synthetic.LAYERED_SIZES else synthetic.SEQUENTIAL_SIZES)[case["model"]][0]))
    for layer in config["layers"]:
        if "mask" in layer["mixer"]:
            layer["mixer"]["mask"]["size"] = case["window"]
    return config


def _is_layered(case):
    return "precision" in case


def _sizes(case):
    """(weights in a step, their bytes, bytes cached per token and read again by every later one, vocabulary, heads' share of attention per pair of tokens in flops)."""
    if _is_layered(case):
        config, each = _config(case), 2 if case["precision"] == "bf16" else 4
        n = sum(math.prod(s) for k, s in _tensors(config).items() if len(s) == 2 and not k.endswith(".conv") and (k != "embed" or config["architecture"] == "Forovik"))
        cached = sum((m["kv_rank"] + m["rot_dim"]) if "kv_rank" in m else m["kv_heads"] * (m["dim"] + m["vdim"]) if "kv_heads" in m else 0 for m in (l["mixer"] for l in config["layers"]))
        return n, n * each, cached * each, config["vocab"], sum(4 * m["heads"] * m["dim"] for m in (l["mixer"] for l in config["layers"]) if "mask" in m)
    m = MODELS[case["model"]]
    layer = m[3] * m[4] * (2 * m[1] + 2 * m[2]) + 3 * m[3] * m[5]
    n = case["layers"] * layer + m[6] * m[3]
    return n, _bytes(case["format"], n), case["layers"] * 2 * m[2] * m[4] * (2 if case["kv"] == "f16" else 4), m[6], case["layers"] * 4 * m[1] * m[4]


def work(case):
    if case["kind"] == "product":
        n = case["rows"] * case["cols"]
        return {"bytes": _bytes(case["format"], n) + case["batch"] * (2 * case["cols"] + 4 * case["rows"]), "flops": 2 * n * case["batch"]}
    n, weights, cached, vocab, pair = _sizes(case)
    head = vocab * (_config(case)["width"] if _is_layered(case) else MODELS[case["model"]][3])
    total = {"bytes": 0, "flops": 0}

    def tokens(start, count, sequences, heads):   # one pass of `count` tokens behind `start` cached ones, `heads` logits rows
        total["bytes"] += weights + sequences * cached * (start + count)
        total["flops"] += sequences * (2 * (n - head) * count + pair * count * (start + count / 2)) + 2 * head * heads

    kind, prompt, new, batch = case["kind"], case.get("prompt", 0), case.get("new", 0), case.get("sequences", 1)
    if kind == "turn":
        tokens(case["prefix"], case["count"], 1, case["want"])
    elif kind == "decode":
        for i in range(new + 1):
            tokens(prompt - 1 + i, 1, 1, 1)
    else:
        for _ in range(batch):
            tokens(0, prompt, 1, 1)
        for i in range(new):
            tokens(prompt + i, 1, batch, batch)
    total["bytes"] += 4 * vocab
    return total


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50) * (8 if _is_layered(case) and case["precision"] == "f32" else 1)


def tolerance(case):
    """About four times what the sums' order and the operands' roundings were seen to cost against 64 bits: products of more than a few rows
    see weights rounded to fp16 (2e-4), whole models fp16 activations or caches (6e-4), layered ones bf16 operands (4e-3)."""
    if case["kind"] == "product":
        return {"rel": 4e-5, "max": 4e-4} if case["batch"] <= 2 else {"rel": 1e-3, "max": 1e-2}
    if _is_layered(case):
        return {"rel": 1.6e-2, "max": 0.2} if case["precision"] == "bf16" else {"rel": 2e-5, "max": 4e-4}
    return {"rel": 2.5e-3, "max": 4e-2}


# ---- seeded tensors ----------------------------------------------------------------------------------------------------------------
def _normal(seed, index, *shape):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed % (1 << 30)) * 4096 + index)
    return torch.randn(*shape, generator=g, device="cuda")


def _successors(seed, vocab):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed % (1 << 30)) * 4096 + 4095)
    return torch.randperm(vocab, generator=g, device="cuda")


def _tokens(seed, stream, count, vocab):
    return np.random.default_rng([seed % (1 << 30), stream]).integers(0, vocab, count).astype(np.uint32)


def _pack(fmt, w):
    """Rows of weights as GGUF blocks: uint8 [rows, bytes]."""
    rows, cols = w.shape
    f16 = lambda t: t.half().unsqueeze(-1).view(torch.uint8)  # noqa: E731
    if fmt == "f16":
        return w.half().view(torch.uint8)
    if fmt == "q8_0":
        b = w.view(rows, cols // 32, 32)
        d = (b.abs().amax(-1) / 127).half().float()
        q = torch.round(b / d.clamp_min(1e-8)[..., None]).clamp(-127, 127).to(torch.int8).view(torch.uint8)
        return torch.cat([f16(d), q], -1).view(rows, -1)
    if fmt == "q4_0":
        b = w.view(rows, cols // 32, 32)
        far = b.gather(-1, b.abs().argmax(-1, keepdim=True))[..., 0]
        d = (far / -8).half().float()
        safe = torch.where(d == 0, torch.ones_like(d), d)
        q = (torch.round(b / safe[..., None]) + 8).clamp(0, 15).to(torch.uint8)
        return torch.cat([f16(d), q[..., :16] | (q[..., 16:] << 4)], -1).view(rows, -1)
    b = w.view(rows, cols // 256, 8, 32)
    low = (-b.amin(-1)).clamp_min(0)                      # sub-blocks: scale * q - low
    scale = (b.amax(-1) + low) / 15
    d, dm = (scale.amax(-1) / 63).half().float(), (low.amax(-1) / 63).half().float()
    sc = torch.round(scale / d.clamp_min(1e-8)[..., None]).clamp(0, 63)
    mn = torch.round(low / dm.clamp_min(1e-8)[..., None]).clamp(0, 63)
    step = (d[..., None] * sc)[..., None]
    q = torch.round((b + (dm[..., None] * mn)[..., None]) / step.clamp_min(1e-8)).clamp(0, 15).to(torch.uint8)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    head = torch.cat([sc[..., :4] | ((sc[..., 4:] >> 4) << 6), mn[..., :4] | ((mn[..., 4:] >> 4) << 6), (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], -1)
    pairs = q.view(rows, cols // 256, 4, 2, 32)
    nibbles = (pairs[..., 0, :] | (pairs[..., 1, :] << 4)).reshape(rows, cols // 256, 128)
    return torch.cat([f16(d), f16(dm), head, nibbles], -1).view(rows, -1)


def _unpack(fmt, raw, cols):
    """What the blocks stand for, in 64 bits."""
    rows = raw.shape[0]
    f64 = lambda t: t.contiguous().view(torch.float16).double()  # noqa: E731
    if fmt == "f16":
        return f64(raw)
    if fmt == "q8_0":
        b = raw.view(rows, -1, 34)
        return (f64(b[..., :2]) * b[..., 2:].contiguous().view(torch.int8).double()).view(rows, cols)
    if fmt == "q4_0":
        b = raw.view(rows, -1, 18)
        q = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], -1).double() - 8
        return (f64(b[..., :2]) * q).view(rows, cols)
    b = raw.view(rows, -1, 144)
    s = b[..., 4:16]
    sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], -1)
    mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1)
    n = b[..., 16:].reshape(rows, -1, 4, 1, 32)
    q = torch.cat([n & 15, n >> 4], 3).reshape(rows, -1, 8, 32)
    return ((f64(b[..., 0:2]) * sc.double())[..., None] * q.double() - (f64(b[..., 2:4]) * mn.double())[..., None]).reshape(rows, cols)


_LINEAR = ("wq", "wk", "wv", "wo", "w1", "w2", "w3")


def _shapes(m):
    a, k, d, h = m[1] * m[4], m[2] * m[4], m[3], m[5]
    return {"wq": (a, d), "wk": (k, d), "wv": (k, d), "wo": (d, a), "w1": (h, d), "w2": (d, h), "w3": (h, d)}


def _linear(case, seed, layer, name):
    m = MODELS[case["model"]]
    rows, cols = _shapes(m)[name]
    std = STD / math.sqrt(2 * case["layers"]) if name in ("wo", "w2") else STD
    return _pack(case["format"], _normal(seed, 16 + 8 * layer + _LINEAR.index(name), rows, cols) * std)


def _norm(seed, index, n):
    return (1 + 0.1 * _normal(seed, index, n)).half()


def _embedding(case, seed):
    m = MODELS[case["model"]]
    return _normal(seed, 0, m[6], m[3]).half()


def _head(case, seed, wrong=0):
    """Output head: the row of a token's successor leans towards the token's embedding; one token in `wrong` has another successor."""
    m = MODELS[case["model"]]
    before = torch.argsort(_successors(seed, m[6]))
    if wrong:
        before = torch.where(torch.arange(m[6], device="cuda") % wrong == 0, before.roll(wrong), before)
    return _pack(case["format"], _normal(seed, 1, m[6], m[3]) * STD + 0.01 * _embedding(case, seed)[before].float())


def _host(t):
    return t.contiguous().view(torch.uint8).cpu().numpy()


def _llama(case, seed, layers=None, own=0, sequences=1, wrong=0):
    """A runtime with the case's weights; `own` shifts the seeds of the layers."""
    m = MODELS[case["model"]]
    layers = case["layers"] if layers is None else layers
    cfg = llama.MultiModelConfig(n_layer=layers, n_head=m[1], n_kv_head=m[2], d_model=m[3], head_dim=m[4], hidden_dim=m[5], vocab=m[6], max_seq=case["context"],
                                 norm_eps=1e-5, rope_theta=m[7])
    rt = llama.LlamaRuntime(cfg, kv_format=FORMATS["f16"] if case["kv"] == "f16" else lib.FORMAT_F32, max_sequences=sequences)
    fmt = FORMATS[case["format"]]
    rt.set_weight(0, llama.SLOT_TOKEN_EMBEDDING, lib.FORMAT_F16, _host(_embedding(case, seed)))
    rt.set_weight(0, llama.SLOT_FINAL_NORM, lib.FORMAT_F16, _host(_norm(seed, 2, m[3])))
    rt.set_weight(0, llama.SLOT_LM_HEAD, fmt, _host(_head(case, seed, wrong)))
    for l in range(layers):
        rt.set_weight(l, llama.SLOT_RMS_ATT, lib.FORMAT_F16, _host(_norm(seed, 1024 + l, m[3])))
        rt.set_weight(l, llama.SLOT_RMS_FFN, lib.FORMAT_F16, _host(_norm(seed, 2048 + l, m[3])))
        for name in _LINEAR:
            rt.set_weight(l, llama.LAYER_SLOTS[name], fmt, _host(_linear(case, seed, l + own, name)))
    rt.finalize()
    return rt


def _tensors(config):
    """Names and shapes of a layered model's weights."""
    d, out = config["width"], {"embed": (config["vocab"], config["width"]), "final.norm": (config["width"],)}
    if config["architecture"] == "Ranavik":
        out.update({"embed.norm": (d,), "head": (config["vocab"], d)})
    for i, layer in enumerate(config["layers"]):
        m, p = layer["mixer"], "l%d." % i
        h, mix = m["heads"], {}
        if layer["type"] == "retention":
            mix = {"q": (h * m["dim"], d), "k": (h * m["dim"], d), "v": (h * m["vdim"], d), "g": (h * m["vdim"], d)}
        elif layer["type"] == "latent_attention":
            mix = {"q": (h * (m["dim"] + m["rot_dim"]), d), "uk": (h * m["dim"], m["kv_rank"]), "uv": (h * m["vdim"], m["kv_rank"]), "sink": (h,), "g": (h, d)}
            if "kv_from" not in m:
                mix.update({"dkv": (m["kv_rank"] + m["rot_dim"], d), "dkv.norm": (m["kv_rank"],)})
        elif layer["type"] == "attention":
            mix = {"q": (h * m["dim"], d), "q.norm": (h * m["dim"],)}
            if "kv_from" not in m:
                mix.update({"k": (m["kv_heads"] * m["dim"], d), "k.norm": (m["kv_heads"] * m["dim"],), "v": (m["kv_heads"] * m["vdim"], d)})
        else:
            inner, shared = h * m["vdim"], m["groups"] * m["state"]
            mix = {"in": (2 * inner + 2 * shared + h, d), "conv": (inner + 2 * shared, m["conv"]), "conv.b": (inner + 2 * shared,), "dt_bias": (h,), "A_log": (h,), "D": (h,),
                   "norm": (inner,)}
        mix["o"] = (d, h * m["vdim"])
        out.update({p + "mix." + k: s for k, s in mix.items()})
        out[p + "norm1"] = (d,)
        if layer["mlp"]:
            ff = layer["mlp"]["ff"]
            out.update({p + "norm2": (d,), p + "mlp.gate": (ff, d), p + "mlp.up": (ff, d), p + "mlp.down": (d, ff)})
    return out


def _layered_tensor(config, seed, index, name, shape):
    """bf16 values: linears that keep the size of their inputs, decays and step sizes of a trained model's range."""
    x = _normal(seed, index, *shape)
    last = name.split(".")[-1]
    if name == "embed":
        pass
    elif name == "head":
        order = _successors(seed, config["vocab"])
        x = x * shape[1] ** -0.5 + 20.0 / shape[1] * _layered_tensor(config, seed, 0, "embed", shape)[torch.argsort(order)].float()
    elif last == "sink":
        x = 0.5 * x
    elif last == "A_log":
        x = torch.log(1 + 15 * torch.special.ndtr(x))
    elif last == "dt_bias":
        x = -6.9 + 4.6 * torch.special.ndtr(x)
    elif name.endswith("conv.b"):
        x = 0.1 * x
    elif len(shape) == 1:
        joins = config["architecture"] == "Forovik" and last in ("norm1", "norm2")   # how strongly a branch joins the stream
        x = (0.4 if joins else 1.0) + 0.1 * x
    else:
        x = x * shape[1] ** -0.5
    return x.bfloat16()


def _layered_weights(config, seed):
    """name -> tensor, one at a time; the embedding is the first."""
    for i, (name, shape) in enumerate(_tensors(config).items()):
        yield name, _layered_tensor(config, seed, i, name, shape)


def _layered(case, seed, sequences=1):
    config = _config(case)
    with tempfile.TemporaryDirectory() as path:
        with open(os.path.join(path, "config.json"), "w") as f:
            json.dump(config, f)
        header, at = {}, 0
        for name, shape in _tensors(config).items():
            n = 2 * math.prod(shape)
            header[name] = {"dtype": "BF16", "shape": list(shape), "data_offsets": [at, at + n]}
            at += n
        text = json.dumps(header).encode()
        with open(os.path.join(path, "model.safetensors"), "wb") as f:
            f.write(len(text).to_bytes(8, "little") + text)
            for _, t in _layered_weights(config, seed):
                f.write(_host(t).data)
        model = engine.RealModelInferenceEngine(engine.load_model_config(path, case["context"]), path,
                                                environment={"ESPRESSO_HIP_PRECISION": case["precision"], "ESPRESSO_HIP_MAX_SEQUENCES": str(sequences)})
    return model.runtime()


# ---- the cases ---------------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    ops.init()
    state = dict(case)
    if case["kind"] == "product":
        state["matrix"] = ops.Matrix(FORMATS[case["format"]], _host(_product_weights(case, seed)), case["rows"], case["cols"])
        state["x"] = _product_inputs(case, seed)
        return state
    sequences = case.get("sequences", 1)
    vocab = _sizes(case)[3]
    state["tokens"] = [_tokens(seed, s, case.get("prompt", 0) + case.get("prefix", 0) + case.get("count", 0), vocab) for s in range(sequences)]
    if sequences > 1:   # requests are not of one length
        state["tokens"] = [t[:max(1, t.size - 3 * s)] for s, t in enumerate(state["tokens"])]
    state["rt"] = rt = _layered(case, seed, sequences) if _is_layered(case) else _llama(case, seed, sequences=sequences)
    if case["kind"] == "draft":
        state["proposer"] = _llama(case, seed, layers=1, own=64, wrong=4)
    elif case["kind"] == "turn":
        rt.prefill(state["tokens"][0][:case["prefix"]])
    elif case["kind"] == "decode":
        rt.prefill(state["tokens"][0])
    return state


def run(state):
    kind = state["kind"]
    if kind == "product":
        return state["matrix"].gemv(state["x"])
    rt, tokens = state["rt"], state["tokens"][0]
    if kind == "prefill":
        rt.prefill(tokens)
        return {"logits": rt.logits(), "hidden": rt.last_hidden()}
    if kind == "turn":
        rt.set_visible(state["prefix"])
        return {"logits": rt.append(tokens[state["prefix"]:], want=range(state["count"] - state["want"], state["count"])), "hidden": rt.last_hidden()}
    if kind == "decode":
        rt.set_visible(tokens.size - 1)
        rt.advance(int(tokens[-1]))
        new = llama.continue_greedy(rt, state["new"])
        return {"tokens": np.array(new), "logits": rt.logits(), "hidden": rt.last_hidden()}
    if kind == "generate":
        new, _ = rt.generate(tokens, state["new"])
        return {"tokens": np.array(new), "logits": rt.logits(), "hidden": rt.last_hidden()}
    if kind == "batch":
        new, _ = llama.generate_batch(rt, state["tokens"], state["new"])
        last = len(new) - 1
        return {"tokens": np.array(new), "logits": rt.append(new[last][-1:], want=[0], sequence=last)[0]}
    new, _ = llama.generate_two_token(rt, state["proposer"], tokens, state["new"])
    rt.set_visible(tokens.size + len(new) - 1)
    return {"tokens": np.array(new), "logits": rt.append(new[-1:], want=[0])[0]}


# ---- the same in 64 bits -----------------------------------------------------------------------------------------------------------
def _product_weights(case, seed):
    return _pack(case["format"], _normal(seed, 0, case["rows"], case["cols"]) * STD)


def _product_inputs(case, seed):
    return np.random.default_rng([seed % (1 << 30), 1]).normal(0, 1, (case["batch"], case["cols"])).astype(np.float16)


def exact(case, seed):
    if case["kind"] == "product":
        w = _unpack(case["format"], _product_weights(case, seed), case["cols"])
        return (torch.from_numpy(_product_inputs(case, seed)).cuda().double() @ w.t().contiguous()).cpu().numpy()
    model = _Layered64(case, seed) if _is_layered(case) else _Llama64(case, seed)
    kind, new = case["kind"], case.get("new", 0)
    streams = [_tokens(seed, s, case.get("prompt", 0) + case.get("prefix", 0) + case.get("count", 0), model.vocab) for s in range(case.get("sequences", 1))]
    streams = [t[:max(1, t.size - 3 * s)] for s, t in enumerate(streams)]
    if kind in ("prefill", "turn"):
        want = case.get("want", 1)
        hidden = model.hidden(streams[0])
        logits = model.logits(hidden[-want:]).cpu().numpy()
        return {"logits": logits if kind == "turn" else logits[0], "hidden": hidden[-1].cpu().numpy()}
    if kind == "decode":
        got, hidden = model.greedy(streams[0], new, new)
        return {"tokens": got, "logits": model.logits(hidden[-1:])[0].cpu().numpy(), "hidden": hidden[-1].cpu().numpy()}
    if kind == "generate":   # the last token is chosen and not consumed
        got, hidden = model.greedy(streams[0], new, new - 1)
        return {"tokens": got, "logits": model.logits(hidden[-1:])[0].cpu().numpy(), "hidden": hidden[-1].cpu().numpy()}
    got, hidden = model.greedy(streams[-1], new, new)
    return {"tokens": None, "logits": model.logits(hidden[-1:])[0].cpu().numpy()}


def _rms64(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _turned(x, freqs, factor=1.0, interleaved=False):
    """x [tokens, heads, size]: the first 2 len(freqs) of every head turn with the position."""
    n = freqs.numel()
    a = torch.arange(x.shape[0], device="cuda", dtype=torch.float64)[:, None] * freqs
    c, s = torch.cos(a)[:, None] * factor, torch.sin(a)[:, None] * factor
    first, second = (slice(0, 2 * n, 2), slice(1, 2 * n, 2)) if interleaved else (slice(0, n), slice(n, 2 * n))
    out = x.clone()
    out[..., first], out[..., second] = x[..., first] * c - x[..., second] * s, x[..., second] * c + x[..., first] * s
    return out


def _weighted(scores, window=None, sink=None):
    """Softmax over the keys a query sees, [queries, keys]; `sink` joins the denominator."""
    n = scores.shape[-1]
    at = torch.arange(n, device="cuda")
    far = at[:, None] - at[None, :]
    scores = scores.masked_fill((far < 0) | (far >= (window or n)), -math.inf)
    if sink is None:
        return torch.softmax(scores, -1)
    return torch.softmax(torch.cat([scores, sink.expand(n, 1)], -1), -1)[:, :-1]


class _Greedy64:
    def greedy(self, prompt, new, consumed):
        """(`new` greedy tokens, hidden rows of the prompt and the first `consumed` of them): guesses are checked all at once."""
        tokens = list(int(t) for t in prompt)
        for _ in range(new):
            tokens.append(self.guess(tokens[-1]))
        while True:
            hidden = self.hidden(np.array(tokens[:-1] if new else tokens))
            best = self.logits(hidden[len(prompt) - 1:]).argmax(-1).tolist()
            wrong = next((i for i in range(new) if tokens[len(prompt) + i] != best[i]), None)
            if wrong is None:
                break
            tokens = tokens[:len(prompt) + wrong] + [best[wrong]]
            while len(tokens) < len(prompt) + new:
                tokens.append(self.guess(tokens[-1]))
        if consumed == new:
            hidden = self.hidden(np.array(tokens))
        return np.array(tokens[len(prompt):]), hidden


class _Llama64(_Greedy64):
    def __init__(self, case, seed):
        self.case, self.seed, self.m = case, seed, MODELS[case["model"]]
        self.vocab, self.next = self.m[6], _successors(seed, self.m[6]).tolist()

    def guess(self, token):
        return self.next[token]

    def hidden(self, tokens):
        m, eps = self.m, 1e-5
        x = _embedding(self.case, self.seed)[torch.from_numpy(np.asarray(tokens).astype(np.int64)).cuda()].double()
        n, share = x.shape[0], m[1] // m[2]
        freqs = torch.tensor([m[7] ** (-2.0 * j / m[4]) for j in range(m[4] // 2)], dtype=torch.float64, device="cuda")
        for l in range(self.case["layers"]):
            times = lambda h, name: h @ _unpack(self.case["format"], _linear(self.case, self.seed, l, name), _shapes(m)[name][1]).t().contiguous()  # noqa: E731
            h = _rms64(x, eps) * _norm(self.seed, 1024 + l, m[3]).double()
            q, k = _turned(times(h, "wq").view(n, m[1], m[4]), freqs), _turned(times(h, "wk").view(n, m[2], m[4]), freqs)
            v = times(h, "wv").view(n, m[2], m[4])
            out = [_weighted(q[:, a] @ k[:, a // share].t().contiguous() * m[4] ** -0.5) @ v[:, a // share].contiguous() for a in range(m[1])]
            x = x + times(torch.stack(out, 1).reshape(n, -1), "wo")
            h = _rms64(x, eps) * _norm(self.seed, 2048 + l, m[3]).double()
            x = x + times(torch.nn.functional.silu(times(h, "w1")) * times(h, "w3"), "w2")
        return x

    def logits(self, hidden):
        h = _rms64(hidden, 1e-5) * _norm(self.seed, 2, self.m[3]).double()
        raw = _head(self.case, self.seed)
        parts = [h @ _unpack(self.case["format"], p, self.m[3]).t().contiguous() for p in raw.split(16384)]
        return torch.cat(parts, -1)


class _Layered64(_Greedy64):
    def __init__(self, case, seed):
        self.config = _config(case)
        self.vocab, self.eps = self.config["vocab"], self.config["norm"]["eps"]
        self.own_head = self.config["architecture"] == "Ranavik"
        self.w = dict(_layered_weights(self.config, seed))
        self.next = _successors(seed, self.vocab).tolist()

    def guess(self, token):
        return self.next[token] if self.own_head else token

    def times(self, h, name):
        return h @ self.w[name].double().t().contiguous()

    def norm(self, x, name):
        return _rms64(x, self.eps) * self.w[name].double()

    def frequencies(self, rot):
        dims, s = rot["dims"], rot.get("scaling")
        f = torch.tensor([rot["base"] ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=torch.float64, device="cuda")
        if s is None:
            return f, 1.0
        if "original" not in s:
            return f / s["factor"], 1.0
        pair = lambda turns: dims * math.log(s["original"] / (2 * math.pi * turns)) / (2 * math.log(rot["base"]))  # noqa: E731
        low, high = max(math.floor(pair(s["fast"])), 0), min(math.ceil(pair(s["slow"])), dims - 1)
        slow = ((torch.arange(dims // 2, dtype=torch.float64, device="cuda") - low) / max(high - low, 0.001)).clamp(0, 1)
        return f / s["factor"] * slow + f * (1 - slow), 0.1 * math.log(s["factor"]) + 1

    def retention(self, h, m, p):
        n, heads = h.shape[0], m["heads"]
        f, factor = self.frequencies(m["rot"])
        q = _turned(self.times(h, p + "q").view(n, heads, -1), f, factor)
        k = _turned(self.times(h, p + "k").view(n, heads, -1), f, factor) * m["dim"] ** -0.5
        v = self.times(h, p + "v").view(n, heads, -1)
        at = torch.arange(n, device="cuda", dtype=torch.float64)
        far = at[:, None] - at[None, :]
        out = []
        for a in range(heads):
            keep = torch.where(far >= 0, m["decay"][a] ** far.clamp_min(0), torch.zeros_like(far))
            out.append((q[:, a] @ k[:, a].t().contiguous() * keep) @ v[:, a].contiguous())
        o = _rms64(torch.stack(out, 1), self.eps).reshape(n, -1) * torch.nn.functional.silu(self.times(h, p + "g"))
        return self.times(o, p + "o")

    def latent(self, h, m, p, cached):
        n, heads, dim = h.shape[0], m["heads"], m["dim"]
        f, factor = self.frequencies(m["rot"])
        q = self.times(h, p + "q").view(n, heads, -1)
        c, key_rot = cached
        k, v = self.times(c, p + "uk").view(n, heads, dim), self.times(c, p + "uv").view(n, heads, -1)
        turned = _turned(q[..., dim:].contiguous(), f, factor, interleaved=True)
        gate, out = torch.sigmoid(self.times(h, p + "g")), []
        for a in range(heads):
            scores = (q[:, a, :dim] @ k[:, a].t().contiguous() + turned[:, a] @ key_rot.t().contiguous()) * m["scale"]
            out.append(_weighted(scores, m["mask"]["size"], self.w[p + "sink"][a].double()) @ v[:, a].contiguous() * gate[:, a:a + 1])
        return self.times(torch.cat(out, -1), p + "o")

    def latents(self, h, m, p):
        f, factor = self.frequencies(m["rot"])
        both = self.times(h, p + "dkv")
        return self.norm(both[:, :m["kv_rank"]], p + "dkv.norm"), _turned(both[:, None, m["kv_rank"]:].contiguous(), f, factor, interleaved=True)[:, 0]

    def attention(self, h, m, p, cached):
        n, heads, share = h.shape[0], m["heads"], m["heads"] // m["kv_heads"]
        f, factor = self.frequencies(m["rot"])
        q = _turned(self.norm(self.times(h, p + "q"), p + "q.norm").view(n, heads, -1), f, factor)
        k, v = cached
        out = [_weighted(q[:, a] @ k[:, a // share].t().contiguous() * m["scale"], m["mask"]["size"]) @ v[:, a // share].contiguous() for a in range(heads)]
        return self.times(torch.cat(out, -1), p + "o")

    def keys(self, h, m, p):
        n, (f, factor) = h.shape[0], self.frequencies(m["rot"])
        k = self.norm(self.times(h, p + "k"), p + "k.norm").view(n, m["kv_heads"], -1)
        return _turned(k, f, factor), self.times(h, p + "v").view(n, m["kv_heads"], -1)

    def mamba2(self, h, m, p):
        n, heads, groups, state, taps = h.shape[0], m["heads"], m["groups"], m["state"], m["conv"]
        inner = heads * m["vdim"]
        z, xbc, dt = self.times(h, p + "in").split([inner, inner + 2 * groups * state, heads], -1)
        padded = torch.cat([xbc.new_zeros(taps - 1, xbc.shape[1]), xbc])
        conv = self.w[p + "conv"].double()
        xbc = torch.nn.functional.silu(sum(padded[t:t + n] * conv[:, t] for t in range(taps)) + self.w[p + "conv.b"].double())
        x, b, c = xbc.split([inner, groups * state, groups * state], -1)
        x, b, c = x.view(n, heads, -1), b.reshape(n, groups, state), c.reshape(n, groups, state)
        dt = torch.nn.functional.softplus(dt + self.w[p + "dt_bias"].double(), threshold=60)
        log = -(dt * self.w[p + "A_log"].double().exp()).cumsum(0)
        seen, out = torch.ones(n, n, dtype=torch.bool, device="cuda").tril(), []
        for a in range(heads):
            g = a * groups // heads
            keep = torch.exp((log[:, a:a + 1] - log[:, a][None, :]).masked_fill(~seen, -math.inf))
            out.append((c[:, g] @ b[:, g].t().contiguous() * keep * dt[:, a][None, :]) @ x[:, a].contiguous() + self.w[p + "D"][a].double() * x[:, a])
        y = torch.stack(out, 1).reshape(n, inner) * torch.nn.functional.silu(z)
        y = _rms64(y.view(n, m["norm_groups"], -1), self.eps).view(n, inner) * self.w[p + "norm"].double()
        return self.times(y, p + "o")

    def hidden(self, tokens):
        x = self.w["embed"][torch.from_numpy(np.asarray(tokens).astype(np.int64)).cuda()].double()
        if self.own_head:
            x = self.norm(x, "embed.norm")
        cached = {}
        for i, layer in enumerate(self.config["layers"]):
            p, m, kind = "l%d." % i, layer["mixer"], layer["type"]
            h = self.norm(x, p + "norm1") if self.own_head else x
            if kind in ("latent_attention", "attention"):
                source = m.get("kv_from", i)
                if source == i:
                    cached[i] = (self.latents if kind == "latent_attention" else self.keys)(h, m, p + "mix.")
                branch = (self.latent if kind == "latent_attention" else self.attention)(h, m, p + "mix.", cached[source])
            else:
                branch = (self.retention if kind == "retention" else self.mamba2)(h, m, p + "mix.")
            if self.own_head:   # branches in parallel
                if layer["mlp"]:
                    h = self.norm(x, p + "norm2")
                    branch = branch + self.times(torch.nn.functional.silu(self.times(h, p + "mlp.gate")) * self.times(h, p + "mlp.up"), p + "mlp.down")
                x = x + self.config["residual_mult"] * branch
            else:               # one after the other, each normed as it joins
                x = x + self.norm(branch, p + "norm1")
                if layer["mlp"]:
                    act = torch.nn.functional.gelu(self.times(x, p + "mlp.gate"), approximate="tanh")
                    x = x + self.norm(self.times(act * self.times(x, p + "mlp.up"), p + "mlp.down"), p + "norm2")
        return x

    def logits(self, hidden):
        z = self.times(self.norm(hidden, "final.norm"), "head" if self.own_head else "embed")
        cap = self.config.get("logit_softcap")
        return cap * torch.tanh(z / cap) if cap else z
