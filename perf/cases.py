"""The work that a program built on this engine has it do, as measurable cases.

Five kinds, each through a public entry point of the package:

- "layer": a transformer layer's projections as the engine's matmul callers
  issue them: qkv with its RMSNorm fused, wo added to the residual, gate | up
  with its norm, w2 added to the residual. One row is a decode step, a few a
  decode batch or a short prompt, hundreds a prefill.
- "square": C = A x B on fp32 matrices, sizes as they come.
- "attention": causal attention over a KV cache, one row (decode) or a whole
  prompt's rows (prefill).
- "quantize": fp32 weights to int8 bytes and column scales, when a model is
  loaded.
- "model": a whole em_model_forward call, tokens in and logits out.

Weights are N(0, 0.02), quantised for int8; activations are N(0, 1).
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

EPS = 1e-5  # RMSNorm


def _engine():
    name = "llm_engine_amd"
    if name not in sys.modules:
        path = os.path.join(os.getcwd(), "llm-engine_amd", "__init__.py")
        spec = importlib.util.spec_from_file_location(name, path)
        sys.modules[name] = mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
    return sys.modules[name]


# ---- the cases ---------------------------------------------------------------

def _layer(dtype, m, dim=4096, kv=4096, hidden=11008, registered=True):
    return {"kind": "layer", "dtype": dtype, "m": m, "dim": dim, "kv": kv, "hidden": hidden,
            "registered": registered and dtype == "q8"}


def _attention(rows, ctx, heads=32, kv_heads=32, head_size=128):
    """`rows` query rows, the last of them at position ctx - 1."""
    return {"kind": "attention", "rows": rows, "ctx": ctx, "heads": heads, "kv_heads": kv_heads,
            "head_size": head_size}


def _model(dtype, feed, ctx, dim, hidden, layers, heads, kv_heads, vocab):
    """`feed` tokens fed after `ctx` cached positions."""
    return {"kind": "model", "dtype": dtype, "feed": feed, "ctx": ctx, "dim": dim,
            "hidden": hidden, "layers": layers, "heads": heads, "kv_heads": kv_heads,
            "vocab": vocab}


def listed():
    return [
        # One decode step's products of a Llama-7B-shaped layer, int8 weights:
        # what serving one stream spends its time on.
        dict(_layer("q8", 1), name="decode_q8"),
        # The same for a batch of streams, or a short prompt: between the
        # memory-bound and the compute-bound end.
        dict(_layer("q8", 40), name="batch_q8"),
        # A 512-token prompt through that layer: time to the first token.
        dict(_layer("q8", 512), name="prefill_q8"),
        # A long prompt, of a length that is no tile's multiple, with grouped
        # kv heads: the largest products.
        dict(_layer("q8", 1900, kv=1024), name="long_prefill_q8"),
        # fp32 weights, one decode step: the unquantised model.
        dict(_layer("f32", 1), name="decode_f32"),
        # fp32 weights, a ragged prompt of ordinary length.
        dict(_layer("f32", 300), name="prefill_f32"),
        # The square product of the engine's matmul benchmark.
        {"name": "square_f32", "kind": "square", "m": 2048, "k": 2048, "n": 2048},
        # Decode attention with grouped kv heads far into a context.
        dict(_attention(1, 16384, kv_heads=8), name="decode_attention"),
        # A prompt's attention, every head with its own keys and values.
        dict(_attention(1000, 1000), name="prefill_attention"),
        # Quantising one projection at load time.
        {"name": "quantize", "kind": "quantize", "rows": 4096, "cols": 11008},
        # stories15M, one decode step: launches and latency, the smallest call.
        dict(_model("q8", 1, 120, 288, 768, 6, 6, 6, 32000), name="model_decode_small"),
        # One Llama-7B-shaped layer and a classifier, a 200-token prompt.
        dict(_model("q8", 200, 0, 4096, 11008, 1, 32, 8, 8000), name="model_prefill"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer"] * 4 + ["square"] * 2 + ["attention"] * 2 + ["quantize", "model"])
    if kind == "layer":
        head = rng.choice([32, 48, 64, 128])
        heads = max(2, _log(rng, 256, 5120) // head)
        dim = heads * head
        kv = dim if rng.random() < 0.5 or heads % 4 else dim // 4
        hidden = 16 * _log(rng, 2.3 * dim / 16, 3.7 * dim / 16)
        m = 1 if rng.random() < 0.15 else _log(rng, 1, 2048)
        dtype = "q8" if rng.random() < 0.6 else "f32"
        # No more work than the listed long prompt's (fp32: a third of it).
        weights = dim * (2 * dim + 2 * kv + 3 * hidden)
        m = min(m, int((3.3e11 if dtype == "q8" else 1.1e11) / weights))
        return _layer(dtype, m, dim, kv, hidden, rng.random() < 0.8)
    if kind == "square":
        n = _log(rng, 200, 4096)
        near = [max(64, int(n * rng.uniform(0.6, 1.2))) for _ in range(3)]
        m, k, n = (x if rng.random() < 0.4 else -(-x // 32) * 32 for x in near)
        return {"kind": "square", "m": m, "k": k, "n": n}
    if kind == "attention":
        head = rng.choice([48, 64, 128])
        kv_heads = rng.choice([4, 6, 8, 16, 32])
        heads = kv_heads * rng.choice([1, 4] if kv_heads <= 8 else [1])
        if rng.random() < 0.5:
            return _attention(_log(rng, 1, 8), _log(rng, 32, 16384), heads, kv_heads, head)
        rows = _log(rng, 16, 1024)
        return _attention(rows, rows + (0 if rng.random() < 0.6 else _log(rng, 16, 1024)), heads,
                          kv_heads, head)
    if kind == "quantize":
        return {"kind": "quantize", "rows": _log(rng, 256, 11008), "cols": _log(rng, 256, 11008)}
    head = rng.choice([32, 48, 64])
    heads = rng.choice([4, 6, 8, 16])
    feed = 1 if rng.random() < 0.5 else _log(rng, 2, 250)
    return _model(rng.choice(["q8", "f32"]), feed, rng.randrange(0, 200), heads * head,
                  16 * _log(rng, heads * head / 7, heads * head / 4), rng.randrange(2, 7), heads,
                  heads if rng.random() < 0.6 else heads // 2, _log(rng, 1000, 32000))


# ---- inputs ------------------------------------------------------------------

def _normal(seed):
    """normal(*shape, std): successive draws of one seeded stream on the GPU."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(*shape, std=1.0):
        return torch.randn(shape, generator=g, device="cuda") * std
    return normal


def _quantise(w):
    """Column absmax / 127, rounded half away from zero: int8 bytes and scales."""
    top = w.abs().amax(dim=0)
    scale = top / torch.full_like(top, 127.0)  # tensor by tensor: an IEEE division
    inv = torch.where(scale > 0, torch.ones_like(scale) / scale, torch.zeros_like(scale))
    x = (w * inv).double()
    return (torch.sign(x) * torch.floor(x.abs() + 0.5)).clamp(-127, 127).to(torch.int8), scale


def _projections(c):
    """name -> (k, n) of a layer's four products."""
    d, h = c["dim"], c["hidden"]
    return {"qkv": (d, d + 2 * c["kv"]), "wo": (d, d), "w13": (d, 2 * h), "w2": (h, d)}


def _layer_inputs(c, seed):
    normal = _normal(seed)
    s = {"x": normal(c["m"], c["dim"]), "attended": normal(c["m"], c["dim"]),
         "act": normal(c["m"], c["hidden"]),
         "rms_att": 1.0 + normal(c["dim"], std=0.1), "rms_ffn": 1.0 + normal(c["dim"], std=0.1)}
    for name, (k, n) in _projections(c).items():
        w = normal(k, n, std=0.02)
        s[name], s[name + "_scale"] = _quantise(w) if c["dtype"] == "q8" else (w, None)
    return s


def _attention_inputs(c, seed):
    normal = _normal(seed)
    kv = c["kv_heads"] * c["head_size"]
    return {"q": normal(c["rows"], c["heads"] * c["head_size"] + 2 * kv),
            "keys": normal(c["ctx"], kv), "values": normal(c["ctx"], kv)}


def _model_inputs(c, seed):
    normal = _normal(seed)
    d, h, v = c["dim"], c["hidden"], c["vocab"]
    kv = c["kv_heads"] * (d // c["heads"])
    gain = lambda: 1.0 + normal(d, std=0.1)  # noqa: E731
    weights = {"token_embedding": normal(v, d), "rms_final": gain(), "wcls": normal(d, v, std=0.02),
               "layers": [{"rms_att": gain(), "wqkv": normal(d, d + 2 * kv, std=0.02),
                           "wo": normal(d, d, std=0.02), "rms_ffn": gain(),
                           "w13": normal(d, 2 * h, std=0.02), "w2": normal(h, d, std=0.02)}
                          for _ in range(c["layers"])]}
    tokens = np.random.RandomState(seed % (1 << 31)).randint(0, v, c["ctx"] + c["feed"])
    return weights, tokens.astype(np.int32)


def _model_config(c):
    return {"dim": c["dim"], "hidden_dim": c["hidden"], "n_layers": c["layers"],
            "n_heads": c["heads"], "n_kv_heads": c["kv_heads"], "vocab_size": c["vocab"],
            "seq_len": max(256, c["ctx"] + c["feed"])}


def _to_host(weights):
    if isinstance(weights, dict):
        return {k: _to_host(v) for k, v in weights.items()}
    if isinstance(weights, list):
        return [_to_host(v) for v in weights]
    return weights.cpu().numpy()


def prepare(case, seed):
    em = _engine()
    c, s = case, {"case": dict(case)}
    if c["kind"] == "layer":
        s.update(_layer_inputs(c, seed))
        for name, (k, n) in _projections(c).items():
            if c["registered"]:
                em.register_q8(s[name])
            s["c_" + name] = torch.empty((c["m"], n), device="cuda")
    elif c["kind"] == "square":
        normal = _normal(seed)
        s.update(a=normal(c["m"], c["k"]), b=normal(c["k"], c["n"]),
                 c=torch.empty((c["m"], c["n"]), device="cuda"))
    elif c["kind"] == "attention":
        s.update(_attention_inputs(c, seed))
        s["shape"] = em.attention_shape(c["heads"], c["kv_heads"], c["head_size"], c["ctx"])
        s["pos"] = torch.tensor([c["ctx"] - c["rows"]], dtype=torch.int32, device="cuda")
        s["out"] = torch.empty((c["rows"], c["heads"] * c["head_size"]), device="cuda")
        floats = em.attention_scratch_floats(s["shape"], c["rows"])
        s["scratch"] = torch.empty((max(1, floats),), device="cuda")
    elif c["kind"] == "quantize":
        s["w"] = _normal(seed)(c["rows"], c["cols"], std=0.02)
    else:
        weights, tokens = _model_inputs(c, seed)
        s["model"] = em.Model(_model_config(c), _to_host(weights), q8=c["dtype"] == "q8")
        s["tokens"] = tokens[c["ctx"]:]
        if c["ctx"]:
            s["model"].forward(tokens[:c["ctx"]], 0)
    return s


def run(s):
    em, c = _engine(), s["case"]
    if c["kind"] == "layer":
        em.matmul(s["x"], s["qkv"], s["c_qkv"], scale=s["qkv_scale"], rms_weight=s["rms_att"])
        s["c_wo"].copy_(s["x"])  # the residual that wo and w2 add to
        em.matmul(s["attended"], s["wo"], s["c_wo"], scale=s["wo_scale"], accumulate=True)
        em.matmul(s["x"], s["w13"], s["c_w13"], scale=s["w13_scale"], rms_weight=s["rms_ffn"])
        s["c_w2"].copy_(s["x"])
        em.matmul(s["act"], s["w2"], s["c_w2"], scale=s["w2_scale"], accumulate=True)
        return [s["c_qkv"], s["c_wo"], s["c_w13"], s["c_w2"]]
    if c["kind"] == "square":
        return em.matmul(s["a"], s["b"], s["c"])
    if c["kind"] == "attention":
        return em.attention(s["shape"], c["rows"], s["pos"], s["q"], s["keys"], s["values"],
                            s["out"], s["scratch"])
    if c["kind"] == "quantize":
        return em.quantize_q8(s["w"])
    return s["model"].forward(s["tokens"], c["ctx"])


# ---- what a pass cannot do without ---------------------------------------------

def work(case):
    c = case
    size = 1 if c.get("dtype") == "q8" else 4
    if c["kind"] == "layer":
        m, d, h = c["m"], c["dim"], c["hidden"]
        kn = sum(k * n for k, n in _projections(c).values())
        columns = sum(n for _, n in _projections(c).values())
        scales = columns * 4 if size == 1 else 0
        # x (the two norms' input and the residual), the attended rows and the activations in.
        rows = m * (2 * d + h + columns) * 4
        return {"bytes": kn * size + scales + 2 * d * 4 + rows, "flops": 2 * m * kn}
    if c["kind"] == "square":
        m, k, n = c["m"], c["k"], c["n"]
        return {"bytes": 4 * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    if c["kind"] == "attention":
        rows, ctx, dim = c["rows"], c["ctx"], c["heads"] * c["head_size"]
        pairs = rows * (ctx - rows) + rows * (rows + 1) // 2
        kv = 2 * ctx * c["kv_heads"] * c["head_size"]
        return {"bytes": 4 * (kv + 2 * rows * dim), "flops": 4 * pairs * dim}
    if c["kind"] == "quantize":
        n = c["rows"] * c["cols"]
        return {"bytes": 5 * n + 4 * c["cols"], "flops": 2 * n}
    d, h, v, feed, ctx = c["dim"], c["hidden"], c["vocab"], c["feed"], c["ctx"]
    kv = c["kv_heads"] * (d // c["heads"])
    layer = d * (d + 2 * kv) + d * d + 3 * d * h
    columns = d + 2 * kv + d + 2 * h + d
    scales = 4 * (c["layers"] * columns + v) if size == 1 else 0
    pairs = feed * ctx + feed * (feed + 1) // 2
    return {"bytes": size * (c["layers"] * layer + d * v) + scales + 4 * v + 4 * feed * d
            + 4 * c["layers"] * 2 * kv * (ctx + feed),
            "flops": c["layers"] * (2 * feed * layer + 4 * pairs * d) + 2 * d * v}


def tolerance(case):
    # About four times what 32-bit sums in another order are off: against 64
    # bits fp32 products measured up to 1.1e-6 at k = 4096 (2e-6 at the
    # deepest), int8 ones and attention 2e-7 to 4.5e-7. A model's logits gather
    # every layer's rounding.
    if case["kind"] == "quantize":
        return "exact"
    if case["kind"] == "model":
        return {"rel": 1e-5, "max": 1e-4}
    if case["kind"] == "square" or case.get("dtype") == "f32":
        return {"rel": 8e-6, "max": 8e-5}
    return {"rel": 2e-6, "max": 2e-5}


# ---- the same in 64 bits -----------------------------------------------------------

def _norm64(x, w):
    x = x.double()
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + EPS) * w.double()


def _attend64(q, keys, values, heads, kv_heads, head_size, pos):
    """q [rows, heads * head_size]; row i sits at pos + i."""
    rows, ctx = q.shape[0], keys.shape[0]
    out = torch.empty((rows, heads * head_size), dtype=torch.float64, device=q.device)
    at = torch.arange(ctx, device=q.device)[None, :]
    hidden = at > (pos + torch.arange(rows, device=q.device))[:, None]
    for h in range(heads):
        g = h // (heads // kv_heads)
        mine, theirs = slice(h * head_size, (h + 1) * head_size), slice(g * head_size,
                                                                      (g + 1) * head_size)
        s = q[:, mine].double() @ keys[:, theirs].double().T.contiguous() / math.sqrt(head_size)
        p = torch.softmax(s.masked_fill(hidden, -math.inf), dim=-1)
        out[:, mine] = p @ values[:, theirs].double().contiguous()
    return out


def _weight64(w, dtype):
    if dtype != "q8":
        return w.double()
    q, scale = _quantise(w)
    return q.double() * scale.double()


def _rope64(x, heads, head_size, start):
    rows, half = x.shape[0], head_size // 2
    freq = 10000.0 ** (-2.0 * torch.arange(half, dtype=torch.float64, device=x.device) / head_size)
    angle = (start + torch.arange(rows, dtype=torch.float64, device=x.device))[:, None] * freq
    x = x.reshape(rows, heads, half, 2)
    cos, sin = angle.cos()[:, None, :], angle.sin()[:, None, :]
    a, b = x[..., 0], x[..., 1]
    return torch.stack((a * cos - b * sin, a * sin + b * cos), dim=-1).reshape(rows, -1)


def _model64(c, seed):
    weights, tokens = _model_inputs(c, seed)
    d, h, heads, kv_heads = c["dim"], c["hidden"], c["heads"], c["kv_heads"]
    hs = d // heads
    kv = kv_heads * hs
    x = weights["token_embedding"][torch.from_numpy(tokens).long().cuda()].double()
    for w in weights["layers"]:
        qkv = _norm64(x, w["rms_att"]) @ _weight64(w["wqkv"], c["dtype"])
        q = _rope64(qkv[:, :d], heads, hs, 0)
        k = _rope64(qkv[:, d:d + kv], kv_heads, hs, 0)
        att = _attend64(q, k, qkv[:, d + kv:].contiguous(), heads, kv_heads, hs, 0)
        x = x + att @ _weight64(w["wo"], c["dtype"])
        gate_up = _norm64(x, w["rms_ffn"]) @ _weight64(w["w13"], c["dtype"])
        act = torch.nn.functional.silu(gate_up[:, :h]) * gate_up[:, h:]
        x = x + act @ _weight64(w["w2"], c["dtype"])
    last = _norm64(x[-1:], weights["rms_final"])
    return (last @ _weight64(weights["wcls"], c["dtype"]))[0]


def exact(case, seed):
    c = case
    if c["kind"] == "layer":
        s = _layer_inputs(c, seed)

        def product(a, name):
            w = s[name].double()
            return a @ (w if s[name + "_scale"] is None else w * s[name + "_scale"].double())

        x = s["x"].double()
        return [product(_norm64(x, s["rms_att"]), "qkv"),
                x + product(s["attended"].double(), "wo"),
                product(_norm64(x, s["rms_ffn"]), "w13"),
                x + product(s["act"].double(), "w2")]
    if c["kind"] == "square":
        normal = _normal(seed)
        a, b = normal(c["m"], c["k"]), normal(c["k"], c["n"])
        return a.double() @ b.double()
    if c["kind"] == "attention":
        s = _attention_inputs(c, seed)
        dim = c["heads"] * c["head_size"]
        return _attend64(s["q"][:, :dim], s["keys"], s["values"], c["heads"], c["kv_heads"],
                         c["head_size"], c["ctx"] - c["rows"])
    if c["kind"] == "quantize":
        return list(_quantise(_normal(seed)(c["rows"], c["cols"], std=0.02)))
    return _model64(c, seed)
