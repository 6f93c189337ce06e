"""The workloads whose speed is measured, through the package's public entry points.

Kinds of case (the ranges that ``draw`` covers):

``linear``    ``PolarQuantLinearMethod.apply``, called eagerly inside
              ``torch.inference_mode`` as vLLM calls a quantization method:
              1..8192 rows, 2..6 bits, fp16 / bf16, with and without a bias,
              input sizes that are no multiple of 128 and output sizes that are
              no multiple of 16.
``layers``    the quantized linears of a stack of decoder layers (merged
              qkv Q5, o Q6, merged gate/up Q3, down Q4), captured once in a HIP
              graph and replayed, as a serving program runs its decode step;
              1..64 rows.
``decode``    a whole decode step of ``DecodeRunner`` (embedding, norms,
              rotary, cache write, attention, linears, lm_head) replayed from
              a HIP graph; batch 1..16, context up to 4096. Few layers, so
              that bf16 roundings do not grow over many.
``moe``       ``PolarQuantMoEMethod.apply``: routing and SwiGLU experts;
              1..4096 tokens.
``kv``        ``PolarKVCache``: a prompt is taken in and some tokens are
              decoded; each update compresses what leaves the bf16 window and
              returns the whole history.
``quantize``  ``PolarQuantizer.quantize_tensor`` of a weight on the GPU.

Weights are codes and norms as the quantizer makes them from normal weights:
a code is the Lloyd-Max cell of an N(0, 1) value, a norm that of 128 values.
"""

import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "polarengine-vllm_amd"))

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
# bits of a decoder layer's linears (the mixed assignment of the C4 layer)
LAYER_BITS = {"qkv_proj": 5, "o_proj": 6, "gate_up_proj": 3, "down_proj": 4}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one token through an MLP up projection: the smallest ordinary call
        {"name": "linear_m1", "kind": "linear", "m": 1, "n": 12288, "k": 4096, "bits": 4,
         "dtype": "fp16", "bias": False},
        # a few tokens through a small projection of odd sizes, with a bias
        {"name": "linear_m7_ragged", "kind": "linear", "m": 7, "n": 1500, "k": 4000, "bits": 5,
         "dtype": "bf16", "bias": True},
        # a short prompt of odd length through a down projection
        {"name": "linear_m300", "kind": "linear", "m": 300, "n": 4096, "k": 12288, "bits": 3,
         "dtype": "bf16", "bias": False},
        # a prompt of 2048 tokens through an up projection
        {"name": "linear_m2048", "kind": "linear", "m": 2048, "n": 12288, "k": 4096, "bits": 4,
         "dtype": "fp16", "bias": False},
        # a large prefill batch through a down projection
        {"name": "linear_m8192", "kind": "linear", "m": 8192, "n": 4096, "k": 12288, "bits": 3,
         "dtype": "fp16", "bias": False},
        # the linears of eight decoder layers for one token
        {"name": "layers_m1", "kind": "layers", "m": 1, "layers": 8, "hidden": 4096, "qkv": 6144,
         "inter": 12288, "dtype": "bf16"},
        # a decode step of one sequence, and of a batch of sixteen
        {"name": "decode_b1", "kind": "decode", "batch": 1, "context": 1024, "layers": 3,
         "hidden": 4096, "heads": 32, "kv_heads": 8, "head_dim": 128, "inter": 12288,
         "vocab": 151936},
        {"name": "decode_b16", "kind": "decode", "batch": 16, "context": 1024, "layers": 3,
         "hidden": 4096, "heads": 32, "kv_heads": 8, "head_dim": 128, "inter": 12288,
         "vocab": 151936},
        # the experts of one layer for a decode batch, and for a prompt
        {"name": "moe_t128", "kind": "moe", "t": 128, "e": 64, "top_k": 8, "h": 2048, "i": 1408,
         "bits13": 3, "bits2": 4, "scoring": "softmax", "dtype": "fp16"},
        {"name": "moe_t2048", "kind": "moe", "t": 2048, "e": 64, "top_k": 8, "h": 2048, "i": 1408,
         "bits13": 3, "bits2": 4, "scoring": "softmax", "dtype": "bf16"},
        # one layer's K/V cache: a prompt of 8000 tokens for each of four
        # sequences, then four decoded tokens
        {"name": "kv_s8000", "kind": "kv", "batch": 4, "heads": 8, "head_dim": 128, "tokens": 8000,
         "steps": 4, "nbits": 3, "residual": 128, "keep": False},
        # quantizing an MLP projection
        {"name": "quantize_q5", "kind": "quantize", "n": 12288, "k": 4096, "bits": 5,
         "dtype": "fp16", "pack": False},
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear"] * 5 + ["layers", "decode", "decode", "moe", "moe", "moe", "kv", "kv",
                                        "quantize"])
    if kind == "linear":
        while True:
            c = {"kind": kind, "m": _log(rng, 1, 8192),
                 "n": rng.choice([_log(rng, 256, 24576), 16 * _log(rng, 64, 1536)]),
                 "k": rng.choice([_log(rng, 512, 12288), 128 * rng.randint(8, 96)]),
                 "bits": rng.choice([2, 3, 4, 5, 6]), "dtype": rng.choice(["fp16", "bf16"]),
                 "bias": rng.random() < 0.3}
            if c["m"] * c["n"] * c["k"] <= 8192 * 4096 * 12288:
                return c
    if kind == "layers":
        hidden = rng.choice([2048, 4096])
        return {"kind": kind, "m": _log(rng, 1, 64), "layers": rng.randint(2, 8), "hidden": hidden,
                "qkv": hidden * 3 // 2, "inter": rng.choice([2, 3]) * hidden,
                "dtype": rng.choice(["fp16", "bf16"])}
    if kind == "decode":
        d = rng.choice([64, 128])
        kvh = rng.choice([2, 4, 8])
        heads = kvh * rng.choice([1, 2, 4])
        batch = _log(rng, 1, 16)
        return {"kind": kind, "batch": batch, "context": _log(rng, 16, min(4096, 16384 // batch)),
                "layers": rng.randint(1, 3), "hidden": rng.choice([1024, 2048, 4096]),
                "heads": heads, "kv_heads": kvh, "head_dim": d,
                "inter": 128 * rng.randint(16, 96), "vocab": _log(rng, 2000, 151936)}
    if kind == "moe":
        e = rng.choice([8, 16, 32, 64])
        return {"kind": kind, "t": _log(rng, 1, 4096), "e": e, "top_k": rng.choice([1, 2, 4, 6, 8]),
                "h": 128 * rng.randint(8, 20), "i": 128 * rng.randint(5, 12),
                "bits13": rng.choice([3, 4, 5]), "bits2": rng.choice([4, 5]),
                "scoring": rng.choice(["softmax", "sigmoid"]),
                "dtype": rng.choice(["fp16", "bf16"])}
    if kind == "kv":
        while True:
            c = {"kind": kind, "batch": rng.randint(1, 4), "heads": rng.choice([4, 8, 16]),
                 "head_dim": rng.choice([64, 128, 256]), "tokens": _log(rng, 64, 8000),
                 "steps": rng.randint(1, 8), "nbits": rng.choice([2, 3, 4]),
                 "residual": rng.choice([64, 128]), "keep": rng.random() < 0.25}
            rows = c["batch"] * c["heads"] * c["tokens"] * (c["steps"] + 1)
            if rows * c["head_dim"] <= 4 * 8 * 8000 * 5 * 128:
                return c
    while True:
        bits = rng.choice([2, 3, 4, 5, 6])
        c = {"kind": kind, "n": _log(rng, 256, 24576), "k": _log(rng, 512, 12288), "bits": bits,
             "dtype": rng.choice(["fp16", "bf16", "fp32"]),
             "pack": bits <= 4 and rng.random() < 0.5}
        if c["n"] * c["k"] <= 12288 * 4096:
            return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
_CENTROIDS = {}


def _lloyd_max(levels, open_ends):
    """Lloyd-Max levels of N(0, 1) after 100 iterations from an even split of
    [-4, 4]; ``open_ends``: the outer cells reach to infinity."""
    key = (levels, open_ends)
    if key not in _CENTROIDS:
        pdf = lambda v: math.exp(-v * v / 2) / math.sqrt(2 * math.pi)  # noqa: E731
        cdf = lambda v: 0.5 * math.erfc(-v / math.sqrt(2))  # noqa: E731
        end = math.inf if open_ends else 4.0
        inner = [-4.0 + 8.0 * i / levels for i in range(1, levels)]
        for _ in range(100):
            b = [-end] + inner + [end]
            cent = []
            for lo, hi in zip(b[:-1], b[1:]):
                p = cdf(hi) - cdf(lo)
                cent.append((pdf(lo) - pdf(hi)) / p if p > 1e-10 else (lo + hi) / 2)
            inner = [(u + v) / 2 for u, v in zip(cent[:-1], cent[1:])]
        _CENTROIDS[key] = cent
    return _CENTROIDS[key]


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _gen(seed):
    return torch.Generator(device=_device()).manual_seed(int(seed))


def _weight(g, rows, k, bits, std, lead=()):
    """int8 codes [*lead, rows, kp] and fp16 norms [*lead, rows, kp / 128]."""
    kp = (k + 127) // 128 * 128
    cent = _lloyd_max(1 << bits, True)
    mid = torch.tensor([(a + b) / 2 for a, b in zip(cent[:-1], cent[1:])], device=_device())
    codes = torch.empty(*lead, rows, kp, dtype=torch.int8, device=_device())
    flat = codes.view(-1, kp)
    for r in range(0, flat.shape[0], 16384):
        z = torch.randn(min(16384, flat.shape[0] - r), kp, generator=g, device=_device())
        flat[r:r + 16384] = torch.bucketize(z, mid).to(torch.int8)
    norms = std * math.sqrt(128) * (1 + torch.randn(*lead, rows, kp // 128, generator=g,
                                                    device=_device()) / 16)
    return codes, norms.half()


def _linear_inputs(c, seed):
    g = _gen(seed)
    codes, norms = _weight(g, c["n"], c["k"], c["bits"], 0.02)
    dt = DTYPES[c["dtype"]]
    x = torch.randn(c["m"], c["k"], generator=g, device=_device()).to(dt)
    bias = (0.1 * torch.randn(c["n"], generator=g, device=_device())).to(dt) if c["bias"] else None
    return codes, norms, x, bias


def _layer_shapes(c):
    """(name, rows, columns) of one decoder layer's merged linears."""
    q = c["qkv"] if "qkv" in c else (c["heads"] + 2 * c["kv_heads"]) * c["head_dim"]
    o = c["hidden"] if "qkv" in c else c["heads"] * c["head_dim"]
    return [("qkv_proj", q, c["hidden"]), ("o_proj", c["hidden"], o),
            ("gate_up_proj", 2 * c["inter"], c["hidden"]), ("down_proj", c["hidden"], c["inter"])]


def _layers_inputs(c, seed):
    """Per layer and linear: bits, codes, norms, x."""
    g = _gen(seed)
    out = []
    for _ in range(c["layers"]):
        for name, n, k in _layer_shapes(c):
            codes, norms = _weight(g, n, k, LAYER_BITS[name], 0.02)
            x = torch.randn(c["m"], k, generator=g, device=_device()).to(DTYPES[c["dtype"]])
            out.append((LAYER_BITS[name], codes, norms, x))
    return out


def _decode_inputs(c, seed):
    g, bf = _gen(seed), torch.bfloat16
    rand = lambda *s: torch.randn(*s, generator=g, device=_device())  # noqa: E731
    w = {"embed": (rand(c["vocab"], c["hidden"]) * 0.02).to(bf),
         "lm_head": (rand(c["vocab"], c["hidden"]) / math.sqrt(c["hidden"])).to(bf), "layers": []}
    for _ in range(c["layers"]):
        w["layers"].append({})
        for name, n, k in _layer_shapes(c):
            codes, norms = _weight(g, n, k, LAYER_BITS[name], 1 / math.sqrt(k))
            w["layers"][-1][name] = {"codes": codes, "norms": norms}
    tokens = torch.randint(0, c["vocab"], (c["batch"],), generator=g, device=_device())
    kv = (c["layers"], c["batch"], c["kv_heads"], c["context"], c["head_dim"])
    return w, tokens, rand(*kv).to(bf), rand(*kv).to(bf)


def _moe_inputs(c, seed):
    g = _gen(seed)
    w13 = _weight(g, 2 * c["i"], c["h"], c["bits13"], 0.02, (c["e"],))
    w2 = _weight(g, c["h"], c["i"], c["bits2"], 0.02, (c["e"],))
    x = torch.randn(c["t"], c["h"], generator=g, device=_device()).to(DTYPES[c["dtype"]])
    logits = torch.randn(c["t"], c["e"], generator=g, device=_device())
    return w13, w2, x, logits


def _kv_inputs(c, seed):
    """K and V of the prompt and of each decoded token, [B, H, S, D] bf16."""
    g = _gen(seed)
    sizes = [c["tokens"]] + [1] * c["steps"]
    return [[torch.randn(c["batch"], c["heads"], s, c["head_dim"], generator=g, device=_device())
             .to(torch.bfloat16) for _ in range(2)] for s in sizes]


def _quantize_inputs(c, seed):
    w = 0.02 * torch.randn(c["n"], c["k"], generator=_gen(seed), device=_device())
    return w.to(torch.float32 if c["dtype"] == "fp32" else DTYPES[c["dtype"]])


# ---------------------------------------------------------------------------
# what a program holds before the call
# ---------------------------------------------------------------------------
def _quant_linear(codes, norms, bits, k):
    from polarengine_vllm.linear_method import PolarQuantLinearMethod
    method, layer = PolarQuantLinearMethod(128, bits), torch.nn.Module()
    method.create_weights(layer, k, [codes.shape[0]], k, codes.shape[0], torch.float16)
    layer.to(codes.device)
    layer.codes.copy_(codes)
    layer.norms.copy_(norms)
    method.process_weights_after_loading(layer)
    return method, layer


def _capture(step):
    """``step`` captured in a HIP graph after two eager passes; (graph, outputs)."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(2):
            step()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            out = step()
    torch.cuda.current_stream().wait_stream(s)
    return graph, out


def prepare(case, seed):
    c = case
    with torch.inference_mode():
        if c["kind"] == "linear":
            codes, norms, x, bias = _linear_inputs(c, seed)
            method, layer = _quant_linear(codes, norms, c["bits"], c["k"])
            return {"kind": "linear", "method": method, "layer": layer, "x": x, "bias": bias}
        if c["kind"] == "layers":
            calls = []
            for bits, codes, norms, x in _layers_inputs(c, seed):
                method, layer = _quant_linear(codes, norms, bits, x.shape[1])
                calls.append((method, layer, x))
            graph, out = _capture(lambda: [m.apply(ly, x) for m, ly, x in calls])
            return {"kind": "layers", "graph": graph, "out": out, "calls": calls}
        if c["kind"] == "decode":
            from polarengine_vllm.decode_runner import DecodeRunner, DecoderConfig
            w, tokens, k, v = _decode_inputs(c, seed)
            cfg = DecoderConfig(hidden=c["hidden"], layers=c["layers"], heads=c["heads"],
                                kv_heads=c["kv_heads"], head_dim=c["head_dim"],
                                intermediate=c["inter"], vocab=c["vocab"], bits=dict(LAYER_BITS))
            runner = DecodeRunner(cfg, c["batch"], c["context"] + 64, _device(), weights=w)
            runner.k_cache[..., :c["context"]] = k.transpose(3, 4)
            runner.v_cache[..., :c["context"], :] = v
            pos = torch.tensor([c["context"]], device=_device())
            graph, out = _capture(lambda: runner.step(tokens, pos))
            return {"kind": "decode", "graph": graph, "runner": runner, "tokens": tokens, "pos": pos,
                    "out": {"logits": out, "k_cache": runner.k_cache, "v_cache": runner.v_cache}}
        if c["kind"] == "moe":
            from polarengine_vllm.moe_method import PolarQuantMoEMethod
            (c13, n13), (c2, n2), x, logits = _moe_inputs(c, seed)
            method, layer = PolarQuantMoEMethod(128, c["bits13"], c["bits2"]), torch.nn.Module()
            method.create_weights(layer, c["e"], c["h"], c["i"], x.dtype)
            layer.to(_device())
            for name, value in (("w13_codes", c13), ("w13_norms", n13), ("w2_codes", c2),
                                ("w2_norms", n2)):
                getattr(layer, name).copy_(value)
            method.process_weights_after_loading(layer)
            return {"kind": "moe", "method": method, "layer": layer, "x": x, "logits": logits,
                    "top_k": c["top_k"], "scoring": c["scoring"]}
        if c["kind"] == "kv":
            from polarengine_vllm.kv_cache import PolarKVCache, PolarKVConfig
            cfg = PolarKVConfig(nbits=c["nbits"], residual_length=c["residual"],
                                head_dim=c["head_dim"], num_kv_heads=c["heads"], num_layers=1)
            return {"kind": "kv", "cache": PolarKVCache(cfg, "cuda", keep_expanded=c["keep"]),
                    "kv": _kv_inputs(c, seed)}
        from polarengine_vllm.quantizer import PolarQuantizer
        return {"kind": "quantize", "quantizer": PolarQuantizer(128), "w": _quantize_inputs(c, seed),
                "bits": c["bits"], "pack": c["pack"]}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    s = state
    with torch.inference_mode():
        if s["kind"] == "linear":
            return s["method"].apply(s["layer"], s["x"], s["bias"])
        if s["kind"] in ("layers", "decode"):
            s["graph"].replay()
            return s["out"]
        if s["kind"] == "moe":
            return s["method"].apply(s["layer"], s["x"], s["logits"], s["top_k"], True,
                                     scoring_func=s["scoring"])
        if s["kind"] == "kv":
            cache = s["cache"]
            cache.reset()
            for k, v in s["kv"]:  # the prompt, then token by token
                full = cache.update(k, v, 0)
            codes = [ly.compressed() for ly in (cache.k_layers[0], cache.v_layers[0])]
            return {"full": full, "codes": codes}
        return s["quantizer"].quantize_tensor(s["w"], s["bits"], pack=s["pack"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _linear_work(m, n, k, bits):
    return {"bytes": n * k * bits / 8 + n * (k / 128) * 2 + 2 * m * (k + n), "flops": 2.0 * m * n * k}


def work(case):
    c = case
    if c["kind"] == "linear":
        return _linear_work(c["m"], c["n"], c["k"], c["bits"])
    if c["kind"] in ("layers", "decode"):
        m = c["m"] if c["kind"] == "layers" else c["batch"]
        w = {"bytes": 0.0, "flops": 0.0}
        for name, n, k in _layer_shapes(c):
            one = _linear_work(m, n, k, LAYER_BITS[name])
            w = {f: w[f] + c["layers"] * one[f] for f in w}
        if c["kind"] == "decode":
            seen = c["context"] + 1
            w["bytes"] += 2 * c["vocab"] * c["hidden"] + 4 * m * c["vocab"]
            w["bytes"] += c["layers"] * m * c["kv_heads"] * seen * c["head_dim"] * 4
            w["flops"] += 2.0 * m * c["vocab"] * c["hidden"]
            w["flops"] += c["layers"] * m * c["heads"] * seen * c["head_dim"] * 4.0
        return w
    if c["kind"] == "moe":
        pairs = c["t"] * c["top_k"]
        active = c["e"] * (1 - (1 - c["top_k"] / c["e"]) ** c["t"])  # expected, even routing
        per = (3 * c["i"] * c["h"] / 128) * 2 + c["h"] * c["i"] * (2 * c["bits13"] + c["bits2"]) / 8
        return {"bytes": active * per + 4 * c["t"] * c["h"] + 4 * c["t"] * c["e"],
                "flops": 6.0 * pairs * c["h"] * c["i"]}
    if c["kind"] == "kv":
        vec, d = 2 * c["batch"] * c["heads"], c["head_dim"]
        code = d * c["nbits"] / 8 + 2
        q = [max(0, c["tokens"] + i - c["residual"]) for i in range(c["steps"] + 1)]
        seen = [c["tokens"] + i for i in range(c["steps"] + 1)]
        rows = sum(2 * d * s for s in seen)  # the history that each update returns
        new = 2 * d * (c["tokens"] + c["steps"]) + code * q[-1]
        return {"bytes": vec * (rows + new + sum(code * n for n in q)),
                "flops": vec * d * 14.0 * (q[-1] + sum(q))}
    item = 4 if c["dtype"] == "fp32" else 2
    kp = (c["k"] + 127) // 128 * 128
    return {"bytes": c["n"] * (c["k"] * item + kp * (0.5 if c["pack"] else 1) + kp / 128 * 2),
            "flops": c["n"] * kp * (7.0 + 2.0 * c["bits"])}


# ---------------------------------------------------------------------------
# accuracy
# ---------------------------------------------------------------------------
def tolerance(case):
    if case["kind"] in ("linear", "layers", "moe"):
        # the transformed activation and the weights are fp16 in the products,
        # sums fp32, the result rounded to 16 bits
        if case["dtype"] == "fp16":
            return {"rel": 2e-3, "max": 2e-2}
        return {"rel": 8e-3, "max": 3e-2}
    if case["kind"] == "decode":
        # bf16 residual stream, attention operands and linear outputs; the
        # logits carry the roundings of all layers (about 1.4e-2 off 64 bits)
        return {"rel": 2.8e-2, "max": 0.3}
    if case["kind"] == "kv":
        # bf16 rows; a code may differ where a value lies between two levels
        # to fp32 rounding, which moves a vector by a quantization step
        return {"rel": 8e-3, "max": 0.5, "differ": 1e-4}
    return {"rel": 1e-3, "max": 2e-3, "differ": 1e-4}


def _hadamard(n):
    i = torch.arange(n)
    bits = i[:, None] & i[None, :]
    sign = torch.zeros(n, n, dtype=torch.float64)
    while bool(bits.any()):
        sign += (bits & 1).double()
        bits = bits >> 1
    return ((1 - 2 * (sign % 2)) / math.sqrt(n)).to(_device())


def _dequant(codes, norms, bits):
    """Rows of the weight in the plain (untransformed) domain, 64 bits."""
    cent = [_f32(v) for v in _lloyd_max(1 << bits, True)]
    ct = torch.tensor(cent, dtype=torch.float64, device=codes.device) / math.sqrt(128)
    w = ct[codes.long()].view(codes.shape[0], -1, 128) * norms.double()[..., None]
    return (w @ _hadamard(128)).view(codes.shape[0], -1)


def _f32(v):
    """``v`` rounded to 32 bits, as the codebook is stored."""
    return float(torch.tensor(v, dtype=torch.float32))


def _linear64(x, codes, norms, bits):
    """x [M, K] in 64 bits times the quantized weight, in chunks of rows."""
    xp = torch.nn.functional.pad(x.double(), (0, codes.shape[1] - x.shape[1]))
    return torch.cat([xp @ _dequant(codes[r:r + 4096], norms[r:r + 4096], bits).T
                      for r in range(0, codes.shape[0], 4096)], 1)


def _rms64(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)


def _exact_decode(c, seed):
    w, tokens, kc, vc = _decode_inputs(c, seed)
    B, H, G, D, ctx = c["batch"], c["heads"], c["kv_heads"], c["head_dim"], c["context"]
    x = w["embed"][tokens].double()
    inv = 1.0 / (1.0e6 ** (torch.arange(0, D, 2, device=x.device).double() / D))
    cos, sin = (ctx * inv).cos(), (ctx * inv).sin()
    ks, vs = [], []
    for i, lw in enumerate(w["layers"]):
        lin = lambda name, v: _linear64(v, lw[name]["codes"], lw[name]["norms"],  # noqa: E731
                                        LAYER_BITS[name])
        qkv = lin("qkv_proj", _rms64(x))
        qk = qkv[:, :(H + G) * D].view(B, H + G, D)
        a, b = qk[..., :D // 2], qk[..., D // 2:]
        qk = torch.cat([a * cos - b * sin, b * cos + a * sin], -1)
        k = torch.cat([kc[i].double(), qk[:, H:, None]], 2)  # [B, G, ctx + 1, D]
        v = torch.cat([vc[i].double(), qkv[:, (H + G) * D:].view(B, G, 1, D)], 2)
        p = torch.softmax(qk[:, :H].view(B, G, H // G, D) @ k.transpose(2, 3) / math.sqrt(D), -1)
        x = x + lin("o_proj", (p @ v).view(B, H * D))
        gu = lin("gate_up_proj", _rms64(x))
        gate, up = gu[:, :c["inter"]], gu[:, c["inter"]:]
        x = x + lin("down_proj", torch.nn.functional.silu(gate) * up)
        ks.append(torch.nn.functional.pad(k, (0, 0, 0, 63)).transpose(2, 3))
        vs.append(torch.nn.functional.pad(v, (0, 0, 0, 63)))
    return {"logits": _rms64(x) @ w["lm_head"].double().T, "k_cache": torch.stack(ks),
            "v_cache": torch.stack(vs)}


def _exact_moe(c, seed):
    (c13, n13), (c2, n2), x, logits = _moe_inputs(c, seed)
    lg = logits.double()
    score = torch.softmax(lg, -1) if c["scoring"] == "softmax" else torch.sigmoid(lg)
    wt, ids = torch.topk(score, c["top_k"], -1)
    wt = wt / wt.sum(-1, keepdim=True)
    y = torch.zeros(c["t"], c["h"], dtype=torch.float64, device=x.device)
    for e in range(c["e"]):
        tok, slot = (ids == e).nonzero(as_tuple=True)
        if not tok.numel():
            continue
        gu = _linear64(x[tok], c13[e], n13[e], c["bits13"])
        h = torch.nn.functional.silu(gu[:, :c["i"]]) * gu[:, c["i"]:]
        y.index_add_(0, tok, _linear64(h, c2[e], n2[e], c["bits2"]) * wt[tok, slot][:, None])
    return y


def _exact_kv(c, seed):
    """The history that the last update returns, through stored bf16 norms."""
    d = c["head_dim"]
    had = _hadamard(d)
    cent = torch.tensor([_f32(v) for v in _lloyd_max(1 << c["nbits"], False)],
                        dtype=torch.float64, device=_device())
    mid = (cent[:-1] + cent[1:]) / 2
    full, norms = [], []
    for kv in zip(*_kv_inputs(c, seed)):
        x = torch.cat(kv, 2).double()  # [B, H, S, D]
        n_q = max(0, x.shape[2] - c["residual"])
        old = x[:, :, :n_q]
        nrm = old.norm(dim=-1, keepdim=True).clamp(min=1e-10)
        codes = torch.bucketize((old / nrm) @ had * math.sqrt(d), mid)
        stored = nrm.float().to(torch.bfloat16)
        back = (cent[codes] / math.sqrt(d)) @ had * stored.double()
        full.append(torch.cat([back, x[:, :, n_q:]], 2))
        norms.append([None, stored.double().reshape(-1) if n_q else None])
    return {"full": full, "codes": norms}


def exact(case, seed):
    c = case
    if c["kind"] == "linear":
        codes, norms, x, bias = _linear_inputs(c, seed)
        y = _linear64(x, codes, norms, c["bits"])
        return y if bias is None else y + bias.double()
    if c["kind"] == "layers":
        return [_linear64(x, codes, norms, bits) for bits, codes, norms, x in _layers_inputs(c, seed)]
    if c["kind"] == "decode":
        return _exact_decode(c, seed)
    if c["kind"] == "moe":
        return _exact_moe(c, seed)
    if c["kind"] == "kv":
        return _exact_kv(c, seed)
    w = _quantize_inputs(c, seed).double()
    w = torch.nn.functional.pad(w, (0, -w.shape[1] % 128)).view(w.shape[0], -1, 128)
    ct = torch.tensor(_lloyd_max(1 << c["bits"], True), dtype=torch.float64, device=w.device)
    return {"codes": None, "norms": w.norm(dim=2).clamp(min=1e-10), "ct_scaled": ct / math.sqrt(128)}
