"""What this framework is timed on: the quantized linears of a decoder, from a
single decode projection to a 4001-token prefill layer, the lm_head, the token
embedding and the conversion of floating weights.

Every case is one of five kinds of work:

* ``module``  one ``W8A16Linear`` called as a module, as a model loaded by
  ``load_w8a16_model`` calls each of its projections;
* ``layers``  the projections of ``layers`` consecutive decoder layers (q/k/v
  in one call, o, gate/up in one call, down), int8 or packed int4, at M rows;
* ``head``    the untied int8 lm_head with greedy tokens (logits kept, as a
  sampler that also looks at them does);
* ``embed``   an int8 token embedding looked up for a batch of token ids;
* ``convert`` a floating ``nn.Linear`` on the device quantized and packed into
  the framework's module, as a model is converted at load time.

Weights follow N(0, 0.02) and go through the framework's own quantizers;
activations are N(0, 1) with 1% of the channels scaled by 20, the outlier
channels of a decoder's hidden states.  Decode cases hold enough layers that
the weights come from memory and not from a cache, as they do in a model.
"""
from __future__ import annotations

import math

import torch

import rhinoforge_amd as rf

# (hidden, q, k/v, o's input, intermediate) of the decoders in bench.py.
QWEN3_06B = (1024, 2048, 1024, 2048, 3072)
QWEN3_4B = (2560, 4096, 1024, 4096, 9728)
QWEN3_8B = (4096, 4096, 1024, 4096, 12288)
QWEN3_VL_32B = (5120, 8192, 1024, 8192, 25600)
QWEN25_VL_7B = (3584, 3584, 512, 3584, 18944)


def _layers(name, fmt, m, dims, layers, bias=False):
    h, q, kv, oin, inter = dims
    return {"name": name, "kind": "layers", "fmt": fmt, "m": m, "h": h, "q": q, "kv": kv,
            "oin": oin, "inter": inter, "layers": layers, "bias": bias}


def listed():
    return [
        # The smallest call there is: one fused q/k/v projection of a 0.6B
        # decoder for one token, through its module.  Latency and launch cost.
        {"name": "module_m1", "kind": "module", "m": 1, "n": 3072, "k": 1024, "bias": False},
        # Single-stream decode of an 8B model: four launches a layer, four
        # layers (772 MB of weights, more than the last-level cache holds).
        _layers("decode_m1", "int8", 1, QWEN3_8B, 4),
        # The same model serving 16 sequences at a time.
        _layers("decode_m16", "int8", 16, QWEN3_8B, 4),
        # lm_head of a 14B model for eight sequences: 778 MB of weights.
        {"name": "head_m8", "kind": "head", "m": 8, "n": 151936, "k": 5120},
        # A mid-sized batch (41 sequences) on a 7B decoder with q/k/v biases.
        _layers("batch_m41", "int8", 41, QWEN25_VL_7B, 2, bias=True),
        # A short prompt (512 tokens) through a 32B decoder's layer.
        _layers("prefill_m512", "int8", 512, QWEN3_VL_32B, 1),
        # A long prompt of an odd length through the same layer: the largest.
        _layers("prefill_m4001", "int8", 4001, QWEN3_VL_32B, 1),
        # Group-wise int4 decode of one sequence, 8B.
        _layers("w4_decode_m1", "int4_g32", 1, QWEN3_8B, 8),
        # Group-wise int4 serving 48 sequences, 4B.
        _layers("w4_batch_m48", "int4_g128", 48, QWEN3_4B, 4),
        # Per-channel int4 prefill of a 1000-token prompt, 8B.
        _layers("w4_prefill_m1000", "int4", 1000, QWEN3_8B, 1),
        # Token embedding of a 700-token prompt from an int8 table.
        {"name": "embed_700", "kind": "embed", "m": 700, "n": 151936, "k": 4096},
        # A bf16 gate projection turned into an int8 module at load time.
        {"name": "convert_int8", "kind": "convert", "fmt": "int8", "n": 12288, "k": 4096,
         "dtype": "bfloat16", "bias": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _multiple(rng, lo, hi, step):
    return max(step, _log_int(rng, lo, hi) // step * step)


def draw(rng):
    kind = rng.choice(["module", "layers", "layers", "layers", "layers", "layers", "head", "embed",
                       "convert"])
    if kind == "module":
        return {"kind": "module", "m": _log_int(rng, 1, 512), "n": _log_int(rng, 256, 16384),
                "k": _multiple(rng, 256, 8192, 8), "bias": rng.random() < 0.5}
    if kind == "head":
        return {"kind": "head", "m": _log_int(rng, 1, 64), "n": _log_int(rng, 18992, 151936),
                "k": _multiple(rng, 1024, 5120, 64)}
    if kind == "embed":
        return {"kind": "embed", "m": _log_int(rng, 1, 8192), "n": _log_int(rng, 32000, 151936),
                "k": _multiple(rng, 1024, 5120, 8)}
    if kind == "convert":
        fmt = rng.choice(["int8", "int8", "int4", "int4_g32", "int4_g64", "int4_g128"])
        step = 8 if fmt == "int8" else 128
        return {"kind": "convert", "fmt": fmt, "n": _multiple(rng, 1024, 25600, 1 if step == 8 else 16),
                "k": _multiple(rng, 1024, 12288, step),
                "dtype": rng.choice(["bfloat16", "float16", "float32"]), "bias": rng.random() < 0.3}
    fmt = rng.choice(["int8", "int8", "int8", "int4", "int4_g32", "int4_g64", "int4_g128"])
    dims = rng.choice([QWEN3_06B, QWEN3_4B, QWEN3_8B, QWEN3_VL_32B, QWEN25_VL_7B, None, None])
    if dims is None:  # a decoder of no particular make, odd widths among them for int8
        step = 8 if fmt == "int8" else 128
        dims = (_multiple(rng, 896, 5120, step), _multiple(rng, 896, 8192, step),
                _multiple(rng, 128, 1024, step), _multiple(rng, 896, 8192, step),
                _multiple(rng, 2048, 25600, step))
    m = _log_int(rng, 1, 4000)
    h, q, kv, oin, inter = dims
    params = h * (q + 2 * kv + oin + 3 * inter)
    per_weight = 1 if fmt == "int8" else 0.5
    layers = min(8, max(1, round(6e8 / (params * per_weight)))) if m <= 64 else 1
    c = _layers("", fmt, m, dims, layers, bias=rng.random() < 0.3)
    del c["name"]
    return c


# ---- inputs --------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _activation(g, m, k):
    x = torch.randn(m, k, generator=g, device="cuda")
    loud = torch.randperm(k, generator=g, device="cuda")[: max(1, k // 100)]
    x[:, loud] *= 20.0
    return x.half()


def _weight(g, n, k):
    return torch.randn(n, k, generator=g, device="cuda").mul_(0.02)


def _group(fmt):
    return int(fmt[6:]) if fmt.startswith("int4_g") else 0


def _quantize(w, fmt):
    if fmt == "int8":
        return rf.quantize_linear_per_channel(w)
    if fmt == "int4":
        return rf.quantize_int4_per_channel(w)
    q, s, _ = rf.quantize_int4_group_wise(w, _group(fmt))
    return q, s


def _projection(g, n, k, fmt, bias):
    """(packed weight, scale, bias or None), and the quantized values they came from."""
    q, s = _quantize(_weight(g, n, k), fmt)
    b = (torch.randn(n, generator=g, device="cuda") * 0.1).half() if bias else None
    pack = rf.pack_weight if fmt == "int8" else rf.pack_weight_int4
    return (pack(q), s, b), q


def _layer_shapes(c):
    """(output widths, input width, which input) of a layer's four calls."""
    return [((c["q"], c["kv"], c["kv"]), c["h"], "hidden"), ((c["h"],), c["oin"], "context"),
            ((c["inter"], c["inter"]), c["h"], "normed"), ((c["h"],), c["inter"], "act")]


def _build(c, seed, keep_q):
    """The state of a case; with keep_q also the quantized values, for exact()."""
    g = _gen(seed)
    kind = c["kind"]
    if kind in ("module", "head"):
        x = _activation(g, c["m"], c["k"])
        (w, s, b), q = _projection(g, c["n"], c["k"], "int8", c.get("bias", False))
        st = {"kind": kind, "x": x, "w": w, "s": s, "b": b}
        if kind == "module":
            st["mod"] = rf.W8A16Linear.from_quantized(q, s, b)
        if keep_q:
            st["q"] = q
        return st
    if kind == "layers":
        xs = {name: _activation(g, c["m"], k) for _, k, name in _layer_shapes(c)}
        st = {"kind": kind, "fmt": c["fmt"], "x": xs, "layers": []}
        for _ in range(c["layers"]):
            calls = []
            for ns, k, name in _layer_shapes(c):
                ps = [_projection(g, n, k, c["fmt"], c["bias"] and name == "hidden") for n in ns]
                call = {"x": name, "w": [p[0][0] for p in ps], "s": [p[0][1] for p in ps],
                        "b": [p[0][2] for p in ps]}
                if keep_q:
                    call["q"] = [p[1] for p in ps]
                calls.append(call)
            st["layers"].append(calls)
        return st
    if kind == "embed":
        q, s = rf.quantize_linear_per_channel(_weight(g, c["n"], c["k"]))
        ids = torch.randint(0, c["n"], (1, c["m"]), generator=g, device="cuda")
        return {"kind": kind, "mod": rf.W8A16Embedding(q, s), "ids": ids}
    lin = torch.nn.Linear(c["k"], c["n"], bias=c["bias"], device="meta")
    lin.weight = torch.nn.Parameter(_weight(g, c["n"], c["k"]).to(getattr(torch, c["dtype"])))
    if c["bias"]:
        lin.bias = torch.nn.Parameter((torch.randn(c["n"], generator=g, device="cuda") * 0.1
                                       ).to(lin.weight.dtype))
    return {"kind": kind, "fmt": c["fmt"], "lin": lin}


def prepare(case, seed):
    return _build(case, seed, False)


# ---- one pass ------------------------------------------------------------------

def run(state):
    kind = state["kind"]
    if kind == "module":
        return state["mod"](state["x"])
    if kind == "head":
        return rf.linear_argmax(state["x"], state["w"], state["s"], return_logits=True)
    if kind == "embed":
        return state["mod"](state["ids"])
    if kind == "convert":
        fmt = state["fmt"]
        if fmt == "int8":
            mod = rf.W8A16Linear.from_linear(state["lin"])
        else:
            mod = rf.W4A16Linear.from_linear(state["lin"], group_size=_group(fmt) or None)
        out = [mod.weight, mod.weight_scale]
        return out if mod.bias is None else out + [mod.bias]
    int8 = state["fmt"] == "int8"
    one = rf.linear if int8 else rf.linear_w4a16
    several = rf.linear_multi if int8 else rf.linear_multi_w4a16
    out = []
    for calls in state["layers"]:
        for call in calls:
            x = state["x"][call["x"]]
            if len(call["w"]) == 1:
                out.append(one(x, call["w"][0], call["s"][0], call["b"][0]))
            else:
                out.extend(several(x, call["w"], call["s"], call["b"]))
    return out


# ---- what a pass cannot do without ----------------------------------------------

def _linear_work(m, n, k, fmt, bias):
    gs = _group(fmt)
    weights = n * k * (1 if fmt == "int8" else 0.5)
    scales = 2 * n * (k // gs if gs else 1)
    return weights + scales + 2 * m * n + (2 * n if bias else 0), 2 * m * n * k


def work(case):
    kind = case["kind"]
    if kind in ("module", "head"):
        by, fl = _linear_work(case["m"], case["n"], case["k"], "int8", case.get("bias", False))
        return {"bytes": int(by + 2 * case["m"] * case["k"]), "flops": fl}
    if kind == "embed":  # ids (int64), the distinct rows and their scales at most, fp16 rows out
        rows = min(case["m"], case["n"])
        return {"bytes": 8 * case["m"] + rows * (case["k"] + 2) + 2 * case["m"] * case["k"],
                "flops": case["m"] * case["k"]}
    if kind == "convert":
        n, k, fmt = case["n"], case["k"], case["fmt"]
        size = 4 if case["dtype"] == "float32" else 2
        by, _ = _linear_work(0, n, k, fmt, False)
        return {"bytes": int(size * n * k + by + ((size + 2) * n if case["bias"] else 0)),
                "flops": 3 * n * k}
    total_b = total_f = 0
    for ns, k, name in _layer_shapes(case):
        total_b += 2 * case["m"] * k
        for n in ns:
            by, fl = _linear_work(case["m"], n, k, case["fmt"], case["bias"] and name == "hidden")
            total_b += by
            total_f += fl
    return {"bytes": int(total_b * case["layers"]), "flops": total_f * case["layers"]}


def tolerance(case):
    """Whole numbers and single-rounding results are exact.  A linear's fp16
    results are one rounding of an fp32 sum: against 64 bits the present code
    is 2.1e-4 off in the 2-norm and at most one fp16 rounding (4.9e-4 of the
    value, 9.8e-4 where the two sides round apart) at any element."""
    if case["kind"] in ("embed", "convert"):
        return "exact"
    return {"rel": 8e-4, "max": 2e-3, "differ": 0.0}


# ---- the same in 64 bits ---------------------------------------------------------

def _linear64(x, q, s, b):
    """x . W^T (+ b) in float64, W = s[n] q[n, k], or the fp16 weight
    RN(s[k / gs, n] q[n, k]) that defines group-wise int4."""
    x64 = x.double()
    y = torch.empty(x.size(0), q.size(0), dtype=torch.float64, device=x.device)
    for r in range(0, q.size(0), 8192):
        qr = q[r:r + 8192].double()
        if s.dim() == 1:
            y[:, r:r + 8192] = (x64 @ qr.t()) * s[r:r + 8192].double()
        else:
            gs = q.size(1) // s.size(0)
            w = qr * s[:, r:r + 8192].t().double().repeat_interleave(gs, dim=1)
            y[:, r:r + 8192] = x64 @ w.half().double().t()
    return y if b is None else y + b.double()


def exact(case, seed):
    kind = case["kind"]
    if kind == "convert":
        return None  # whole numbers and fp16 steps, compared as they are
    st = _build(case, seed, True)
    if kind == "module":
        return _linear64(st["x"], st["q"], st["s"], st["b"])
    if kind == "head":
        return None, _linear64(st["x"], st["q"], st["s"], None)
    if kind == "embed":
        mod, ids = st["mod"], st["ids"]
        return mod.weight[ids].double() * mod.weight_scale[ids].double().unsqueeze(-1)
    out = []
    for calls in st["layers"]:
        for call in calls:
            x = st["x"][call["x"]]
            out.extend(_linear64(x, q, s, b) for q, s, b in zip(call["q"], call["s"], call["b"]))
    return out
