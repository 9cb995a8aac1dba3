"""The work that a program has this library do, as cases that can be timed and compared.

One case is one pass through the public entry points (the operator events of `emel_hip`, its generic
envelope, row gather and logits sampler), at the sizes of a decoder's layers: the prompt's pass over
hundreds of tokens, the decode step of one or a few sequences, the output head and the sampler over a
vocabulary, the embedding lookup, and the gradients that the envelope serves.  Sizes are those of this
repository's benchmark (hidden 4096, MLP 11008, 512-token prompts, 32 heads, 151936 logits) and generic
ones around them.

  listed()           the named cases
  draw(rng)          one more case of the same ranges
  prepare(c, seed)   inputs on the GPU, made from the seed, and the views and handles a program keeps
  run(state)         one pass; returns every output it writes
  work(c)            bytes and operations that the pass cannot do without
  tolerance(c)       how far another correct implementation may be
  exact(c, seed)     the same outputs in 64 bits, by plain torch
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "emel.rs_amd"))
import emel_hip as eh  # noqa: E402

EPS = 1e-5
# values and bytes of one block of each packed format
PACKED = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144)}


def listed():
    return [
        # One token of one sequence through a layer's residual and norm: three launches on 16 KB, so the call itself counts.
        {"name": "norm_decode", "kind": "norm", "cols": 4096, "rows": 1},
        # The same over a long prompt (the benchmark's normalisation size).
        {"name": "norm_prompt", "kind": "norm", "cols": 4096, "rows": 2048},
        # The MLP's gate over a 512-token prompt.
        {"name": "gate_prompt", "kind": "gate", "act": "swiglu", "cols": 11008, "rows": 512},
        # Attention weights of a 512-token prompt chunk behind 3584 cached tokens: scale, causal mask, soft_max.
        {"name": "softmax_prompt", "kind": "softmax", "kv": 4096, "q": 512, "heads": 32, "batch": 1},
        # A decode step of 8 sequences: one query each; the number of cached tokens grows by one a step, so it is rarely round.
        {"name": "softmax_decode", "kind": "softmax", "kv": 3001, "q": 1, "heads": 32, "batch": 8},
        # Greedy tokens of 64 sequences from their logits.
        {"name": "greedy_batch", "kind": "greedy", "card": 151936, "rows": 64},
        # Sampled tokens of 64 sequences served together.
        {"name": "sample_batch", "kind": "sample", "card": 151936, "rows": 64, "top_k": 40, "temperature": 0.8},
        # The sampled token of one sequence: latency.
        {"name": "sample_one", "kind": "sample", "card": 151936, "rows": 1, "top_k": 40, "temperature": 0.8},
        # The embedding rows of a 512-token prompt from a packed table, ids as the tokenizer leaves them (host memory).
        {"name": "embed_prompt", "kind": "embed", "format": "q4_k", "cols": 4096, "vocab": 32000, "ids": 512, "on_host": True},
        # A projection of a 512-token prompt with half-precision weights.
        {"name": "project_prompt", "kind": "project", "dtype": "f16", "k": 4096, "m": 4096, "n": 512},
        # The greedy output head of one sequence: hidden state times the whole head, only the best row's index and value.
        {"name": "head_greedy", "kind": "head", "k": 4096, "m": 151936},
        # The gradients that the envelope serves, for one layer of a 512-token sequence: norm, MLP gate, attention weights.
        {"name": "backward_layer", "kind": "backward", "tokens": 512, "cols": 4096, "width": 11008, "kv": 512, "heads": 32},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["norm", "gate", "softmax", "greedy", "sample", "embed", "project", "head", "backward"])
    if kind == "norm":  # hidden sizes are multiples of 32, token counts any
        return {"kind": kind, "cols": 32 * _log(rng, 16, 256), "rows": _log(rng, 1, 4000)}
    if kind == "gate":
        return {"kind": kind, "act": rng.choice(["swiglu", "silu", "gelu"]), "cols": 32 * _log(rng, 32, 448),
                "rows": _log(rng, 1, 1024)}
    if kind == "softmax":
        kv, heads = _log(rng, 64, 16384), rng.choice([8, 16, 32, 40])
        batch = _log(rng, 1, 16)
        q = min(_log(rng, 1, 512), max(1, 40_000_000 // (kv * heads * batch)))
        return {"kind": kind, "kv": kv, "q": q, "heads": heads, "batch": batch}
    if kind == "greedy":
        return {"kind": kind, "card": _log(rng, 32000, 200000), "rows": _log(rng, 1, 64)}
    if kind == "sample":
        return {"kind": kind, "card": _log(rng, 32000, 151936), "rows": _log(rng, 1, 64), "top_k": _log(rng, 1, 256),
                "temperature": round(rng.uniform(0.5, 1.3), 2)}
    if kind == "embed":
        return {"kind": kind, "format": rng.choice(["f32", "f16", "bf16", "q8_0", "q4_0", "q4_k"]),
                "cols": 256 * _log(rng, 2, 32), "vocab": _log(rng, 8000, 64000), "ids": _log(rng, 1, 4096),
                "on_host": rng.random() < 0.7}
    if kind == "project":
        k, m = 32 * _log(rng, 16, 256), _log(rng, 512, 11008)
        n = min(_log(rng, 1, 512), max(1, 8_000_000_000 // (k * m)))
        return {"kind": kind, "dtype": rng.choice(["f16", "f32"]), "k": k, "m": m, "n": n}
    if kind == "head":
        return {"kind": kind, "k": 32 * _log(rng, 16, 128), "m": _log(rng, 32000, 151936)}
    return {"kind": kind, "tokens": _log(rng, 16, 640), "cols": 32 * _log(rng, 16, 160), "width": 32 * _log(rng, 32, 400),
            "kv": _log(rng, 33, 700), "heads": rng.choice([8, 16, 32])}


# ---- inputs -------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, n, scale=1.0):
    return torch.empty(n, device="cuda").normal_(0.0, scale, generator=g)


def _view(t, ne, dtype=eh.DType.F32):
    return eh.TensorView(t, eh.Layout.dense(dtype, ne))


def _out(ne, dtype=torch.float32):
    t = torch.empty(math.prod(ne), dtype=dtype, device="cuda")
    return t, eh.TensorViewMut(t, eh.Layout.dense(eh.DType.I32 if dtype == torch.int32 else eh.DType.F32, ne))


def _norm_inputs(c, g):
    n = c["cols"] * c["rows"]
    x = _normal(g, n)
    # activations have a few tokens with far larger values: 1% of them x100, as in the benchmark
    big = torch.rand(c["rows"], device="cuda", generator=g) < 0.01
    x.view(c["rows"], c["cols"])[big] *= 100.0
    return x, _normal(g, n), torch.empty(c["cols"], device="cuda").uniform_(0.5, 1.5, generator=g)


def _softmax_inputs(c, g):
    kv, q = c["kv"], c["q"]
    x = _normal(g, kv * q * c["heads"] * c["batch"], 2.0 * math.sqrt(128.0))  # scores before the scale
    last = torch.arange(q, device="cuda")[:, None] + (kv - q)
    mask = torch.zeros(q, kv, dtype=torch.float16, device="cuda")
    mask.masked_fill_(torch.arange(kv, device="cuda")[None, :] > last.clamp_min(0), float("-inf"))
    return x, mask.reshape(-1), float(np.float32(1.0 / math.sqrt(128.0)))


def _sample_inputs(c, g):
    # a head's logits: a wide bulk; the tail of 151936 normal values makes the few likely tokens
    logits = _normal(g, c["card"] * c["rows"], 2.5)
    states = torch.randint(1, 2**31 - 1, (c["rows"],), device="cuda", generator=g).cpu().numpy().astype(np.uint32)
    return logits, states


def _embed_inputs(c, g):
    f, cols, vocab = c["format"], c["cols"], c["vocab"]
    ids = torch.randint(0, vocab, (c["ids"],), device="cuda", generator=g, dtype=torch.int32)
    if f not in PACKED:
        kind = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[f]
        return _normal(g, cols * vocab).to(kind), ids
    values, size = PACKED[f]
    blocks = cols * vocab // values
    table = torch.randint(0, 256, (blocks, size), device="cuda", generator=g, dtype=torch.uint8)
    heads = 2 if f == "q4_k" else 1  # the half-precision scale (and minimum) that opens a block
    scales = torch.empty(blocks, heads, device="cuda").uniform_(0.001, 0.02, generator=g).half()
    table[:, : 2 * heads] = scales.view(torch.uint8)
    return table.reshape(-1), ids


def _project_inputs(c, g):
    w = _normal(g, c["k"] * c["m"], 0.02)
    x = _normal(g, c["k"] * c["n"])
    return (w.half(), x.half()) if c["dtype"] == "f16" else (w, x)


def _head_inputs(c, g):
    w, h = _normal(g, c["k"] * c["m"], 0.02), _normal(g, c["k"])
    best = int(torch.randint(0, c["m"], (1,), device="cuda", generator=g))
    w.view(c["m"], c["k"])[best] += 0.01 * h  # a head that knows its next token
    return w, h


def _backward_inputs(c, g):
    t, n, wide, rows = c["tokens"], c["cols"], c["width"], c["tokens"] * c["heads"]
    p = torch.softmax(_normal(g, rows * c["kv"], 2.0).view(rows, c["kv"]), 1).reshape(-1)
    return {"x": _normal(g, t * n), "dy": _normal(g, t * n, 0.01), "gate": _normal(g, t * wide),
            "dgate": _normal(g, t * wide, 0.01), "p": p, "dp": _normal(g, rows * c["kv"], 0.01)}


def prepare(c, seed):
    g, kind = _gen(seed), c["kind"]
    s = {"case": c, "kernel": eh.Kernel(synchronous=False)}
    if kind == "norm":
        ne = [c["cols"], c["rows"], 1, 1]
        x, dx, w = _norm_inputs(c, g)
        s["x"], s["dx"], s["w"] = _view(x, ne), _view(dx, ne), _view(w, [c["cols"], 1, 1, 1])
        h, s["h"] = _out(ne)
        y, s["y"] = _out(ne)
        s["h_in"], s["y_in"] = _view(h, ne), _view(y, ne)
        s["out"] = {"residual": h, "normed": y}
    elif kind == "gate":
        ne = [c["cols"], c["rows"], 1, 1]
        n = c["cols"] * c["rows"]
        s["a"] = _view(_normal(g, n), ne)
        if c["act"] == "swiglu":
            s["b"] = _view(_normal(g, n), ne)
        y, s["y"] = _out(ne)
        s["out"] = y
    elif kind == "softmax":
        ne = [c["kv"], c["q"], c["heads"], c["batch"]]
        x, mask, s["scale"] = _softmax_inputs(c, g)
        s["x"], s["mask"] = _view(x, ne), _view(mask, [c["kv"], c["q"], 1, 1], eh.DType.F16)
        y, s["y"] = _out(ne)
        s["out"] = y
    elif kind == "greedy":
        s["x"] = _view(_normal(g, c["card"] * c["rows"]), [c["card"], c["rows"], 1, 1])
        y, s["y"] = _out([1, c["rows"], 1, 1], torch.int32)
        s["out"] = y
    elif kind == "sample":
        rows, card, k = c["rows"], c["card"], c["top_k"]
        logits, s["states"] = _sample_inputs(c, g)
        s["logits"], s["probs"] = logits, torch.empty_like(logits)
        i32 = dict(dtype=torch.int32, device="cuda")
        s["sorted"] = torch.zeros(rows * card, **i32)
        s["top_p"], s["top_i"] = torch.zeros(rows * k, device="cuda"), torch.zeros(rows * k, **i32)
        s["token"], s["score"] = torch.zeros(rows, **i32), torch.zeros(rows, device="cuda")
        s["sampler"] = eh.Sampler()
        s["out"] = {n: s[n] for n in ("probs", "top_p", "top_i", "token", "score")}
    elif kind == "embed":
        f, cols, vocab, n = c["format"], c["cols"], c["vocab"], c["ids"]
        table, ids = _embed_inputs(c, g)
        code = {"f32": eh.DType.F32, "f16": eh.DType.F16, "bf16": eh.DType.BF16, "q8_0": eh.DType.Q8_0,
                "q4_0": eh.DType.Q4_0, "q4_k": eh.DType.Q4_K}[f]
        make = eh.Layout.packed if f in PACKED else eh.Layout.dense
        s["table"] = eh.TensorView(table, make(code, [cols, vocab, 1, 1]))
        s["ids"] = ids.cpu().numpy() if c["on_host"] else ids
        s["event"] = {"f32": eh.OpGetRows, "f16": eh.OpGetRowsF16, "bf16": eh.OpGetRowsBf16, "q8_0": eh.OpGetRowsQ8_0,
                      "q4_0": eh.OpGetRowsQ4_0, "q4_k": eh.OpGetRowsQ4K}[f]
        y, s["y"] = _out([cols, n, 1, 1])
        s["out"] = y
    elif kind == "project":
        k, m, n = c["k"], c["m"], c["n"]
        w, x = _project_inputs(c, g)
        if c["dtype"] == "f16":
            s["w"], s["x"] = _view(w, [k, m, 1, 1], eh.DType.F16), _view(x, [k, n, 1, 1], eh.DType.F16)
            y, s["y"] = _out([m, n, 1, 1])
        else:
            s["w"], s["x"] = _view(w, [k, m, 1, 1]), _view(x, [n, k, 1, 1])
            y, s["y"] = _out([n, m, 1, 1])
        s["out"] = y
    elif kind == "head":
        w, h = _head_inputs(c, g)
        s["w"], s["h"] = _view(w, [c["k"], c["m"], 1, 1]), _view(h, [c["k"], 1, 1, 1])
        y, s["y"] = _out([1, 1, 1, 1])
        s["index"] = torch.zeros(1, dtype=torch.int32, device="cuda")
        s["out"] = {"value": y, "index": s["index"]}
    else:
        v = _backward_inputs(c, g)
        ne = {"x": [c["cols"], c["tokens"], 1, 1], "gate": [c["width"], c["tokens"], 1, 1],
              "p": [c["kv"], c["tokens"], c["heads"], 1]}
        ne.update(dy=ne["x"], dgate=ne["gate"], dp=ne["p"])
        s["in"] = {n: _view(t, ne[n]) for n, t in v.items()}
        outs = {n: _out(ne[n]) for n in ("x", "gate", "p")}
        s["grad"] = {n: o[1] for n, o in outs.items()}
        s["out"] = {n: o[0] for n, o in outs.items()}
    return s


# ---- one pass -----------------------------------------------------------------------------


def _ok(status):
    if status != eh.Status.OK:
        raise RuntimeError(f"{eh.Status(status).name}: {eh.last_error()}")


def _generic(s, op, src0, src1, dst, params=None, index_out=None):
    r = eh.GenericRequest(op, src0, src1, None, dst, params or eh.OpParams.empty())
    if index_out is not None:
        r.with_index_out(index_out)
    _ok(s["kernel"].process_event(eh.GenericEvent(r)))


def run(s):
    c, call = s["case"], s["kernel"].process_event
    kind = c["kind"]
    if kind == "norm":
        _ok(call(eh.OpAdd(s["x"], s["dx"], s["h"])))
        if c["rows"] > 1:
            _ok(call(eh.OpRmsNormMul(s["h_in"], s["w"], s["y"], EPS)))
        else:  # a row broadcast asks for two rows or more: one token's norm is followed by a product
            _ok(call(eh.OpRmsNorm(s["h_in"], s["y"], EPS)))
            _ok(call(eh.OpMul(s["y_in"], s["w"], s["y"])))
    elif kind == "gate":
        if c["act"] == "swiglu":
            _ok(call(eh.OpSwiglu(s["a"], s["b"], s["y"])))
        else:
            _ok(call((eh.OpSilu if c["act"] == "silu" else eh.OpGelu)(s["a"], s["y"])))
    elif kind == "softmax":
        _ok(call(eh.OpSoftMaxExt(s["x"], s["mask"], s["scale"], s["y"])))
    elif kind == "greedy":
        _ok(call(eh.OpArgmaxRows(s["x"], s["y"])))
    elif kind == "sample":
        # the sampler turns its logits into probabilities in place; the copy stands for the head that writes them anew
        _ok(call(eh.DenseOpDup(s["logits"], s["probs"])))
        req = eh.SampleTemperatureTopK(c["card"], c["temperature"], c["top_k"], s["probs"], s["sorted"], s["top_p"],
                                       s["top_i"], s["states"], s["token"], s["score"])
        _ok(s["sampler"].sample_temperature_top_k_rows(req, c["rows"], c["card"], c["card"], c["top_k"])[0])
    elif kind == "embed":
        _ok(call(s["event"](s["table"], eh.IndexView(s["ids"], [c["ids"], 1, 1]), s["y"])))
    elif kind == "project":
        _generic(s, eh.GenericOp.MUL_MAT, s["w"], s["x"], s["y"])
    elif kind == "head":
        _generic(s, eh.GenericOp.MUL_MAT_ARGMAX, s["w"], s["h"], s["y"], index_out=s["index"])
    else:
        i, d = s["in"], s["grad"]
        _generic(s, eh.GenericOp.RMS_NORM_BACK, i["x"], i["dy"], d["x"], eh.OpParams.f32(EPS))
        _ok(call(eh.OpSiluBack(i["gate"], i["dgate"], d["gate"])))
        _generic(s, eh.GenericOp.SOFT_MAX_BACK, i["p"], i["dp"], d["p"], eh.OpParams.i32(c["kv"]))
    return s["out"]


# ---- what a pass costs at least, and how exact it is -----------------------------------------


def work(c):
    kind = c["kind"]
    if kind == "norm":  # x, dx, w in; residual and normed out
        n = c["cols"] * c["rows"]
        return {"bytes": 16 * n + 4 * c["cols"], "flops": 5 * n}
    if kind == "gate":
        n = c["cols"] * c["rows"]
        return {"bytes": (12 if c["act"] == "swiglu" else 8) * n, "flops": 4 * n}
    if kind == "softmax":
        n = c["kv"] * c["q"] * c["heads"] * c["batch"]
        return {"bytes": 8 * n + 2 * c["kv"] * c["q"], "flops": 6 * n}
    if kind == "greedy":
        return {"bytes": 4 * (c["card"] + 1) * c["rows"], "flops": c["card"] * c["rows"]}
    if kind == "sample":  # logits in, probabilities and the ranked top_k out
        return {"bytes": c["rows"] * (8 * c["card"] + 12 * c["top_k"] + 8), "flops": 4 * c["rows"] * c["card"]}
    if kind == "embed":
        values, size = PACKED.get(c["format"], (1, 4 if c["format"] == "f32" else 2))
        return {"bytes": c["ids"] * (c["cols"] * size // values + 4 * c["cols"] + 4), "flops": c["ids"] * c["cols"]}
    if kind == "project":
        size = 2 if c["dtype"] == "f16" else 4
        k, m, n = c["k"], c["m"], c["n"]
        return {"bytes": size * k * (m + n) + 4 * m * n, "flops": 2 * k * m * n}
    if kind == "head":
        return {"bytes": 4 * c["k"] * (c["m"] + 1) + 8, "flops": 2 * c["k"] * c["m"]}
    a, b, p = c["tokens"] * c["cols"], c["tokens"] * c["width"], c["tokens"] * c["heads"] * c["kv"]
    return {"bytes": 12 * (a + b + p), "flops": 8 * a + 8 * b + 4 * p}


def tolerance(c):
    kind = c["kind"]
    if kind in ("greedy", "embed"):
        return "exact"  # whole numbers; decoded values, whose few roundings have a fixed order
    if kind == "gate" and c["act"] == "gelu":
        return {"rel": 2e-3}  # the formula rounds through half precision
    if kind == "sample":
        # a 32-bit sum of up to 151936 terms, most of them below half a unit of its last place: measured 2.4e-4
        return {"rel": 1e-3, "max": 5e-3, "differ": 0.02}
    if kind == "project":
        # measured against 64 bits: 5e-7 for 32-bit sums, 2.5e-8 for the half products' 64-bit sums
        return {"rel": 2e-6, "max": 1e-4} if c["dtype"] == "f32" else {"rel": 1e-7, "max": 1e-5}
    if kind == "head":
        return {"rel": 3e-6}
    return {"rel": 1e-6, "max": 6e-4}  # measured 5e-8 to 2e-7, single values to 1.5e-4 of the rms


def _decode(c, rows):
    """f64 values of packed rows [ids, blocks, block bytes]."""
    f = c["format"]
    half = lambda i: rows[..., i : i + 2].contiguous().view(torch.float16).double()  # noqa: E731
    if f == "q8_0":
        return half(0) * rows[..., 2:].contiguous().view(torch.int8).double()
    if f == "q4_0":
        q = rows[..., 2:]
        return half(0) * (torch.cat([q & 15, q >> 4], -1).double() - 8.0)
    s, q = rows[..., 4:16].int(), rows[..., 16:]
    sc = torch.cat([s[..., :4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], -1).double()
    mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1).double()
    q = q.reshape(*q.shape[:-1], 4, 1, 32)
    q = torch.cat([q & 15, q >> 4], -2).reshape(*q.shape[:-3], 8, 32).double()
    return (half(0) * sc).unsqueeze(-1) * q - (half(2) * mn).unsqueeze(-1)


def exact(c, seed):
    g, kind = _gen(seed), c["kind"]
    if kind == "norm":
        x, dx, w = (t.double() for t in _norm_inputs(c, g))
        h = (x + dx).view(c["rows"], c["cols"])
        y = h * torch.rsqrt(h.square().mean(1, keepdim=True) + EPS) * w
        return {"residual": h.reshape(-1), "normed": y.reshape(-1)}
    if kind == "gate":
        n = c["cols"] * c["rows"]
        a = _normal(g, n).double()
        if c["act"] == "swiglu":
            return a * torch.sigmoid(a) * _normal(g, n).double()
        if c["act"] == "silu":
            return a * torch.sigmoid(a)
        return torch.nn.functional.gelu(a, approximate="tanh")
    if kind == "softmax":
        x, mask, scale = _softmax_inputs(c, g)
        x = x.double().view(c["batch"] * c["heads"], c["q"], c["kv"]) * scale
        return torch.softmax(x + mask.double().view(c["q"], c["kv"]), -1).reshape(-1)
    if kind == "greedy":
        return None  # indices of values that are not computed
    if kind == "sample":
        logits, _ = _sample_inputs(c, g)
        p = torch.softmax(logits.double().view(c["rows"], c["card"]) / c["temperature"], -1)
        top = torch.topk(p, c["top_k"], -1).values
        return {"probs": p.reshape(-1), "top_p": top.reshape(-1), "top_i": None, "token": None, "score": None}
    if kind == "embed":
        table, ids = _embed_inputs(c, g)
        rows = table.view(c["vocab"], -1)[ids.long()]
        if c["format"] in PACKED:
            rows = _decode(c, rows.view(c["ids"], -1, PACKED[c["format"]][1]))
        return rows.double().reshape(-1)
    if kind == "project":
        w, x = (t.double() for t in _project_inputs(c, g))
        if c["dtype"] == "f16":  # [n, m], the inner dimension last in both
            return (x.view(c["n"], c["k"]) @ w.view(c["m"], c["k"]).T.contiguous()).reshape(-1)
        return (w.view(c["m"], c["k"]) @ x.view(c["k"], c["n"])).reshape(-1)
    if kind == "head":
        w, h = _head_inputs(c, g)
        return {"value": (w.view(c["m"], c["k"]).double() @ h.double()).max().reshape(1), "index": None}
    v = {n: t.double() for n, t in _backward_inputs(c, g).items()}
    x, dy = v["x"].view(-1, c["cols"]), v["dy"].view(-1, c["cols"])
    inv = torch.rsqrt(x.square().mean(1, keepdim=True) + EPS)
    gx = dy * inv - x * inv**3 * (x * dy).mean(1, keepdim=True)
    s = torch.sigmoid(v["gate"])
    p, dp = v["p"].view(-1, c["kv"]), v["dp"].view(-1, c["kv"])
    return {"x": gx.reshape(-1), "gate": v["dgate"] * s * (1.0 + v["gate"] * (1.0 - s)),
            "p": (p * (dp - (p * dp).sum(1, keepdim=True))).reshape(-1)}
