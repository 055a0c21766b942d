"""Performance cases: what a program that runs a quantized GGUF model through ``HipBackend`` asks of it.

A case is a dict of plain values.  Kinds:

* ``matmul``: one linear operator, ``Backend::quantized_matmul`` on device tensors.
* ``layer``: the quantized operators of one decoder layer: the Q, K and V projections as one batch call, the
  output projection, the feed-forward block.  A step of decoding has one row per sequence, a prefill chunk one row
  per token of the prompt.
* ``moe``: router and routed experts of one mixture-of-experts layer.
* ``lm_head``: the output matrix and the greedy token behind it.
* ``embedding``: the lookup of a step's or a prompt's tokens in a quantized table.
* ``dequantize``: a whole matrix to f32.

``elem`` is the element type of activations and outputs ("f32", "f16", "bf16"; "f32_bf16": f32 tensors whose
activations the call rounds to bf16).  ``mix`` names the formats of a layer's matrices as GGUF files combine them.
"""
from __future__ import annotations

import math

import torch

from gllm_amd import backend as B
from gllm_amd.ggml import block_bytes, block_size, row_bytes

Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14
FORMATS = {"q8_0": Q8_0, "q4_k": Q4_K, "q5_k": Q5_K, "q6_k": Q6_K}
#: (attention and gate/up format, down format)
MIXES = {"q4_k_m": (Q4_K, Q6_K), "q5_k_m": (Q5_K, Q6_K), "q6_k": (Q6_K, Q6_K), "q8_0": (Q8_0, Q8_0), "q4_k_s": (Q4_K, Q4_K)}
ELEMS = {"f32": torch.float32, "f32_bf16": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # the smallest projection of a small model, one token: latency of the call and its launch
        {"name": "matmul_small", "kind": "matmul", "format": "q4_k", "elem": "f32", "m": 1, "n": 512, "k": 2048},
        # one token through a layer of an 8B-class model in the most common mix
        {"name": "decode_layer", "kind": "layer", "mix": "q4_k_m", "elem": "f32", "m": 1, "hidden": 4096, "kv": 1024, "ffn": 14336},
        # sixteen sequences decoded together by a bf16 executor
        {"name": "decode_layer_batch", "kind": "layer", "mix": "q4_k_m", "elem": "bf16", "m": 16, "hidden": 4096, "kv": 1024, "ffn": 14336},
        # a short prompt against a matrix whose rows are no multiple of anything but the format's block
        {"name": "matmul_ragged", "kind": "matmul", "format": "q8_0", "elem": "f16", "m": 77, "n": 4999, "k": 2880},
        # a larger decode batch on a 13B-class gate projection
        {"name": "matmul_batch", "kind": "matmul", "format": "q5_k", "elem": "f32", "m": 48, "n": 13824, "k": 5120},
        # a prefill chunk, f32 activations as the reference passes them
        {"name": "matmul_prefill", "kind": "matmul", "format": "q4_k", "elem": "f32", "m": 512, "n": 14336, "k": 4096},
        # a long prompt through a whole layer
        {"name": "prefill_layer", "kind": "layer", "mix": "q4_k_m", "elem": "bf16", "m": 2048, "hidden": 4096, "kv": 1024, "ffn": 14336},
        # a decode batch through a layer of many small experts
        {"name": "moe_decode", "kind": "moe", "mix": "q4_k_m", "elem": "f32", "m": 16, "hidden": 4096, "ffn": 1536, "experts": 128, "top_k": 8},
        # a prefill chunk through the same layer: every expert sees some tens of tokens
        {"name": "moe_prefill", "kind": "moe", "mix": "q4_k_m", "elem": "bf16", "m": 512, "hidden": 4096, "ffn": 1536, "experts": 128, "top_k": 8},
        # the end of a greedy decode step
        {"name": "lm_head", "kind": "lm_head", "format": "q6_k", "n": 128256, "k": 4096, "logits": False},
        # a prompt's tokens looked up in the table
        {"name": "embedding", "kind": "embedding", "format": "q4_k", "elem": "bf16", "m": 2048, "vocab": 128256, "hidden": 4096},
        # a matrix decoded for a consumer that wants f32
        {"name": "dequantize", "kind": "dequantize", "format": "q6_k", "n": 14336, "k": 4096},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5))))))


def _wide(rng, lo, hi, unit):
    """A size from lo to hi, a multiple of unit."""
    return unit * _log(rng, -(-lo // unit), hi // unit)


def draw(rng):
    largest = work(next(c for c in listed() if c["name"] == "prefill_layer"))
    while True:
        kind = rng.choice(["matmul"] * 5 + ["layer"] * 5 + ["moe"] * 2 + ["lm_head", "embedding", "dequantize"])
        form = rng.choice(["q4_k", "q4_k", "q6_k", "q5_k", "q8_0"])
        unit = 32 if form == "q8_0" else 256
        elem = rng.choice(["f32", "f32", "bf16", "bf16", "f16", "f32_bf16"])
        mix = rng.choice(["q4_k_m", "q4_k_m", "q5_k_m", "q6_k", "q8_0", "q4_k_s"])
        m = _log(rng, 1, 2048)
        if kind == "matmul":
            c = {"kind": kind, "format": form, "elem": elem, "m": m, "n": _log(rng, 512, 28672), "k": _wide(rng, 1024, 14336, unit)}
        elif kind == "layer":
            hidden = _wide(rng, 1024, 8192, 256)
            c = {"kind": kind, "mix": mix, "elem": "f32" if elem == "f32_bf16" else elem, "m": m, "hidden": hidden,
                 "kv": max(256, hidden // rng.choice([1, 4, 8]) // 32 * 32), "ffn": _wide(rng, 2 * hidden, 4 * hidden, 256)}
        elif kind == "moe":
            experts = rng.choice([8, 16, 32, 60, 64, 128])
            c = {"kind": kind, "mix": rng.choice(["q4_k_m", "q5_k_m", "q4_k_s", "q8_0"]), "elem": "f32" if elem == "f32_bf16" else elem,
                 "m": _log(rng, 1, 512), "hidden": _wide(rng, 1024, 4096, 256), "ffn": _wide(rng, 512, 2048, 256),
                 "experts": experts, "top_k": rng.choice([2, 4, 6, 8])}
        elif kind == "lm_head":
            c = {"kind": kind, "format": form, "n": _log(rng, 32000, 160000), "k": _wide(rng, 1024, 8192, 256),
                 "logits": form in ("q4_k", "q5_k") or rng.random() < 0.5}
        elif kind == "embedding":
            c = {"kind": kind, "format": form, "elem": "f32" if elem == "f32_bf16" else elem, "m": m,
                 "vocab": _log(rng, 32000, 160000), "hidden": _wide(rng, 1024, 8192, unit)}
        else:
            c = {"kind": kind, "format": form, "n": _log(rng, 1024, 16384), "k": _wide(rng, 1024, 8192, unit)}
        w = work(c)
        terms = 2 if c.get("elem") == "f32" else 1  # f32 activations carry two 16-bit terms
        if terms * w["flops"] <= largest["flops"] and w["bytes"] <= 2e9:
            return c


# ------------------------------------------------------------------ inputs
def _weights(gen, dtype, n, k):
    """``n`` rows of ``k`` elements as raw blocks.  The packed fields are uniform, the super-block scales such that the
    weights are centred on zero with a spread of some hundredths, as trained matrices have them."""
    rows = torch.randint(0, 256, (n * -(-k // block_size(dtype)), block_bytes(dtype)), dtype=torch.uint8, device="cuda", generator=gen)

    def scale(lo, hi):
        return torch.empty(rows.shape[0], 1, device="cuda").uniform_(lo, hi, generator=gen)

    if dtype in (Q4_K, Q5_K):
        d = scale(5e-5, 1.5e-4)
        mid = 7.5 if dtype == Q4_K else 15.5  # the middle of the quants: sub-block minima of about scale * mid
        rows[:, 0:2] = d.half().view(torch.uint8)
        rows[:, 2:4] = (d * mid * scale(0.9, 1.1)).half().view(torch.uint8)
    elif dtype == Q6_K:
        rows[:, 208:210] = scale(1e-5, 3e-5).half().view(torch.uint8)
    else:
        rows[:, 0:2] = scale(1e-4, 5e-4).half().view(torch.uint8)
    return rows.view(-1)


def _activations(gen, m, k, elem):
    """Normalised activations; a few channels are much larger than the rest, as in trained models."""
    x = torch.randn(m, k, device="cuda", generator=gen)
    x[:, torch.randint(0, k, (max(1, k // 512),), device="cuda", generator=gen)] *= 20
    return x.to(ELEMS[elem])


_hip = None


def _backend():
    """The program's one backend."""
    global _hip
    if _hip is None:
        _hip = B.HipBackend(0)
    return _hip


def prepare(case, seed):
    gen = torch.Generator("cuda")
    gen.manual_seed(seed)
    hip, kind, c = _backend(), case["kind"], case
    s = {"hip": hip, "case": c}

    def out(*shape, elem="f32"):
        return torch.zeros(*shape, device="cuda", dtype=ELEMS[elem])

    if kind == "matmul":
        s["w"] = _weights(gen, FORMATS[c["format"]], c["n"], c["k"])
        s["x"] = _activations(gen, c["m"], c["k"], c["elem"])
        s["y"] = out(c["m"], c["n"], elem=c["elem"])
        s["mode"] = B.ACT_BF16 if c["elem"] == "f32_bf16" else B.ACT_F32_SPLIT
    elif kind == "layer":
        main, down = MIXES[c["mix"]]
        m, h, kv, f, e = c["m"], c["hidden"], c["kv"], c["ffn"], c["elem"]
        s["x"] = _activations(gen, m, h, e)
        s["qkv"] = [(_weights(gen, main, n, h), s["x"], out(m, n, elem=e), main, m, n, h) for n in (h, kv, kv)]
        s["batch"] = hip.make_batch(s["qkv"])
        s["wo"], s["attn"], s["o"] = _weights(gen, main, h, h), _activations(gen, m, h, e), out(m, h, elem=e)
        s["gate"], s["up"], s["down"] = _weights(gen, main, f, h), _weights(gen, main, f, h), _weights(gen, down, h, f)
        s["mid"], s["y"] = _activations(gen, m, h, e), out(m, h, elem=e)
    elif kind == "moe":
        main, down = MIXES[c["mix"]]
        t, h, f, n, k = c["m"], c["hidden"], c["ffn"], c["experts"], c["top_k"]
        s["gate_up"], s["down"] = _weights(gen, main, n * 2 * f, h), _weights(gen, down, n * h, f)
        s["x"], s["y"] = _activations(gen, t, h, c["elem"]), out(t, h, elem=c["elem"])
        s["logits"] = torch.randn(t, n, device="cuda", generator=gen)
        s["expert"] = torch.zeros(t, k, dtype=torch.int32, device="cuda")
        s["weight"], s["len"] = out(t, k), torch.zeros(t, dtype=torch.int32, device="cuda")
    elif kind == "lm_head":
        s["w"] = _weights(gen, FORMATS[c["format"]], c["n"], c["k"])
        s["x"] = _activations(gen, 1, c["k"], "f32")
        s["logits"] = out(c["n"]) if c["logits"] else None
        s["token"], s["value"] = torch.zeros(1, dtype=torch.int32, device="cuda"), out(1)
    elif kind == "embedding":
        s["w"] = _weights(gen, FORMATS[c["format"]], c["vocab"], c["hidden"])
        s["ids"] = torch.randint(0, c["vocab"], (c["m"],), dtype=torch.int32, device="cuda", generator=gen)
        s["y"] = out(c["m"], c["hidden"], elem=c["elem"])
    else:
        s["w"] = _weights(gen, FORMATS[c["format"]], c["n"], c["k"])
        s["y"] = out(c["n"], c["k"])
    return s


def run(s):
    c, hip = s["case"], s["hip"]
    kind = c["kind"]
    if kind == "matmul":
        hip.quantized_matmul(s["w"], s["x"], s["y"], FORMATS[c["format"]], c["m"], c["n"], c["k"], s["mode"])
        return s["y"]
    if kind == "layer":
        main, down = MIXES[c["mix"]]
        hip.run_batch(s["batch"])
        hip.quantized_matmul(s["wo"], s["attn"], s["o"], main, c["m"], c["hidden"], c["hidden"])
        hip.ffn_swiglu(s["gate"], s["up"], main, s["down"], down, s["mid"], s["y"], c["m"], c["hidden"], c["ffn"])
        q, k, v = (e[2] for e in s["qkv"])
        return {"q": q, "k": k, "v": v, "o": s["o"], "y": s["y"]}
    if kind == "moe":
        main, down = MIXES[c["mix"]]
        # every routed pair is computed: an expert takes as many tokens as choose it
        hip.moe_route(s["logits"], c["top_k"], s["expert"], s["weight"], s["len"], capacity_factor=float(c["experts"]))
        hip.moe_matvec(s["gate_up"], main, s["down"], down, s["x"], s["y"], c["hidden"], c["ffn"], c["experts"],
                       s["expert"], s["weight"], s["len"])
        return {"expert": s["expert"], "weight": s["weight"], "len": s["len"], "y": s["y"]}
    if kind == "lm_head":
        hip.lm_head_argmax(s["w"], s["x"], FORMATS[c["format"]], c["n"], c["k"], s["token"], logits=s["logits"], value=s["value"])
        got = {"token": s["token"], "value": s["value"]}
        return got if s["logits"] is None else dict(got, logits=s["logits"])
    if kind == "embedding":
        hip.quant_gather(s["w"], FORMATS[c["format"]], c["vocab"], c["hidden"], s["ids"], s["y"])
        return s["y"]
    hip.dequantize(s["w"], s["y"], FORMATS[c["format"]])
    return s["y"]


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    c, kind = case, case["kind"]
    e = 4 if c.get("elem", "f32").startswith("f32") else 2
    if kind in ("matmul", "lm_head"):
        m, n, k, dt = c.get("m", 1), c["n"], c["k"], FORMATS[c["format"]]
        y = m * n * e if kind == "matmul" else 8 + (4 * n if c["logits"] else 0)
        return {"bytes": n * row_bytes(dt, k) + m * k * e + y, "flops": 2 * m * n * k}
    if kind == "layer":
        m, h, kv, f = c["m"], c["hidden"], c["kv"], c["ffn"]
        main, down = MIXES[c["mix"]]
        weights = (2 * h + 2 * kv + 2 * f) * row_bytes(main, h) + h * row_bytes(down, f)
        return {"bytes": weights + m * e * (3 * h + h + 2 * kv + 2 * h), "flops": 2 * m * (2 * h * h + 2 * kv * h + 3 * f * h)}
    if kind == "moe":
        t, h, f, n, k = c["m"], c["hidden"], c["ffn"], c["experts"], c["top_k"]
        main, down = MIXES[c["mix"]]
        hit = n * (1 - (1 - k / n) ** t)  # experts that somebody chooses, for independent choices
        return {"bytes": hit * (2 * f * row_bytes(main, h) + h * row_bytes(down, f)) + 2 * t * h * e + t * n * 4 + t * (8 * k + 4),
                "flops": 2 * t * k * 3 * h * f}
    if kind == "embedding":
        return {"bytes": c["m"] * (row_bytes(FORMATS[c["format"]], c["hidden"]) + 4 + c["hidden"] * e), "flops": c["m"] * c["hidden"]}
    return {"bytes": c["n"] * (row_bytes(FORMATS[c["format"]], c["k"]) + 4 * c["k"]), "flops": 2 * c["n"] * c["k"]}


def tolerance(case):
    """Sums of f32 products from activations of at least 22 bits, rounded once to the element type.  Decoded values
    have one right answer."""
    if case["kind"] in ("embedding", "dequantize"):
        return "exact"
    elem = case.get("elem", "f32")
    return {"rel": {"f32": 1e-5, "f32_bf16": 1e-5, "f16": 1e-3, "bf16": 4e-3}[elem]}
