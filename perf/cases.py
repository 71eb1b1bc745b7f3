"""Timed work of the per-token inference path, as a program that uses this
package calls it: attention over plain tensors and over KV-cache views, the
MLP block of one decoder layer, the dense head, and whole forwards of the
native decoder engine.

Geometries are the package's own configurations (``LLAMA3_8B``,
``LLAMA32_3B``) and the small fp32 attention of the benchmark (8 query heads,
2 KV heads, head size 64).  Weights and activations are random-init, as in
``bench.py``.
"""
from __future__ import annotations

import math
from dataclasses import replace

import torch

from lokahi_amd import ops
from lokahi_amd.llama import (LLAMA3_8B, LLAMA32_3B, DecoderEngine, HipLlamaForCausalLM,
                              random_weights)

MODELS = {"8b": LLAMA3_8B, "3b": LLAMA32_3B}
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
DEV = "cuda"


# ------------------------------------------------------------------- cases
def _attn(name, dtype, batch, hq, hkv, d, lq, past, cached):
    """Causal attention of lq new tokens per row after ``past`` earlier ones;
    ``cached``: K and V are views into a longer KV cache and the query
    positions are given, as the decoder layer passes them."""
    return {"name": name, "kind": "attention", "dtype": dtype, "batch": batch, "hq": hq,
            "hkv": hkv, "d": d, "lq": lq, "past": past, "cached": cached}


def _mlp(name, model, rows, layout):
    """RMSNorm, gate/up, SiLU * up, down; ``layout``: over the load-time
    decode layout (1..8 rows)."""
    return {"name": name, "kind": "mlp", "model": model, "rows": rows, "layout": layout}


def _head(name, model, rows):
    return {"name": name, "kind": "head", "model": model, "rows": rows}


def _model(name, model, batch, prompt, steps):
    return {"name": name, "kind": "model", "model": model, "batch": batch, "prompt": prompt,
            "steps": steps}


def listed():
    return [
        # the chunked fp32 attention the reference's tests and small models run
        _attn("attn_f32_512", "f32", 1, 8, 2, 64, 512, 0, False),
        # an ordinary prompt through one layer, a length no tile divides
        _attn("attn_prompt_1500", "bf16", 1, 24, 8, 128, 1500, 0, False),
        # a long document
        _attn("attn_prompt_8192", "bf16", 1, 32, 8, 128, 8192, 0, False),
        # the next turn of a chat: a short message over a long cached history
        _attn("attn_extend_100", "bf16", 1, 32, 8, 128, 100, 4000, True),
        # one decode step of one sequence
        _attn("attn_decode_2k", "bf16", 1, 32, 8, 128, 1, 2048, True),
        # one decode step of a served batch with long contexts
        _attn("attn_decode_16x8k", "bf16", 16, 32, 8, 128, 1, 8192, True),
        # one decode token through the MLP (the weights laid out at load time)
        _mlp("mlp_decode", "8b", 1, True),
        # a very short prompt, or the candidates of speculative decoding
        _mlp("mlp_24", "3b", 24, False),
        # an ordinary prompt
        _mlp("mlp_200", "8b", 200, False),
        # a long document
        _mlp("mlp_8192", "8b", 8192, False),
        # logits of every position of a prompt (scoring; logits="all")
        _head("head_300", "8b", 300),
        # a small batch of prompts, then a few greedy decode steps
        _model("model_4x100", "3b", 4, 100, 8),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["prompt", "prompt", "extend", "extend", "decode", "mlp", "mlp", "mlp",
                       "head", "model"])
    if kind in ("prompt", "extend", "decode"):
        if rng.random() < 0.25:  # the fp32 flow of the small configuration
            dtype, hq, hkv, d, most = "f32", 8, 2, 64, 2048
        else:
            dtype, hq, hkv, d, most = "bf16", rng.choice([24, 32]), 8, 128, 8192
        if kind == "prompt":
            batch = rng.choice([1, 1, 1, 2, 4])
            lq, past = _log(rng, 16, most // batch), 0
        elif kind == "extend":
            batch = rng.choice([1, 1, 1, 2, 4])
            lq, past = _log(rng, 2, 512), _log(rng, 64, most)
        else:
            batch = _log(rng, 1, 16)
            lq, past = 1, _log(rng, 64, most)
        case = _attn("", dtype, batch, hq, hkv, d, lq, past, kind != "prompt")
    elif kind == "mlp":
        rows = _log(rng, 1, 8192)
        case = _mlp("", rng.choice(["8b", "3b"]), rows, rows <= 8 and rng.random() < 0.5)
    elif kind == "head":
        case = _head("", rng.choice(["8b", "3b"]), _log(rng, 1, 512))
    else:
        batch = rng.choice([1, 2, 3, 4, 6, 8])
        case = _model("", "3b", batch, _log(rng, 2, 400 // batch), rng.randint(1, 8))
    del case["name"]
    return case


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(gen, *shape, std=1.0, dtype=torch.bfloat16):
    return (torch.randn(shape, generator=gen, device=DEV) * std).to(dtype)


def _q4(gen, n, k):
    return ops.quantize(torch.randn((n, k), generator=gen, device=DEV) * 0.02)


def prepare(case, seed):
    gen = _gen(seed)
    kind = case["kind"]
    if kind == "attention":
        b, hq, hkv, d = case["batch"], case["hq"], case["hkv"], case["d"]
        lq, lk, dt = case["lq"], case["past"] + case["lq"], DTYPES[case["dtype"]]
        s = {"kind": kind, "q": _randn(gen, b, hq, lq, d, dtype=dt), "pos": None, "strides": None}
        # a cache has room for the tokens still to come
        lmax = (lk + 64 + 255) // 256 * 256 if case["cached"] else lk
        k, v = (_randn(gen, b, hkv, lmax, d, dtype=dt) for _ in range(2))
        if case["cached"]:
            s["pos"] = torch.arange(case["past"], lk, dtype=torch.int32, device=DEV)
            s["strides"] = (hkv * lmax * d, lmax * d)
            k, v = k[:, :, :lk], v[:, :, :lk]
        s["k"], s["v"] = k, v
        return s
    cfg = MODELS[case["model"]]
    h, f = cfg.hidden_size, cfg.intermediate_size
    if kind == "mlp":
        s = {"kind": kind, "x": _randn(gen, 1, case["rows"], h), "eps": cfg.rms_norm_eps,
             "norm": _randn(gen, h, std=0.1) + 1, "gate": _q4(gen, f, h), "up": _q4(gen, f, h),
             "down": _q4(gen, h, f), "gate_up_layout": None, "down_layout": None}
        if case["layout"]:
            s["gate_up_layout"] = ops.Q4Layout([s["gate"], s["up"]])
            s["down_layout"] = ops.Q4Layout([s["down"]])
        return s
    if kind == "head":
        return {"kind": kind, "x": _randn(gen, 1, case["rows"], h),
                "head": _randn(gen, cfg.vocab_size, h, std=0.02)}
    # Small weights and a unit-scale embedding keep the map from rounding
    # errors to logits tame: with larger random weights a random-init model
    # of this depth is chaotic, which no trained one is.
    cfg = replace(cfg)
    w = random_weights(cfg, seed, std=0.003)
    w["embed_tokens"] = _randn(gen, cfg.vocab_size, h)
    b, l, steps = case["batch"], case["prompt"], case["steps"]
    model = HipLlamaForCausalLM(cfg, w)
    cache = model.new_cache(b, l + steps)
    engine = DecoderEngine(model, cache, max_batch=b, max_tokens=b * l)
    ids = torch.randint(0, cfg.vocab_size, (b, l + steps), generator=gen, device=DEV,
                        dtype=torch.int32)
    return {"kind": kind, "engine": engine, "cache": cache, "prompt": ids[:, :l].contiguous(),
            "next": [ids[:, l + i:l + i + 1].contiguous() for i in range(steps)]}


# --------------------------------------------------------------------- run
def run(s):
    kind = s["kind"]
    if kind == "attention":
        return ops.attention(s["q"], s["k"], s["v"], query_positions=s["pos"],
                             kv_strides=s["strides"])
    if kind == "mlp":
        xn = ops.rmsnorm(s["x"], s["norm"], s["eps"])
        if s["gate_up_layout"] is not None:
            gate, up = s["gate_up_layout"](xn)
            return s["down_layout"](ops.silu_mul(gate, up))[0]
        gate, up = ops.linear_multi(xn, [s["gate"], s["up"]])
        return ops.linear(ops.silu_mul(gate, up), *s["down"])
    if kind == "head":
        return ops.linear(s["x"], s["head"], None, None, out_dtype=torch.float32)
    s["cache"].clear()
    logits = [s["engine"].forward(s["prompt"])]
    for ids in s["next"]:
        logits.append(s["engine"].forward(ids))
    return logits


# -------------------------------------------------------------------- work
def _q4_bytes(n, k):
    return n * k // 2 + 4 * n * (k // 64)


def _visible(case):
    """(query, key) pairs of one head under the causal mask."""
    lq, past = case["lq"], case["past"]
    return lq * past + lq * (lq + 1) // 2


def work(case):
    kind = case["kind"]
    if kind == "attention":
        size = 2 if case["dtype"] == "bf16" else 4
        b, hq, hkv, d, lq = (case[n] for n in ("batch", "hq", "hkv", "d", "lq"))
        lk = case["past"] + lq
        return {"bytes": size * d * b * (2 * hq * lq + 2 * hkv * lk),
                "flops": 4 * d * b * hq * _visible(case)}
    cfg = MODELS[case["model"]]
    h, f, v = cfg.hidden_size, cfg.intermediate_size, cfg.vocab_size
    if kind == "mlp":
        m = case["rows"]
        return {"bytes": 3 * _q4_bytes(f, h) + 2 * 2 * m * h + 2 * h, "flops": 2 * m * 3 * f * h}
    if kind == "head":
        m = case["rows"]
        return {"bytes": 2 * v * h + 2 * m * h + 4 * m * v, "flops": 2 * m * v * h}
    b, l, steps = case["batch"], case["prompt"], case["steps"]
    qw, kw = cfg.num_attention_heads * cfg.head_dim, cfg.num_key_value_heads * cfg.head_dim
    n = cfg.num_hidden_layers
    weights = n * (_q4_bytes(qw + 2 * kw, h) + _q4_bytes(h, qw) + 3 * _q4_bytes(f, h)) + 2 * v * h
    params = n * ((qw + 2 * kw) * h + qw * h + 3 * f * h)
    kv_read = sum(l + i + 1 for i in range(steps)) + l
    pairs = l * (l + 1) // 2 + sum(l + i + 1 for i in range(steps))
    return {"bytes": (1 + steps) * (weights + 4 * b * v) + 2 * 2 * n * kw * b * kv_read,
            "flops": 2 * params * b * (l + steps) + 2 * v * h * b * (1 + steps)
            + 4 * qw * n * b * pairs}


def tolerance(case):
    kind = case["kind"]
    if kind == "attention":
        return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 1e-5}
    if kind == "mlp":
        return {"rel": 1e-2}
    if kind == "head":
        return {"rel": 1e-5}
    return {"rel": 5e-3}


# ------------------------------------------------------------------- exact
def _dequant(t, n, k):
    w, s, b = t
    words = w.view(torch.int32)
    codes = torch.stack([(words >> (4 * i)) & 15 for i in range(8)], dim=-1).reshape(n, k // 64, 64)
    return (codes * s.double()[..., None] + b.double()[..., None]).reshape(n, k)


def exact(case, seed):
    kind = case["kind"]
    if kind == "model":
        return None
    s = prepare(case, seed)
    if kind == "attention":
        hq, hkv, d, lq, past = (case[n] for n in ("hq", "hkv", "d", "lq", "past"))
        out = torch.empty(s["q"].shape, dtype=torch.float64, device=DEV)
        key = torch.arange(past + lq, device=DEV)
        for b in range(case["batch"]):
            for i in range(hq):
                k, v = (s[n][b, i // (hq // hkv)].double() for n in "kv")
                for r in range(0, lq, 2048):
                    sc = s["q"][b, i, r:r + 2048].double() @ k.T / math.sqrt(d)
                    row = torch.arange(past + r, past + r + sc.shape[0], device=DEV)
                    sc.masked_fill_(key[None, :] > row[:, None], -math.inf)
                    out[b, i, r:r + 2048] = torch.softmax(sc, dim=-1) @ v
        return out
    x = s["x"].double()
    if kind == "head":
        y = torch.empty((1, case["rows"], s["head"].shape[0]), dtype=torch.float64, device=DEV)
        for c in range(0, s["head"].shape[0], 16384):
            y[..., c:c + 16384] = x @ s["head"][c:c + 16384].double().T
        return y
    cfg = MODELS[case["model"]]
    h, f = cfg.hidden_size, cfg.intermediate_size
    xn = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + s["eps"]) * s["norm"].double()
    gate = xn @ _dequant(s["gate"], f, h).T
    act = gate * torch.sigmoid(gate) * (xn @ _dequant(s["up"], f, h).T)
    del gate
    return act @ _dequant(s["down"], h, f).T
