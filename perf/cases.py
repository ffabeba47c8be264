"""The performance cases of the MI355X quantized-matmul library.

Each listed case is work that a program using this library hands it through its
public Python entry points (sllm_qmm): the matmuls of a decode step and of a
prompt, the FFN block, the output head, the attention section, the
host-buffer calls, and whole calls of a decoder. Sizes are those of this
repository's own configurations (SmolLM2-135M / 1.7B and Llama-3-8B shapes) or
generic. `draw` gives more cases of the same ranges.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "scriptling-llm-lib_amd"))

import sllm_qmm as sq  # noqa: E402

EPS = 1e-5
Q4_0, Q4_1, Q5_0, Q8_0, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K = 2, 3, 6, 8, 10, 11, 12, 13, 14
# GGUF type: elements and bytes of a block, bytes per 32 weights on the device
BLOCK = {Q4_0: (32, 18, 18.0), Q4_1: (32, 20, 20.0), Q5_0: (32, 22, 22.0), Q8_0: (32, 34, 34.0),
         Q2_K: (256, 84, 10.5), Q3_K: (256, 110, 14.5), Q4_K: (256, 144, 20.0), Q5_K: (256, 176, 26.0),
         Q6_K: (256, 210, 34.0)}


def listed():
    return [
        # the smallest call: one linear layer of SmolLM2-135M for one token (latency)
        {"name": "linear_q8_135m", "op": "matmul", "type": Q8_0, "rows": 1536, "cols": 576, "m": 1},
        # one token's FFN block of SmolLM2-1.7B in Q4_0
        {"name": "ffn_q4_0_1p7b", "op": "ffn", "gate": Q4_0, "down": Q4_0, "hidden": 2048, "inner": 8192, "m": 1},
        # one token through a Llama-3-8B Q4_K_M layer, 1000 tokens into the context
        {"name": "layer_q4km_8b", "op": "layer", "type": Q4_K, "down": Q6_K, "hidden": 4096, "inner": 14336,
         "heads": 32, "kv_heads": 8, "dk": 128, "pos": 1000, "m": 1},
        # final norm, output head and greedy token of Llama-3-8B
        {"name": "head_q6k_8b", "op": "head", "type": Q6_K, "rows": 128256, "cols": 4096, "m": 1},
        # one token's attention at the end of an 8K context (Llama-3-8B heads)
        {"name": "attn_decode_8b_8k", "op": "attn", "heads": 32, "kv_heads": 8, "dk": 128, "pos": 8000, "m": 1},
        # a 1024-token prompt's attention in one layer (Llama-3-8B heads)
        {"name": "attn_prompt_8b_1k", "op": "attn", "heads": 32, "kv_heads": 8, "dk": 128, "pos": 0, "m": 1024},
        # a short prompt's q / k / v projections in Q5_K
        {"name": "qkv_q5k_prompt30", "op": "qkv", "type": Q5_K, "hidden": 4096, "kv": 1024, "m": 30},
        # a prompt's FFN block, Llama-3-8B Q4_K_M, 512 tokens
        {"name": "ffn_q4km_prompt512", "op": "ffn", "gate": Q4_K, "down": Q6_K, "hidden": 4096, "inner": 14336,
         "m": 512},
        # a Q5_0 FFN matmul of a prompt whose length is no multiple of anything
        {"name": "linear_q5_0_prompt100", "op": "matmul", "type": Q5_0, "rows": 14336, "cols": 4096, "m": 100},
        # a low-bit model's FFN block on a 64-token prompt
        {"name": "ffn_q3k_prompt64", "op": "ffn", "gate": Q3_K, "down": Q3_K, "hidden": 4096, "inner": 14336,
         "m": 64},
        # the drop-in host-buffer call of one FFN matmul (SmolLM2-1.7B, Q4_1)
        {"name": "host_q4_1_1p7b", "op": "host", "type": Q4_1, "rows": 8192, "cols": 2048, "m": 1},
        # a whole call: a 200-token prompt through a SmolLM2-1.7B-wide decoder layer and the head
        {"name": "model_q4km_prompt200", "op": "model", "type": Q4_K, "down": Q6_K, "hidden": 2048, "inner": 8192,
         "heads": 32, "kv_heads": 32, "dk": 64, "rows": 49152, "layers": 1, "pos": 0, "m": 200},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["matmul", "matmul", "matmul", "ffn", "ffn", "qkv", "qkv", "attn", "attn", "attn", "head", "host"])
    heads = [(32, 8, 128), (32, 32, 64), (9, 3, 64), (32, 4, 128), (16, 16, 80), (40, 8, 128), (8, 1, 256)]
    if op == "matmul":
        t = rng.choice([Q8_0, Q4_0, Q4_1, Q5_0, Q5_K, Q4_K, Q6_K, Q2_K, Q3_K])
        step = 256 if BLOCK[t][0] == 256 else 32
        return {"op": op, "type": t, "rows": _log(rng, 64, 14336), "cols": step * _log(rng, 512 // step, 14336 // step),
                "m": _log(rng, 1, 512)}
    if op == "ffn":
        g, d = rng.choice([(Q4_K, Q6_K), (Q4_K, Q4_K), (Q5_K, Q6_K), (Q8_0, Q8_0), (Q4_0, Q4_0), (Q4_1, Q4_1),
                           (Q5_0, Q5_0), (Q2_K, Q3_K), (Q3_K, Q5_K)])
        return {"op": op, "gate": g, "down": d, "hidden": 256 * rng.randint(2, 16), "inner": 256 * _log(rng, 5, 56),
                "m": _log(rng, 1, 512)}
    if op == "qkv":
        return {"op": op, "type": rng.choice([Q4_K, Q5_K, Q6_K, Q8_0, Q4_0, Q5_0, Q3_K]), "hidden": 256 * rng.randint(2, 16),
                "kv": 64 * rng.randint(2, 32), "m": _log(rng, 1, 512)}
    if op == "attn":
        h, kv, dk = rng.choice(heads)
        if rng.random() < 0.4:
            return {"op": op, "heads": h, "kv_heads": kv, "dk": dk, "pos": _log(rng, 16, 8000), "m": 1}
        return {"op": op, "heads": h, "kv_heads": kv, "dk": dk, "pos": rng.choice([0, 0, rng.randint(1, 300)]),
                "m": _log(rng, 2, 700)}
    if op == "head":
        return {"op": op, "type": rng.choice([Q6_K, Q8_0, Q4_K]), "rows": _log(rng, 8000, 128256),
                "cols": 256 * rng.randint(2, 16), "m": 1}
    return {"op": op, "type": rng.choice([Q4_0, Q4_1, Q8_0, Q4_K, Q6_K]), "rows": _log(rng, 512, 14336),
            "cols": 256 * rng.randint(2, 16), "m": rng.choice([1, 1, 1, _log(rng, 2, 64)])}


# ----------------------------------------------------------------- inputs ----

def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + salt * 7919 + 17) & 0x7FFFFFFF)


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * std


def _put16(raw, off, v):
    raw[:, off:off + 2] = v.to(torch.float16).view(torch.uint8).reshape(-1, 2)


def _raw(t, rows, cols, g):
    """GGUF blocks of a weight: random codes and sub-scales, block scales that
    give weights of about the size a trained layer holds, centred on zero."""
    elems, size, _ = BLOCK[t]
    nb = rows * cols // elems
    raw = torch.randint(0, 256, (nb, size), generator=g, device="cuda", dtype=torch.uint8)
    u = torch.rand(nb, generator=g, device="cuda") + 0.5
    if t == Q8_0:
        _put16(raw, 0, u * 3e-4)
    elif t == Q4_0:
        _put16(raw, 0, u * 4e-3)
    elif t == Q4_1:
        _put16(raw, 0, u * 4e-3)
        _put16(raw, 2, u * -3e-2)
    elif t == Q5_0:
        _put16(raw, 0, u * 2e-3)
    elif t == Q2_K:
        _put16(raw, 80, u * 2e-3)
        _put16(raw, 82, u * 3e-3)
    elif t == Q3_K:
        _put16(raw, 108, u * 5e-4)
    elif t == Q4_K:
        _put16(raw, 0, u * 1.5e-4)
        _put16(raw, 2, u * 1.1e-3)
    elif t == Q5_K:
        _put16(raw, 0, u * 1.3e-4)
        _put16(raw, 2, u * 2e-3)
    elif t == Q6_K:
        _put16(raw, 208, u * 1.5e-4)
        # small sub-scales, so that the block scale stays a normal f16
        sc = torch.randint(-24, 25, (nb, 16), generator=g, device="cuda", dtype=torch.int8)
        raw[:, 192:208] = sc.view(torch.uint8)
    return raw


def _weight(t, rows, cols, g):
    return sq.load_weight_f32_direct(t, _raw(t, rows, cols, g).reshape(-1).cpu().numpy(), rows, cols)


def _freqs(dk):
    return torch.tensor([1.0 / math.pow(10000.0, 2.0 * i / dk) for i in range(dk // 2)], dtype=torch.float32).cuda()


class _Mem:
    """Device memory of the library's as a tensor's storage; it keeps its owner alive."""

    def __init__(self, ptr, shape, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (ptr, False), "version": 2}


def _cache(c, seed, layers):
    """A KV cache holding c["pos"] rows per layer, and views of its K and V."""
    kv, pos = c["kv_heads"], c["pos"]
    cap = pos + c["m"] + 8
    cache = sq.KVCache(layers, kv, c["dk"], cap)
    views = []
    g = _gen(seed, 90)
    for layer in range(layers):
        k, v = (torch.as_tensor(_Mem(p, (kv, cap, c["dk"]), cache), device="cuda") for p in cache.data(layer))
        k[:, :pos] = _normal(g, kv, pos, c["dk"], std=0.7)
        v[:, :pos] = _normal(g, kv, pos, c["dk"])
        views.append((k, v))
    return cache, views


def _attn_params(c):
    f = _freqs(c["dk"])
    p = sq.AttnParams(n_heads=c["heads"], n_kv_heads=c["kv_heads"], d_k=c["dk"], rope_half_dim=c["dk"] // 2,
                      rope_freqs=f.data_ptr(), norm_eps=EPS)
    return p, f


def _qkv_input(c, seed):
    g = _gen(seed, 1)
    n, kvn = c["heads"] * c["dk"], c["kv_heads"] * c["dk"]
    return _normal(g, c["m"], n), _normal(g, c["m"], kvn, std=0.7), _normal(g, c["m"], kvn)


def _x(c, cols, seed):
    return _normal(_gen(seed, 2), c["m"], cols)


def _norm_w(cols, seed):
    return 0.4 + _normal(_gen(seed, 3), cols, std=0.04)


def _empty(*shape):
    return torch.empty(*shape, device="cuda")


def _layer_state(c, seed, salt):
    h, f, n, kvn = c["hidden"], c["inner"], c["heads"] * c["dk"], c["kv_heads"] * c["dk"]
    t, d = c["type"], c["down"]
    ws = [_weight(a, r, k, _gen(seed, salt + i)) for i, (a, r, k) in enumerate(
        [(t, n, h), (t, kvn, h), (d, kvn, h), (t, h, n), (t, f, h), (t, f, h), (d, h, f)])]
    return {"w": ws, "n1": 0.4 + _normal(_gen(seed, salt + 8), h, std=0.04),
            "n2": 0.4 + _normal(_gen(seed, salt + 9), h, std=0.04)}


def prepare(c, seed):
    torch.cuda.set_device(0)
    s = {"c": c, "stream": torch.cuda.current_stream().cuda_stream}
    op, m = c["op"], c["m"]
    if op in ("matmul", "host", "head"):
        s["w"] = _weight(c["type"], c["rows"], c["cols"], _gen(seed, 10))
        s["x"] = _x(c, c["cols"], seed)
        if op == "host":
            s["x"] = s["x"].cpu().numpy().reshape(-1)
        else:
            s["y"] = _empty(m, c["rows"])
        if op == "head":
            s["n"] = _norm_w(c["cols"], seed)
            s["tok"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    elif op == "qkv":
        shapes = [c["hidden"], c["kv"], c["kv"]]
        s["w"] = [_weight(c["type"], r, c["hidden"], _gen(seed, 10 + i)) for i, r in enumerate(shapes)]
        s["x"], s["n"] = _x(c, c["hidden"], seed), _norm_w(c["hidden"], seed)
        s["y"] = [_empty(m, r) for r in shapes]
    elif op == "ffn":
        h, f = c["hidden"], c["inner"]
        s["gate"], s["up"] = (_weight(c["gate"], f, h, _gen(seed, 10 + i)) for i in range(2))
        s["down"] = _weight(c["down"], h, f, _gen(seed, 12))
        s["x"], s["n"], s["h"] = _x(c, h, seed), _norm_w(h, seed), _empty(m, f)
    elif op == "attn":
        s["kv"], s["views"] = _cache(c, seed, 1)
        s["p"], s["f"] = _attn_params(c)
        s["q"], s["k"], s["v"] = _qkv_input(c, seed)
        s["y"] = _empty(m, c["heads"] * c["dk"])
    else:
        layers = c.get("layers", 1)
        s["kv"], s["views"] = _cache(c, seed, layers)
        s["p"], s["f"] = _attn_params(c)
        s["layers"] = [_layer_state(c, seed, 20 * (i + 1)) for i in range(layers)]
        s["x"] = _x(c, c["hidden"], seed)
        n, kvn = c["heads"] * c["dk"], c["kv_heads"] * c["dk"]
        s["q"], s["k"], s["v"], s["a"] = _empty(m, n), _empty(m, kvn), _empty(m, kvn), _empty(m, n)
        s["h"] = _empty(m, c["inner"])
        if op == "model":
            s["w"], s["n"] = _weight(Q6_K, c["rows"], c["hidden"], _gen(seed, 10)), _norm_w(c["hidden"], seed)
            s["y"], s["tok"] = _empty(1, c["rows"]), torch.zeros(1, dtype=torch.int32, device="cuda")
    return s


# -------------------------------------------------------------------- run ----

def _new_rows(s, layer):
    c = s["c"]
    k, v = s["views"][layer]
    return k[:, c["pos"]:c["pos"] + c["m"]], v[:, c["pos"]:c["pos"] + c["m"]]


def _forward(s, layer, x):
    """forwardBlock: x is the residual stream, updated in place."""
    c, st, L = s["c"], s["stream"], s["layers"][layer]
    m, hid = c["m"], c["hidden"]
    wq, wk, wv, wo, wg, wu, wd = L["w"]
    q, k, v, a, h = s["q"], s["k"], s["v"], s["a"], s["h"]
    sq.rmsnorm_matmul_multi_dev([wq, wk, wv], x.data_ptr(), L["n1"].data_ptr(), EPS, m, hid,
                                [q.data_ptr(), k.data_ptr(), v.data_ptr()], st)
    sq.attention_dev(s["kv"], layer, s["p"], q.data_ptr(), k.data_ptr(), v.data_ptr(), m, c["pos"], a.data_ptr(), st)
    sq.matmul_add_dev(wo, a.data_ptr(), m, a.shape[1], x.data_ptr(), st)
    sq.rmsnorm_matmul_swiglu_dev(wg, wu, x.data_ptr(), L["n2"].data_ptr(), EPS, m, hid, h.data_ptr(), st)
    sq.matmul_add_dev(wd, h.data_ptr(), m, h.shape[1], x.data_ptr(), st)


def run(s):
    c, st = s["c"], s["stream"]
    op, m = c["op"], c["m"]
    if op == "matmul":
        sq.matmul_dev(s["w"], s["x"].data_ptr(), m, c["cols"], s["y"].data_ptr(), st)
        return s["y"]
    if op == "host":
        return sq.model_matmul_quant_into_f32(s["w"], s["x"], m, c["cols"])[0]
    if op == "head":
        sq.rmsnorm_matmul_argmax_dev(s["w"], s["x"].data_ptr(), s["n"].data_ptr(), EPS, s["tok"].data_ptr(),
                                     s["y"].data_ptr(), st)
        return s["y"], s["tok"]
    if op == "qkv":
        sq.rmsnorm_matmul_multi_dev(s["w"], s["x"].data_ptr(), s["n"].data_ptr(), EPS, m, c["hidden"],
                                    [y.data_ptr() for y in s["y"]], st)
        return s["y"]
    if op == "ffn":
        y = s["x"].clone()  # the residual stream, as the layer before left it
        sq.rmsnorm_matmul_swiglu_dev(s["gate"], s["up"], y.data_ptr(), s["n"].data_ptr(), EPS, m, c["hidden"],
                                     s["h"].data_ptr(), st)
        sq.matmul_add_dev(s["down"], s["h"].data_ptr(), m, c["inner"], y.data_ptr(), st)
        return s["h"], y
    s["kv"].set_length(c["pos"])
    if op == "attn":
        sq.attention_dev(s["kv"], 0, s["p"], s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), m, c["pos"],
                         s["y"].data_ptr(), st)
        return (s["y"], *_new_rows(s, 0))
    x = s["x"].clone()
    for layer in range(len(s["layers"])):
        _forward(s, layer, x)
    if op == "layer":
        return (x, s["a"], s["h"], *_new_rows(s, 0))
    sq.rmsnorm_matmul_argmax_dev(s["w"], x[m - 1:].data_ptr(), s["n"].data_ptr(), EPS, s["tok"].data_ptr(),
                                 s["y"].data_ptr(), st)
    # the logits say it all: an order of sums can move two close ones past each other
    return s["y"], x


# ------------------------------------------------------------------- work ----

def _mm(t, rows, cols, m):
    return rows * cols / 32 * BLOCK[t][2] + 4 * m * (rows + cols), 2 * m * rows * cols


def _at(c):
    n, kvn = c["heads"] * c["dk"], c["kv_heads"] * c["dk"]
    pairs = c["m"] * c["pos"] + c["m"] * (c["m"] + 1) // 2
    # q, k, v in, out and the new rows out, the held rows in
    return 4 * (c["m"] * (2 * n + 4 * kvn) + 2 * c["pos"] * kvn), 4 * pairs * n


def work(c):
    op, m = c["op"], c["m"]
    if op in ("matmul", "host", "head"):
        parts = [_mm(c["type"], c["rows"], c["cols"], m)]
    elif op == "qkv":
        parts = [_mm(c["type"], r, c["hidden"], m) for r in (c["hidden"], c["kv"], c["kv"])]
    elif op == "attn":
        parts = [_at(c)]
    elif op == "ffn":
        parts = [_mm(c["gate"], c["inner"], c["hidden"], m)] * 2 + [_mm(c["down"], c["hidden"], c["inner"], m)]
    else:
        h, f, n, kvn, t, d = c["hidden"], c["inner"], c["heads"] * c["dk"], c["kv_heads"] * c["dk"], c["type"], c["down"]
        one = [_mm(a, r, k, m) for a, r, k in ((t, n, h), (t, kvn, h), (d, kvn, h), (t, h, n), (t, f, h), (t, f, h), (d, h, f))]
        parts = (one + [_at(c)]) * c.get("layers", 1)
        if op == "model":
            parts.append(_mm(Q6_K, c["rows"], h, 1))
    return {"bytes": float(sum(p[0] for p in parts)), "flops": float(sum(p[1] for p in parts))}


def tolerance(c):
    """One quantization: the sums' order only, over up to 14336 fp32 terms.
    ffn / layer / model quantize computed activations again: a value that moves
    by its last bit across a truncation boundary moves one int8 code, in
    the block after it and in all that follow."""
    op = c["op"]
    if op in ("matmul", "host"):
        return {"rel": 2e-6, "max": 2e-5}
    if op in ("qkv", "head"):
        # the fused RMSNorm's last bit can move single codes of its rows
        return {"rel": 2e-3, "max": 0.02, "differ": 0.0}
    if op == "attn":
        return {"rel": 2e-6, "max": 1e-4}
    if op == "ffn":
        return {"rel": 0.01, "max": 0.1}
    return {"rel": 0.03, "max": 0.3, "differ": 0.0}


# ------------------------------------------------------------------ exact ----

def _h(raw, off):
    return raw[:, off:off + 2].contiguous().view(torch.float16).double()


def _trunc16(v):
    """float64 -> the f16 the remaps write: mantissa truncated, below the normal range zero."""
    m, e = torch.frexp(v)  # v = m 2^e, 0.5 <= |m| < 1
    out = torch.ldexp(torch.trunc(m * 2048.0), e - 11)
    return torch.where(v.abs() < 2.0 ** -14, torch.zeros_like(v), out)


def _sc_min(q):
    """getScaleMinK4: 12 bytes -> 8 six-bit scales and mins."""
    q = q.to(torch.int32)
    lo, mid, hi = q[:, 0:4], q[:, 4:8], q[:, 8:12]
    sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1)
    mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1)
    return sc.double(), mn.double()


def _nibbles(b):
    return torch.cat([b & 15, b >> 4], -1).double()


def _dense(t, raw):
    """The weights in fp64 as the library's path defines them: Q4_K / Q5_K after their Q4_1 remap,
    Q6_K after its Q8_0 one, Q2_K / Q3_K as float32 values. raw: (blocks, bytes)."""
    n = raw.shape[0]
    if t == Q8_0:
        return _h(raw, 0) * raw[:, 2:].contiguous().view(torch.int8).double()
    if t == Q4_0:
        return _h(raw, 0) * (_nibbles(raw[:, 2:]) - 8)
    if t == Q4_1:
        return _h(raw, 0) * _nibbles(raw[:, 4:]) + _h(raw, 2)
    if t == Q5_0:
        bit = torch.arange(8, device=raw.device, dtype=torch.uint8)
        hb = ((raw[:, 2:6, None] >> bit) & 1).reshape(n, 32).double()
        return _h(raw, 0) * (_nibbles(raw[:, 6:]) + 16 * hb - 16)
    if t in (Q4_K, Q5_K):
        sc, mn = _sc_min(raw[:, 4:16])
        d = _h(raw, 0) * sc
        q = raw[:, 16 if t == Q4_K else 48:].reshape(n, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(n, 8, 32).double()
        w = _trunc16(d)[:, :, None] * q + _trunc16(-_h(raw, 2) * mn)[:, :, None]
        if t == Q5_K:
            bit = torch.arange(8, device=raw.device, dtype=torch.uint8)
            w = w + _trunc16(16 * d)[:, :, None] * ((raw[:, None, 16:48] >> bit[None, :, None]) & 1).double()
        return w.reshape(n, 256)
    if t == Q6_K:
        ql, qh = raw[:, :128].reshape(n, 2, 2, 32), raw[:, 128:192].reshape(n, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)  # quarter k of a half: 32 codes
        sh = torch.tensor([0, 2, 4, 6], device=raw.device, dtype=torch.uint8).reshape(1, 1, 4, 1)
        q = (lo.to(torch.int32) | (((qh >> sh) & 3).to(torch.int32) << 4)).double() - 32
        sc = raw[:, 192:208].contiguous().view(torch.int8).double().reshape(n, 2, 4, 2).repeat_interleave(16, 3)
        v = (_h(raw, 208)[:, :, None, None] * sc * q).reshape(n * 8, 32)
        s = v.abs().amax(1, keepdim=True) / 127.0
        p = v * (1.0 / s)
        code = torch.where(s > 0, torch.trunc(p + torch.copysign(torch.full_like(p, 0.5), p)), torch.zeros_like(p))
        return (_trunc16(s) * code.clamp(-128, 127)).reshape(n, 256)
    sh = torch.tensor([0, 2, 4, 6], device=raw.device, dtype=torch.uint8).reshape(1, 1, 4, 1)
    if t == Q2_K:
        sc = raw[:, :16].to(torch.int32)
        q = ((raw[:, 16:80].reshape(n, 2, 1, 32) >> sh) & 3).reshape(n, 16, 16).double()
        w = (_h(raw, 80) * (sc & 15))[:, :, None] * q - (_h(raw, 82) * (sc >> 4))[:, :, None]
    else:
        b = raw[:, 96:108].to(torch.int32)
        lo = torch.cat([b[:, :8] & 15, b[:, :8] >> 4], 1)
        sc = lo | (torch.cat([(b[:, 8:] >> k) & 3 for k in (0, 2, 4, 6)], 1) << 4)
        q = ((raw[:, 32:96].reshape(n, 2, 1, 32) >> sh) & 3).reshape(n, 8, 32).double()
        bit = torch.arange(8, device=raw.device, dtype=torch.uint8)
        q = q - 4 * (1 - ((raw[:, None, :32] >> bit[None, :, None]) & 1).double())
        w = (_h(raw, 108) * (sc - 32))[:, :, None] * q.reshape(n, 16, 16)
    return w.float().double().reshape(n, 256)


def _codes(x):
    """x as the Q8_0 activations hold it: fp32 scale and inverse per 32 elements, truncated codes."""
    b = x.double().reshape(-1, 32)
    s = (b.abs().amax(1, keepdim=True) / 127.0).float().double()
    inv = torch.where(s > 0, (1.0 / s).float().double(), torch.zeros_like(s))
    return (torch.trunc((b * inv).float().double()).clamp(-128, 127) * s).reshape(x.shape)


def _exact_mm(t, rows, cols, g, x):
    raw = _raw(t, rows, cols, g)
    a = x.double() if t in (Q5_0, Q2_K, Q3_K) else _codes(x)
    per, out = max(1, (1 << 26) // cols), []
    nb = cols // BLOCK[t][0]
    for r in range(0, rows, per):
        w = _dense(t, raw[r * nb:min(rows, r + per) * nb]).reshape(-1, cols)
        out.append(a @ w.t().contiguous())
    return torch.cat(out, 1)


def _exact_norm(x, w):
    ss = x.double().square().sum(1, keepdim=True).float().double()
    inv = (1.0 / torch.sqrt(ss / x.shape[1] + EPS).float().double()).float()
    return (x * inv) * w


def _exact_attn(c, seed):
    q, k, v = _qkv_input(c, seed)
    m, dk, pos, kvh = c["m"], c["dk"], c["pos"], c["kv_heads"]
    ang = (_freqs(dk)[None, :] * torch.arange(pos, pos + m, device="cuda").float()[:, None]).double()
    cs, sn = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]

    def rope(t):
        a = t.double().reshape(m, -1, dk // 2, 2)
        return torch.stack([a[..., 0] * cs - a[..., 1] * sn, a[..., 0] * sn + a[..., 1] * cs], -1).reshape(m, -1, dk)

    g = _gen(seed, 90)
    hk, hv = _normal(g, kvh, pos, dk, std=0.7).double(), _normal(g, kvh, pos, dk).double()
    qr, kr, vr = rope(q), rope(k).transpose(0, 1), v.double().reshape(m, kvh, dk).transpose(0, 1)
    K, V = torch.cat([hk, kr], 1), torch.cat([hv, vr], 1)
    mask = torch.arange(pos + m, device="cuda")[None, :] > torch.arange(pos, pos + m, device="cuda")[:, None]
    out = torch.empty(m, c["heads"], dk, dtype=torch.float64, device="cuda")
    rep = c["heads"] // kvh
    for h in range(c["heads"]):
        p = (qr[:, h] @ K[h // rep].t().contiguous()) / math.sqrt(dk)
        out[:, h] = torch.softmax(p.masked_fill(mask, -math.inf), 1) @ V[h // rep]
    return out.reshape(m, -1), kr, vr


def exact(c, seed):
    """What run(prepare(c, seed)) returns, in 64 bits. Second quantizations (ffn's second output, layer, model)
    have no such value: their codes follow the first part's rounding."""
    op = c["op"]
    if op == "attn":
        return _exact_attn(c, seed)
    if op in ("layer", "model"):
        return None
    x = _x(c, c.get("cols", c.get("hidden")), seed)
    if op in ("matmul", "host"):
        y = _exact_mm(c["type"], c["rows"], c["cols"], _gen(seed, 10), x)
        return y if op == "matmul" else y.reshape(-1)
    n = _exact_norm(x, _norm_w(x.shape[1], seed))
    if op == "head":
        return _exact_mm(c["type"], c["rows"], c["cols"], _gen(seed, 10), n), None
    if op == "qkv":
        return [_exact_mm(c["type"], r, c["hidden"], _gen(seed, 10 + i), n) for i, r in
                enumerate((c["hidden"], c["kv"], c["kv"]))]
    gate, up = (_exact_mm(c["gate"], c["inner"], c["hidden"], _gen(seed, 10 + i), n) for i in range(2))
    return gate / (1.0 + torch.exp(-gate)) * up, None
