"""Performance cases of the quantized-matmul library: what a language-model runtime asks of it, by size.

A runtime keeps its weights in device handles and calls the device tier with f32 activations:

  gemv     one matrix times one token, quantized in the launch (a K or V projection, a small model's layer)
  decode   the seven products of Llama layers for one token, eagerly, as a generation loop does
  head     the greedy output head: logits and their argmax
  vec_dot  one matrix times one f32 token with no activation quantization
  bitnet   a BitNet feed-forward block (sub-layer norm + absmax quantizer, ternary products, ReLU^2)
  ternary  ternary products of a batch of prompt tokens that share one sub-layer norm
  proj     projections of one batch of tokens that share its quantization (Q/K/V, gate/up), 3 tokens
           of a speculative step up to a 2048-token prompt, bit-exact or in tolerance mode
  ffn      a Llama feed-forward block for a batch of tokens, SwiGLU fused into the second quantizer

Sizes are those of Llama-3-8B, Llama-7B and BitNet-2B layers; draw() spreads them over the ranges in
between, odd and ragged ones among them. Activations are normal with a few channels several times
larger, as residual streams have; weights are random quants with block scales of trained magnitude.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "jero-kernels-rvv_amd"))

import jk  # noqa: E402

FORMATS = {"Q4_0": jk.Q4_0, "Q8_0": jk.Q8_0, "Q4_K": jk.Q4_K, "Q5_K": jk.Q5_K, "Q6_K": jk.Q6_K, "TQ2_0": jk.TQ2_0,
           "I2_S": jk.I2_S}
EPS = 1e-5
DEV = "cuda"


def listed():
    return [
        # a K or V projection of one token: the smallest call a decode loop makes
        {"name": "gemv_k_proj", "kind": "gemv", "quant": "Q4_K", "rows": 1024, "cols": 4096},
        # four Llama-3-8B layers of one generated token (552 MB of weights: they come from HBM)
        {"name": "decode_llama3_8b_x4", "kind": "decode", "hidden": 4096, "ffn": 14336, "layers": 4},
        # the greedy step's output head at Llama-3's vocabulary
        {"name": "lm_head_q6k", "kind": "head", "quant": "Q6_K", "rows": 128256, "cols": 4096},
        # an attention output projection of a runtime that keeps activations in f32
        {"name": "vec_dot_q4k", "kind": "vec_dot", "quant": "Q4_K", "rows": 4096, "cols": 4096, "mode": "exact"},
        # one token through a BitNet-2B feed-forward block
        {"name": "bitnet_decode", "kind": "bitnet", "quant": "TQ2_0", "hidden": 2560, "ffn": 6912, "tokens": 1},
        # a short prompt through BitNet-2B's gate and up
        {"name": "ternary_i2s_m128_tol", "kind": "ternary", "quant": "I2_S", "rows": "6912+6912", "cols": 2560,
         "tokens": 128, "mode": "tol"},
        # a speculative step or four concurrent sequences through a Q4_K_M feed-forward block
        {"name": "ffn_q4km_m4", "kind": "ffn", "quant": "Q4_K", "quant_down": "Q6_K", "hidden": 4096, "ffn": 14336,
         "tokens": 4},
        # a short ragged prompt through the attention projections
        {"name": "qkvo_q4k_m33", "kind": "proj", "quant": "Q4_K", "rows": "4096+1024+1024+4096", "cols": 4096,
         "tokens": 33, "mode": "exact"},
        # Llama-7B gate and up, a paragraph of prompt, tolerance mode
        {"name": "gate_up_q4_0_m150_tol", "kind": "proj", "quant": "Q4_0", "rows": "11008+11008", "cols": 4096,
         "tokens": 150, "mode": "tol"},
        # a 512-token prompt chunk through a Q4_K_M feed-forward block, bit-exact
        {"name": "ffn_q4km_m512", "kind": "ffn", "quant": "Q4_K", "quant_down": "Q6_K", "hidden": 4096,
         "ffn": 14336, "tokens": 512},
        # the Q8_0 prefill product at a 512-token chunk, tolerance mode
        {"name": "up_q8_0_m512_tol", "kind": "proj", "quant": "Q8_0", "rows": "14336", "cols": 4096, "tokens": 512,
         "mode": "tol"},
        # a long prompt chunk through gate and up, tolerance mode: the largest call
        {"name": "gate_up_q4k_m2048_tol", "kind": "proj", "quant": "Q4_K", "rows": "14336+14336", "cols": 4096,
         "tokens": 2048, "mode": "tol"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _rows(case):
    """The row counts of a case's matrices ("4096+1024": two that share one activation)."""
    return [int(r) for r in str(case["rows"]).split("+")]


def _cols(rng, quant, lo=1024, hi=14336):
    """A column count: whole weight blocks (256, 128 or 32 elements)."""
    be = jk.BLOCK_ELEMENTS[FORMATS[quant]]
    return max(be, _log_int(rng, lo, hi) // be * be)


def draw(rng):
    kind = rng.choice(["gemv", "decode", "head", "vec_dot", "bitnet", "ternary", "proj", "proj", "proj", "ffn", "ffn"])
    if kind == "gemv":
        q = rng.choice(["Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"])
        return {"kind": kind, "quant": q, "rows": _log_int(rng, 1024, 16384), "cols": _cols(rng, q, 2048, 8192)}
    if kind == "decode":
        return {"kind": kind, "hidden": 256 * rng.randint(8, 20), "ffn": 256 * rng.randint(20, 56),
                "layers": rng.randint(2, 5)}
    if kind == "head":
        q = rng.choice(["Q6_K", "Q8_0", "Q4_K"])
        return {"kind": kind, "quant": q, "rows": _log_int(rng, 32000, 151936), "cols": _cols(rng, q, 1024, 4096)}
    if kind == "vec_dot":
        q = rng.choice(["Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"])
        return {"kind": kind, "quant": q, "rows": _log_int(rng, 1024, 14336), "cols": _cols(rng, q, 2048, 14336),
                "mode": rng.choice(["exact", "tol"])}
    if kind == "bitnet":
        return {"kind": kind, "quant": rng.choice(["TQ2_0", "I2_S"]), "hidden": 256 * rng.randint(6, 16),
                "ffn": 256 * rng.randint(16, 43), "tokens": rng.choice([1, 1, 2, 5, 17])}
    if kind == "ternary":
        q = rng.choice(["TQ2_0", "I2_S"])
        return {"kind": kind, "quant": q, "rows": str(_log_int(rng, 640, 8192)), "cols": _cols(rng, q, 1024, 8192),
                "tokens": _log_int(rng, 16, 600), "mode": rng.choice(["exact", "tol"])}
    if kind == "ffn":
        q, d = rng.choice([("Q4_K", "Q6_K"), ("Q4_K", "Q4_K"), ("Q5_K", "Q6_K"), ("Q8_0", "Q8_0"), ("Q4_0", "Q4_0")])
        return {"kind": kind, "quant": q, "quant_down": d, "hidden": 256 * rng.randint(8, 20),
                "ffn": 256 * rng.randint(20, 56), "tokens": _log_int(rng, 3, 700)}
    q = rng.choice(["Q4_0", "Q8_0", "Q4_K", "Q4_K", "Q5_K", "Q6_K"])
    rows = "+".join(str(_log_int(rng, 512, 14336)) for _ in range(rng.choice([1, 2, 3])))
    return {"kind": kind, "quant": q, "rows": rows, "cols": _cols(rng, q, 1024, 8192),
            "tokens": _log_int(rng, 3, 1400), "mode": rng.choice(["exact", "tol"])}


# ------------------------------------------------------------------ inputs
def _layer(case):
    """A Llama layer's matrices at four query heads per key / value head: (name, format, rows, cols)."""
    d, f = case["hidden"], case["ffn"]
    return [("q", "Q4_K", d, d), ("k", "Q4_K", d // 4, d), ("v", "Q4_K", d // 4, d), ("o", "Q4_K", d, d),
            ("gate", "Q4_K", f, d), ("up", "Q4_K", f, d), ("down", "Q6_K", d, f)]


def _gen(seed, salt):
    return torch.Generator(device=DEV).manual_seed((seed * 1000003 + salt * 7919) & 0x7FFFFFFFFFFF)


def _f16(g, n, c):
    """n positive block scales around c as f16 byte pairs [n, 2]."""
    v = (torch.rand(n, generator=g, device=DEV) + 0.5) * c
    return v.to(torch.float16).view(torch.uint8).reshape(n, 2)


def _blocks(quant, rows, cols, g):
    """Random GGUF blocks [rows, blocks, block bytes] on the device."""
    q = FORMATS[quant]
    n, bb = rows * (cols // jk.BLOCK_ELEMENTS[q]), jk.BLOCK_BYTES[q]
    b = torch.randint(0, 256, (n, bb), generator=g, device=DEV, dtype=torch.uint8)
    if quant == "Q4_0":
        b[:, :2] = _f16(g, n, 0.02 / 8)
    elif quant == "Q8_0":
        b[:, :2] = _f16(g, n, 0.06 / 127)
        b[:, 2:].masked_fill_(b[:, 2:] == 128, 0)  # quants lie in -127 .. 127
    elif quant in ("Q4_K", "Q5_K"):
        c = 0.02 / 8 / 32 if quant == "Q4_K" else 0.02 / 16 / 32
        b[:, :2], b[:, 2:4] = _f16(g, n, c), _f16(g, n, c * (7.5 if quant == "Q4_K" else 15.5))
    elif quant == "Q6_K":
        b[:, 192:208] = torch.randint(-64, 64, (n, 16), generator=g, device=DEV, dtype=torch.int8).view(torch.uint8)
        b[:, 208:] = _f16(g, n, 0.02 / 16 / 32)
    else:  # ternary: 2-bit fields 0..2
        t = torch.randint(0, 3, (n, bb - (2 if quant == "TQ2_0" else 0), 4), generator=g, device=DEV, dtype=torch.uint8)
        packed = t[..., 0] | (t[..., 1] << 2) | (t[..., 2] << 4) | (t[..., 3] << 6)
        if quant == "TQ2_0":
            b[:, 2:] = packed
            b[:, :2] = torch.full((n,), 0.03125 * 1.5, device=DEV).to(torch.float16).view(torch.uint8).reshape(n, 2)
        else:
            b = packed
    return b.reshape(rows, -1, b.shape[1])


I2S_SCALE = 0.046875


def _weight(quant, rows, cols, g):
    data = _blocks(quant, rows, cols, g).reshape(-1).cpu().numpy()
    if quant == "I2_S":
        data = np.concatenate([data, np.zeros(32, np.uint8)])
        data[-32:-28] = np.frombuffer(np.float32(I2S_SCALE).tobytes(), np.uint8)
    return jk.Weight(jk.TensorView("w", FORMATS[quant], (rows, cols), data), rows, cols)


def _acts(m, k, g):
    x = torch.randn(m, k, generator=g, device=DEV)
    big = torch.randint(0, k, (max(1, k // 512),), generator=g, device=DEV)
    x[:, big] *= 6.0
    return x


def _f32(*shape):
    return torch.empty(*shape, dtype=torch.float32, device=DEV)


def _u8(n):
    return torch.empty(n, dtype=torch.uint8, device=DEV)


def _act_q8(m, k):
    store = _u8(jk.act_q8_bytes(m, k))
    return store, jk.act_q8_bind(store, store.numel(), m, k)


def prepare(case, seed):
    jk.init(torch.cuda.current_device())
    s, kind = {"case": case}, case["kind"]
    if kind in ("gemv", "vec_dot", "head"):
        s["w"] = _weight(case["quant"], case["rows"], case["cols"], _gen(seed, 1))
        s["x"] = _acts(1, case["cols"], _gen(seed, 2))
        s["y"] = _f32(case["rows"])
        if kind == "head":
            s["ws"] = _u8(jk.argmax_workspace_bytes(case["rows"]))
            s["index"] = torch.empty(1, dtype=torch.int32, device=DEV)
    elif kind == "decode":
        n = case["layers"]
        s["w"] = [{nm: _weight(q, r, c, _gen(seed, 100 * i + j)) for j, (nm, q, r, c) in enumerate(_layer(case))}
                  for i in range(n)]
        for j, nm in enumerate(("x", "attn", "ffn_in")):
            s[nm] = _acts(n, case["hidden"], _gen(seed, 50 + j))
        s["out"] = {nm: _f32(n, r) for nm, _, r, _ in _layer(case)}
        s["h"] = _u8(case["ffn"] // 256 * jk.BLOCK_Q8K.itemsize)
        s["jobs"] = []
        for i, w in enumerate(s["w"]):
            def job(nm, xf=None, xq=None):
                return (w[nm], xq, xf, s["out"][nm][i], 0, w[nm].rows)
            s["jobs"].append([jk.gemv_jobs([job("q", s["x"][i]), job("k", s["x"][i]), job("v", s["x"][i])]),
                              jk.gemv_jobs([job("o", s["attn"][i])]),
                              jk.gemv_jobs([job("gate", s["ffn_in"][i]), job("up", s["ffn_in"][i])]),
                              jk.gemv_jobs([job("down", None, s["h"])])])
    elif kind == "bitnet":
        m, d, f, q = case["tokens"], case["hidden"], case["ffn"], case["quant"]
        s["w"] = [_weight(q, r, c, _gen(seed, 10 + j)) for j, (r, c) in enumerate([(f, d), (f, d), (d, f)])]
        s["x"], s["norm"], s["norm2"] = _acts(m, d, _gen(seed, 2)), _norm(d, seed, 3), _norm(f, seed, 4)
        s["q1"], s["q2"] = (torch.empty(m, k, dtype=torch.int8, device=DEV) for k in (d, f))
        s["s1"], s["s2"] = _f32(m), _f32(m)
        s["gate"], s["up"], s["h"], s["y"] = _f32(m, f), _f32(m, f), _f32(m, f), _f32(m, d)
    elif kind == "ternary":
        m, k = case["tokens"], case["cols"]
        s["w"] = [_weight(case["quant"], r, k, _gen(seed, 10 + j)) for j, r in enumerate(_rows(case))]
        s["x"], s["norm"] = _acts(m, k, _gen(seed, 2)), _norm(k, seed, 3)
        s["q1"], s["s1"] = torch.empty(m, k, dtype=torch.int8, device=DEV), _f32(m)
        s["y"] = [_f32(m, r) for r in _rows(case)]
    elif kind == "proj":
        m, k = case["tokens"], case["cols"]
        s["w"] = [_weight(case["quant"], r, k, _gen(seed, 10 + j)) for j, r in enumerate(_rows(case))]
        s["x"] = _acts(m, k, _gen(seed, 2))
        s["store"], s["act"] = _act_q8(m, k)
        s["y"] = [_f32(m, r) for r in _rows(case)]
    elif kind == "ffn":
        m, d, f = case["tokens"], case["hidden"], case["ffn"]
        s["w"] = [_weight(q, r, c, _gen(seed, 10 + j))
                  for j, (q, r, c) in enumerate([(case["quant"], f, d), (case["quant"], f, d),
                                                 (case["quant_down"], d, f)])]
        s["x"] = _acts(m, d, _gen(seed, 2))
        s["store"], s["act"] = _act_q8(m, d)
        s["store2"], s["act2"] = _act_q8(m, f)
        s["gate"], s["up"], s["y"] = _f32(m, f), _f32(m, f), _f32(m, d)
    torch.cuda.synchronize()
    return s


def _norm(k, seed, salt):
    return 1.0 + 0.1 * torch.randn(k, generator=_gen(seed, salt), device=DEV)


# -------------------------------------------------------------------- run
def run(s):
    case, st = s["case"], torch.cuda.current_stream().cuda_stream
    kind = case["kind"]
    if kind == "gemv":
        jk.dev_gemv_q8_f32(s["w"], s["x"], case["cols"], s["y"], case["rows"], st)
        return s["y"]
    if kind == "vec_dot":
        f = jk.dev_vec_dot_f32 if case["mode"] == "exact" else jk.dev_vec_dot_f32_tol
        f(s["w"], s["x"], case["cols"], s["y"], case["rows"], st)
        return s["y"]
    if kind == "head":
        jk.dev_gemv_q8_argmax(s["w"], None, s["x"], case["cols"], s["y"], s["index"], s["ws"], st)
        return {"logits": s["y"], "token": s["index"]}
    if kind == "decode":
        out, f = s["out"], case["ffn"]
        for i, (qkv, o, gu, down) in enumerate(s["jobs"]):
            jk.dev_gemv_q8_batch(qkv, st)
            jk.dev_gemv_q8_batch(o, st)
            jk.dev_gemv_q8_batch(gu, st)
            jk.dev_quantize_row_q8_k_gated(jk.ACT_SWIGLU, out["gate"][i], out["up"][i], f, s["h"],
                                            f // 256, st)
            jk.dev_gemv_q8_batch(down, st)
        return out
    m = case["tokens"]
    if kind == "bitnet":
        d, f = case["hidden"], case["ffn"]
        gate, up, down = s["w"]
        jk.dev_subln_quantize_absmax_i8(s["x"], s["norm"], m, d, EPS, s["q1"], s["s1"], st)
        jk.dev_bitlinear_i8(gate, s["q1"], s["s1"], m, d, s["gate"], m * f, st)
        jk.dev_bitlinear_i8(up, s["q1"], s["s1"], m, d, s["up"], m * f, st)
        jk.dev_relu_squared_gate_f32(s["gate"], s["up"], m * f, s["h"], st)
        jk.dev_subln_quantize_absmax_i8(s["h"], s["norm2"], m, f, EPS, s["q2"], s["s2"], st)
        jk.dev_bitlinear_i8(down, s["q2"], s["s2"], m, f, s["y"], m * d, st)
        return {"gate": s["gate"], "up": s["up"], "y": s["y"]}
    if kind == "ternary":
        k = case["cols"]
        mul = jk.dev_bitlinear_i8 if case["mode"] == "exact" else jk.dev_bitlinear_i8_tol
        jk.dev_subln_quantize_absmax_i8(s["x"], s["norm"], m, k, EPS, s["q1"], s["s1"], st)
        for w, y in zip(s["w"], s["y"]):
            mul(w, s["q1"], s["s1"], m, k, y, m * w.rows, st)
        return s["y"]
    if kind == "proj":
        k = case["cols"]
        mul = jk.dev_gemm_repacked if case["mode"] == "exact" else jk.dev_gemm_repacked_tol
        jk.dev_quantize_act_q8(s["x"], m, k, s["act"], st)
        for w, y in zip(s["w"], s["y"]):
            mul(w, s["act"], y, m * w.rows, 0, w.rows, st)
        return s["y"]
    d, f = case["hidden"], case["ffn"]
    gate, up, down = s["w"]
    jk.dev_quantize_act_q8(s["x"], m, d, s["act"], st)
    jk.dev_gemm_repacked(gate, s["act"], s["gate"], m * f, 0, f, st)
    jk.dev_gemm_repacked(up, s["act"], s["up"], m * f, 0, f, st)
    jk.dev_quantize_act_q8_gated(jk.ACT_SWIGLU, s["gate"], s["up"], m, f, s["act2"], st)
    jk.dev_gemm_repacked(down, s["act2"], s["y"], m * d, 0, d, st)
    return {"gate": s["gate"], "up": s["up"], "y": s["y"]}


# ------------------------------------------------------------------- work
def _wbytes(quant, rows, cols):
    q = FORMATS[quant]
    return rows * (cols // jk.BLOCK_ELEMENTS[q]) * jk.BLOCK_BYTES[q]


def work(case):
    """f32 activations and GGUF weights in, f32 results out; a multiply and an add per weight and token."""
    kind, m = case["kind"], case.get("tokens", 1)
    if kind == "decode":
        mats, per, n = [(q, r, c) for _, q, r, c in _layer(case)], 4 * 3 * case["hidden"], case["layers"]
    elif kind in ("bitnet", "ffn"):
        d, f = (case["hidden"], case["ffn"])
        q2 = case.get("quant_down", case["quant"])
        mats, per, n = [(case["quant"], f, d), (case["quant"], f, d), (q2, d, f)], 4 * m * d, 1
    else:
        mats, per, n = [(case["quant"], r, case["cols"]) for r in _rows(case)], 4 * m * case["cols"], 1
    w = sum(_wbytes(*x) for x in mats)
    out = sum(4 * m * r for _, r, _ in mats)
    return {"bytes": n * (w + per + out), "flops": n * sum(2 * m * r * c for _, r, c in mats)}


def tolerance(case):
    """The bit-exact entry points promise the reference's arithmetic and order: any difference is a fault.
    Tolerance mode sums 32-bit floats in any order: 2e-7 to 3e-7 against 64 bits, and for Q8_0 at 512 tokens,
    whose group sums carry a bias of 1.5 * 2^23 through the accumulator, 2.3e-5. Through SwiGLU another
    correct exponential moves some of the second quantizer's roundings by one of 127 levels: 2e-4 of one
    token's output for each, 7.6e-5 measured over a batch of 512."""
    if case["kind"] in ("decode", "ffn"):
        return {"rel": 1e-3}
    if case.get("mode") == "tol":
        return {"rel": 1e-4 if case["quant"] == "Q8_0" else 1.5e-6}
    return "exact"


# ------------------------------------------------------------------ exact
def _half(b):
    return b.contiguous().view(torch.float16)[..., 0].double()


def _unpack(quant, b):
    """GGUF blocks [rows, nb, bytes] -> weights without their mins, and the mins per 32 (or None), in 64 bits."""
    rows = b.shape[0]
    if quant == "Q4_0":
        q = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], -1).double() - 8
        return (q * _half(b[..., :2])[..., None]).reshape(rows, -1), None
    if quant == "Q8_0":
        return (b[..., 2:].contiguous().view(torch.int8).double() * _half(b[..., :2])[..., None]).reshape(rows, -1), None
    if quant in ("Q4_K", "Q5_K"):
        p = b[..., 4:16]
        lo, hi = p[..., :4], p[..., 4:8]
        sc = torch.cat([lo & 63, (p[..., 8:] & 15) | ((lo >> 6) << 4)], -1).double()
        mn = torch.cat([hi & 63, (p[..., 8:] >> 4) | ((hi >> 6) << 4)], -1).double()
        qs = b[..., -128:].reshape(rows, -1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 3).reshape(rows, -1, 8, 32)
        if quant == "Q5_K":
            sh = torch.arange(8, device=b.device, dtype=torch.uint8).reshape(8, 1)
            q = q + (((b[..., 16:48].unsqueeze(2) >> sh) & 1) << 4)
        d, dm = _half(b[..., :2])[..., None], _half(b[..., 2:4])[..., None]
        return (q.double() * (d * sc)[..., None]).reshape(rows, -1), (dm * mn).reshape(rows, -1)
    if quant == "Q6_K":
        out = []
        for h in range(2):
            ql, qh = b[..., 64 * h:64 * h + 64], b[..., 128 + 32 * h:160 + 32 * h]
            for k in range(4):
                lo = ql[..., 32 * (k % 2):32 * (k % 2) + 32]
                out.append(((lo & 15) if k < 2 else (lo >> 4)) | (((qh >> (2 * k)) & 3) << 4))
        q = torch.cat(out, -1).double().reshape(rows, -1, 16, 16) - 32
        sc = b[..., 192:208].contiguous().view(torch.int8).double() * _half(b[..., 208:])[..., None]
        return (q * sc[..., None]).reshape(rows, -1), None
    if quant == "TQ2_0":
        q = torch.stack([(b[..., 2:] >> (2 * j)) & 3 for j in range(4)], -1).double().reshape(rows, b.shape[1], 256) - 1
        return (q * _half(b[..., :2])[..., None]).reshape(rows, -1), None
    q = torch.cat([(b >> sh) & 3 for sh in (6, 4, 2, 0)], -1).double() - 1  # I2_S
    return (q * I2S_SCALE).reshape(rows, -1), None


def _round_away(v):
    return torch.sign(v) * torch.floor(v.abs() + 0.5)


def _block_quant(x, block):
    """The formats' f32 quantizer over blocks of a row: whole levels times the block scale."""
    xb = x.float().reshape(x.shape[0], -1, block)
    amax = xb.abs().amax(-1, keepdim=True)
    c = torch.full_like(amax, 127.0)  # (a tensor: torch turns division by or of a number into a reciprocal)
    q = _round_away((xb * (c / amax)).double()).clamp(-127, 127)
    return torch.where(amax > 1e-30, q * (amax / c).double(), 0.0).reshape(x.shape[0], -1)


def _absmax_quant(x, norm):
    """RMS sub-layer norm and per-token absmax levels, in f32 as specified (its sum runs in order)."""
    sq = np.cumsum((x.float() * x.float()).cpu().numpy(), axis=1, dtype=np.float32)[:, -1]
    inv = (np.float32(1.0) / np.sqrt(sq / np.float32(x.shape[1]) + np.float32(EPS))).astype(np.float32)
    xn = x.float() * torch.from_numpy(inv).to(x.device)[:, None] * norm
    amax = xn.abs().amax(1, keepdim=True)
    scale = amax / torch.full_like(amax, 127.0)
    return _round_away((xn / scale).double()).clamp(-128, 127) * scale.double()


def _product(quant, rows, cols, g, xq, xsum=None):
    """xq [m, cols] times the weight that _weight() makes from g, in 64 bits, a slice of rows at a time."""
    b = _blocks(quant, rows, cols, g)
    out = []
    for r in range(0, rows, 16384):
        w, mins = _unpack(quant, b[r:r + 16384])
        y = xq @ w.T
        if mins is not None:
            y -= xsum @ mins.T
        out.append(y)
    return torch.cat(out, 1)


def _sums32(x):
    return x.double().reshape(x.shape[0], -1, 32).sum(-1)


def _swiglu(g, u):
    return g / (1.0 + torch.exp(-g)) * u


def exact(case, seed):
    kind = case["kind"]

    def gemv(q, r, c, salt, x, f32=False):
        xq = x.double() if f32 else _block_quant(x, 32 if q in ("Q4_0", "Q8_0") else 256)
        return _product(q, r, c, _gen(seed, salt), xq, _sums32(xq))

    if kind in ("gemv", "vec_dot", "head"):
        x = _acts(1, case["cols"], _gen(seed, 2))
        y = gemv(case["quant"], case["rows"], case["cols"], 1, x, kind == "vec_dot").reshape(-1)
        return {"logits": y, "token": None} if kind == "head" else y
    if kind == "decode":
        n = case["layers"]
        a = {nm: _acts(n, case["hidden"], _gen(seed, 50 + j)) for j, nm in enumerate(("x", "attn", "ffn_in"))}
        src = {"q": "x", "k": "x", "v": "x", "o": "attn", "gate": "ffn_in", "up": "ffn_in"}
        out = {nm: [] for nm, *_ in _layer(case)}
        for i in range(n):
            for j, (nm, q, r, c) in enumerate(_layer(case)):
                x = a[src[nm]][i:i + 1] if nm in src else _swiglu(out["gate"][i], out["up"][i])
                out[nm].append(gemv(q, r, c, 100 * i + j, x))
        return {nm: torch.cat(v) for nm, v in out.items()}
    m = case["tokens"]
    if kind in ("bitnet", "ternary"):
        k = case["hidden"] if kind == "bitnet" else case["cols"]
        xq = _absmax_quant(_acts(m, k, _gen(seed, 2)), _norm(k, seed, 3))
        if kind == "ternary":
            return [_product(case["quant"], r, k, _gen(seed, 10 + j), xq) for j, r in enumerate(_rows(case))]
        f = case["ffn"]
        gate, up = (_product(case["quant"], f, k, _gen(seed, 10 + j), xq) for j in range(2))
        h = gate.clamp_min(0.0) ** 2 * up
        return {"gate": gate, "up": up,
                "y": _product(case["quant"], k, f, _gen(seed, 12), _absmax_quant(h, _norm(f, seed, 4)))}

    def gemm(q, r, c, salt, x):
        return _product(q, r, c, _gen(seed, salt), _block_quant(x, 32), _sums32(x))

    if kind == "proj":
        x = _acts(m, case["cols"], _gen(seed, 2))
        return [gemm(case["quant"], r, case["cols"], 10 + j, x) for j, r in enumerate(_rows(case))]
    d, f = case["hidden"], case["ffn"]
    x = _acts(m, d, _gen(seed, 2))
    gate, up = (gemm(case["quant"], f, d, 10 + j, x) for j in range(2))
    return {"gate": gate, "up": up, "y": gemm(case["quant_down"], d, f, 12, _swiglu(gate, up))}
