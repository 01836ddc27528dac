"""The calls a user of this library makes, as cases to be timed and checked.

A case is one linear layer (or one expert layer) of a quantised language model: the token counts of
decode, small batches and prefill, over the weight formats, the layer sizes and the activation
forms that the definitions, the tests and the benchmark of this repository use.

  linear   out[M][N] = x[M][K] . W[N][K]^T through ops.forward, activations quantised in the call
           (act "float32"; "w8a8c8" and "deepseek_v2" by those operators' rules) or before it
           ("q8_1": one quantised input that several projections share)
  fp16     the same from float16 activations, through ops.gemm_q4_0_fp16_fused (out [N][M])
  w16      float32 activations against dequantised weights (W4A16 / W8A16), ops.gemm_w16
  moe      routing, top-k and the experts' up-projection, ops.moe_gemm
"""
from __future__ import annotations

import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "k-search_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from ksq import ops  # noqa: E402

# name: (library type, elements per block, bytes per block, entry for fp32 input, for block_q8_1 input)
FORMATS = {
    "q4_0": (0, 32, 18, "gemm_w4a32c8_q4_0_fp32_int8", "ksq_gemm_q4_0_q8_1"),
    "q8_0": (1, 32, 34, "gemm_w8a32c8_q8_0_fp32_int8", "ksq_gemm_q8_0_q8_1"),
    "q4_K": (2, 256, 144, "gemm_w4a32c8_q4_k_fp32_int8", "ksq_gemm_q4_k_q8_1"),
    "q6_K": (3, 256, 210, "gemm_w6a32c8_q6_k_fp32_int8", "ksq_gemm_q6_k_q8_1"),
    "q4_1": (4, 32, 20, "gemm_w4a32c8_q4_1_fp32_int8", "ksq_gemm_q4_1_q8_1"),
    "q5_0": (5, 32, 22, "gemm_w5a32c8_q5_0_fp32_int8", "ksq_gemm_q5_0_q8_1"),
    "q5_1": (6, 32, 24, "gemm_w5a32c8_q5_1_fp32_int8", "ksq_gemm_q5_1_q8_1"),
}


def _linear(name, weight, act, M, N, K):
    return {"name": name, "op": "linear", "weight": weight, "act": act, "M": M, "N": N, "K": K}


def listed():
    return [
        # one token through an attention projection: the smallest call, latency counts
        _linear("decode_q4_0", "q4_0", "float32", 1, 4096, 4096),
        # one token through the vocabulary head: the largest weight matrix a decode step reads
        _linear("lm_head_q4_0", "q4_0", "float32", 1, 128256, 4096),
        # five sequences decoded together through a small fused qkv projection
        _linear("batch5_q4_1", "q4_1", "float32", 5, 1536, 7168),
        # small serving batches
        _linear("batch8_q8_0", "q8_0", "float32", 8, 4096, 4096),
        _linear("batch32_q8_0", "q8_0", "float32", 32, 4096, 4096),
        # a short prompt, or a large decode batch, through a K-quant up-projection
        _linear("chunk128_q4_K", "q4_K", "float32", 128, 14336, 4096),
        _linear("chunk128_q6_K", "q6_K", "float32", 128, 14336, 4096),
        # a prompt of no particular length through a small model's projection
        _linear("prompt333_q4_1", "q4_1", "float32", 333, 2560, 2560),
        # a prefill chunk through an 8-bit up-projection
        _linear("prefill512_q8_0", "q8_0", "float32", 512, 14336, 4096),
        # a long prompt through an attention projection
        _linear("prefill2048_q4_0", "q4_0", "float32", 2048, 4096, 4096),
        # the same where the activations must not be quantised
        {"name": "prefill2048_w4a16", "op": "w16", "weight": "q4_0", "M": 2048, "N": 4096, "K": 4096},
        # a batch of tokens through eight experts, two for each token
        {"name": "moe512_q4_0", "op": "moe", "weight": "q4_0", "T": 512, "N": 14336, "K": 4096, "E": 8, "top_k": 2,
         "renorm": False},
    ]


MAX_MACS = 2.4e10       # of a drawn case: below the largest listed ones'
MAX_WEIGHTS = 2.9e8     # bytes


def _log(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def _layer(rng, weight, rows, n_hi, step):
    """N and K of a layer: K a multiple of `step`, N any whole number half of the time."""
    _, be, bb, _, _ = FORMATS[weight]
    step = max(step, be)
    K = max(step, int(_log(rng, 1024, 18944) / step) * step)
    n_hi = min(n_hi, MAX_MACS / (rows * K), MAX_WEIGHTS / (K / be * bb))
    N = int(_log(rng, min(512, n_hi / 2), n_hi))
    return (N if rng.random() < 0.5 else max(32, N // 32 * 32)), K


def draw(rng):
    kind = rng.choice(["decode", "decode", "batch", "batch", "chunk", "prefill", "prefill", "fp16", "w16", "moe"])
    if kind == "decode":
        weight = rng.choice(list(FORMATS))
        M = rng.choice([1, 1, 1, 2])
        act = rng.choice(["float32", "float32", "q8_1"])
        if weight == "q4_0" and rng.random() < 0.2:
            act = "deepseek_v2"
        if weight == "q8_0" and rng.random() < 0.3:
            act = "w8a8c8"
        N, K = _layer(rng, weight, M, 152064, 256 if act == "deepseek_v2" or rng.random() < 0.7 else 32)
        c = {"op": "linear", "weight": weight, "act": act, "M": M, "N": N, "K": K}
    elif kind == "batch":
        weight = rng.choice(list(FORMATS))
        M = int(_log(rng, 3, 33))
        N, K = _layer(rng, weight, M, 28672, 256 if rng.random() < 0.8 else 32)
        c = {"op": "linear", "weight": weight, "act": rng.choice(["float32", "float32", "q8_1"]), "M": M, "N": N, "K": K}
    elif kind in ("chunk", "prefill"):
        weight = rng.choice(list(FORMATS) + ["q4_0", "q8_0", "q4_1"])
        M = int(_log(rng, 33, 257)) if kind == "chunk" else int(_log(rng, 256, 2049))
        act = rng.choice(["float32", "float32", "q8_1"])
        if weight == "q4_0" and rng.random() < 0.15:
            act = "deepseek_v2"
        if weight == "q8_0" and rng.random() < 0.2:
            act = "w8a8c8"
        N, K = _layer(rng, weight, M, 18944, 256)
        c = {"op": "linear", "weight": weight, "act": act, "M": M, "N": N, "K": K}
    elif kind == "fp16":
        M = rng.choice([1, 1, int(_log(rng, 3, 9)), int(_log(rng, 9, 1025))])
        N, K = _layer(rng, "q4_0", M, 18944, 256)
        c = {"op": "fp16", "weight": "q4_0", "M": M, "N": N, "K": K}
    elif kind == "w16":
        weight = rng.choice(["q4_0", "q8_0"])
        M = int(_log(rng, 1, 2049))
        N, K = _layer(rng, weight, M, 18944, 64)
        c = {"op": "w16", "weight": weight, "M": M, "N": N, "K": K}
    else:
        weight = rng.choice(["q4_0", "q4_0", "q4_1", "q8_0", "q5_0", "q5_1"])
        E = rng.choice([4, 8, 8, 16, 32, 64])
        top_k = rng.choice([1, 2, 2, 2, 4, 6])
        top_k = min(top_k, E)
        T = int(_log(rng, 4, 1025))
        K = 256 * int(_log(rng, 4, 29))
        _, be, bb, _, _ = FORMATS[weight]
        n_hi = min(14336, MAX_MACS / (T * top_k * K), MAX_WEIGHTS / (E * K / be * bb))
        N = int(_log(rng, min(256, n_hi / 2), n_hi))
        c = {"op": "moe", "weight": weight, "T": T, "N": N if rng.random() < 0.4 else max(32, N // 32 * 32), "K": K,
             "E": E, "top_k": top_k, "renorm": rng.random() < 0.5}
    return c


# ---- inputs ------------------------------------------------------------------------------------

def _f16_bytes(v):
    return v.to(torch.float16).contiguous().view(torch.uint8).reshape(*v.shape, 2)


def _weights(fmt, rows, K, g):
    """Random blocks as trained layers have them: uniform quants, small positive scales, block minima
    near the lower end of a centred block."""
    _, be, bb, _, _ = FORMATS[fmt]
    nb = K // be
    w = torch.randint(0, 256, (rows, nb, bb), dtype=torch.uint8, device="cuda", generator=g)

    def n(sigma):
        return (torch.randn((rows, nb), device="cuda", generator=g) * sigma).abs()

    def u(lo, hi):
        return torch.rand((rows, nb), device="cuda", generator=g) * (hi - lo) + lo

    if fmt == "q4_0":
        w[:, :, 0:2] = _f16_bytes(n(0.02))
    elif fmt == "q8_0":
        w[:, :, 0:2] = _f16_bytes(n(0.01))
        q = w[:, :, 2:]
        q[q == 128] = 129      # int8 quants in [-127, 127]
    elif fmt == "q4_K":
        w[:, :, 0:2] = _f16_bytes(n(0.02))
        w[:, :, 2:4] = _f16_bytes(n(0.02))
    elif fmt == "q6_K":
        w[:, :, 208:210] = _f16_bytes(n(0.002))
    elif fmt == "q4_1":
        d = n(0.02)
        w[:, :, 0:2] = _f16_bytes(d)
        w[:, :, 2:4] = _f16_bytes(-d * u(6.0, 9.0))
    elif fmt == "q5_0":
        w[:, :, 0:2] = _f16_bytes(n(0.01))
    else:
        d = n(0.01)
        w[:, :, 0:2] = _f16_bytes(d)
        w[:, :, 2:4] = _f16_bytes(-d * u(13.0, 18.0))
    return w


def _inputs(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    K = case["K"]
    if case["op"] == "moe":
        w = _weights(case["weight"], case["E"] * case["N"], K, g)
        x = torch.randn((case["T"], K), device="cuda", generator=g)
        return w, x, torch.randn((case["T"], case["E"]), device="cuda", generator=g)
    w = _weights(case["weight"], case["N"], K, g)
    x = torch.randn((case["M"], K), device="cuda", generator=g)
    return w, (x.half() if case["op"] == "fp16" else x), None


def prepare(case, seed):
    w, x, logits = _inputs(case, seed)
    if case["op"] == "linear" and case["act"] == "q8_1":
        x = ops.quantize_q8_1(x)
    return {"case": case, "w": w, "x": x, "logits": logits}


def run(state):
    c, w, x = state["case"], state["w"], state["x"]
    op = c["op"]
    if op == "linear":
        wt, _, _, entry, entry_q = FORMATS[c["weight"]]
        entry = {"float32": entry, "q8_1": entry_q, "w8a8c8": "gemm_w8a8c8_q8_0_q8_1",
                 "deepseek_v2": "gemm_w4a32c8_q4_0_fp32_int8_deepseek_v2"}[c["act"]]
        return ops.forward(w, x, c["M"], c["N"], c["K"], entry=entry)
    if op == "fp16":
        return ops.gemm_q4_0_fp16_fused(w, x, c["N"], c["M"], c["K"])
    wt = FORMATS[c["weight"]][0]
    if op == "w16":
        return ops.gemm_w16(wt, x, w, c["M"], c["N"], c["K"])
    return ops.moe_gemm(wt, w, x, state["logits"], c["T"], c["N"], c["K"], c["E"], c["top_k"], renorm=c["renorm"])


def work(case):
    _, be, bb, _, _ = FORMATS[case["weight"]]
    N, K = case["N"], case["K"]
    matrix = N * (K // be) * bb
    if case["op"] == "moe":
        T, E, k = case["T"], case["E"], case["top_k"]
        return {"bytes": matrix * min(E, T * k) + 4 * (T * K + T * E + T * N), "flops": 2 * T * k * N * K}
    M = case["M"]
    act = M * K * {"q8_1": 36 / 32}.get(case.get("act"), 2 if case["op"] == "fp16" else 4)
    return {"bytes": matrix + act + 4 * M * N, "flops": 2 * M * N * K}


def tolerance(case):
    # 32-bit sums of exact block dots in another order: about 3e-7 against 64 bits
    return {"rel": 2e-6, "max": 2e-5}


# ---- the same in 64 bits ---------------------------------------------------------------------------

def _half(b):
    return b.contiguous().view(torch.float16)[..., 0].double()


def _dequant(fmt, w):
    """Blocks [rows][nb][bytes] -> scaled quants [rows][K] (scale times the quant as the integer dot
    takes it) and the factor [rows][K / 32] of each block's activation sum (None: the format has none)."""
    rows, nb, _ = w.shape
    if fmt == "q8_0":
        return (_half(w[:, :, :2])[..., None] * w[:, :, 2:].view(torch.int8).double()).reshape(rows, -1), None
    if fmt == "q6_K":
        ql, qh = w[:, :, :128].reshape(rows, nb, 2, 64), w[:, :, 128:192].reshape(rows, nb, 2, 32)
        q = torch.stack([(ql[..., :32] & 15) | ((qh & 3) << 4), (ql[..., 32:] & 15) | (((qh >> 2) & 3) << 4),
                         (ql[..., :32] >> 4) | (((qh >> 4) & 3) << 4), (ql[..., 32:] >> 4) | ((qh >> 6) << 4)], 3)
        q = q.reshape(rows, nb, 16, 16).double() - 32.0
        sc = w[:, :, 192:208].contiguous().view(torch.int8).double()
        return (q * (sc * _half(w[:, :, 208:210])[..., None])[..., None]).reshape(rows, -1), None
    if fmt == "q4_K":
        s = w[:, :, 4:16]
        sc = torch.cat([s[..., :4] & 63, (s[..., 8:] & 15) | ((s[..., :4] >> 6) << 4)], -1).double()
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1).double()
        q = w[:, :, 16:].reshape(rows, nb, 4, 32)
        q = torch.stack([q & 15, q >> 4], 3).reshape(rows, nb, 8, 32).double()
        d, dmin = _half(w[:, :, :2])[..., None], _half(w[:, :, 2:4])[..., None]
        return (q * (d * sc)[..., None]).reshape(rows, -1), (-dmin * mn).reshape(rows, -1)
    qs = w[:, :, -16:]
    q = torch.cat([qs & 15, qs >> 4], -1).double()
    if fmt in ("q5_0", "q5_1"):
        at = 2 if fmt == "q5_0" else 4
        h = w[:, :, at:at + 4].contiguous().view(torch.int32)
        q += 16.0 * ((h >> torch.arange(32, device=w.device, dtype=torch.int32)) & 1).double()
    d = _half(w[:, :, :2])
    side = {"q4_0": -8.0 * d, "q5_0": -16.0 * d}.get(fmt)
    return (q * d[..., None]).reshape(rows, -1), _half(w[:, :, 2:4]) if side is None else side


def _f32(v):
    return v.float().double()   # a 64-bit result of 32-bit operands rounded once: the 32-bit operation


def _away(v):
    return torch.sign(v) * torch.floor(v.abs() + 0.5)


def _quantise(x, rule):
    """x [M][K] -> the quantised values d * q [M][K] and the sums [M][K / 32] by the operator's rule."""
    M, K = x.shape
    b = x.double().reshape(M, K // 32, 32)
    d = _f32(b.abs().amax(-1) / 127.0)
    if rule == "fp16":
        s = b
        for h in (16, 8, 4, 2, 1):
            s = _f32(s[..., :h] + s[..., h:2 * h])
        s = s[..., 0].half().double()
        d = d.half().double()
        i = torch.where(d > 0, _f32(1.0 / d), 0.0)
        return (d[..., None] * _away(_f32(b * i[..., None])).clamp(-127, 127)).reshape(M, K), s
    s = torch.zeros_like(d)
    for j in range(32):
        s = _f32(s + b[..., j])
    if rule == "w8a8c8":
        d = torch.where(d < 1e-6, 1.0, d)
        q = _away(_f32(b / d[..., None])).clamp(-128, 127)
    elif rule == "deepseek_v2":
        d = torch.where(d > 0, d, 1.0)
        q = torch.round(_f32(b / d[..., None])).clamp(-128, 127)
    else:
        i = torch.where(d > 0, _f32(1.0 / d), 0.0)
        q = _away(_f32(b * i[..., None])).clamp(-128, 127)
        d, s = d.half().double(), s.half().double()
    return (d[..., None] * q).reshape(M, K), s


def _product(fmt, w, x, s):
    """x . W^T plus the sums' term, in slices of weight rows."""
    out = torch.empty((x.shape[0], w.shape[0]), dtype=torch.float64, device=w.device)
    step = max(1, int(6e7 // x.shape[1]))
    for r in range(0, w.shape[0], step):
        q, side = _dequant(fmt, w[r:r + step])
        if s is None:              # no activation quantisation: the plain dequantised product
            if side is not None:
                q = q + side.repeat_interleave(32, 1)
            out[:, r:r + step] = x @ q.t().contiguous()
        else:
            out[:, r:r + step] = x @ q.t().contiguous()
            if side is not None:
                out[:, r:r + step] += s @ side.t().contiguous()
    return out


def exact(case, seed):
    w, x, logits = _inputs(case, seed)
    fmt = case["weight"]
    if case["op"] == "w16":
        return _product(fmt, w, x.double(), None)
    if case["op"] == "fp16":
        return _product(fmt, w, *_quantise(x, "fp16")).t().contiguous()
    if case["op"] == "linear":
        return _product(fmt, w, *_quantise(x, case["act"]))
    N, k = case["N"], case["top_k"]
    a, s = _quantise(x, "float32")
    p = torch.softmax(logits.double(), -1)
    ids = torch.topk(logits, k, -1).indices
    p = torch.gather(p, 1, ids)
    if case["renorm"]:
        p = p / p.sum(-1, keepdim=True)
    out = torch.zeros((case["T"], N), dtype=torch.float64, device=w.device)
    for e in range(case["E"]):
        t, slot = (ids == e).nonzero(as_tuple=True)
        if t.numel():
            out.index_add_(0, t, _product(fmt, w[e * N:(e + 1) * N], a[t], s[t]) * p[t, slot][:, None])
    return out
