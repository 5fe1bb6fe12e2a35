"""Performance cases of the quantized matrix multiplication path.

What a program on this backend has it do: the projections of a decoder layer
at decode (one token, a few sequences, a speculative batch) and at prefill
(ragged and full batches, up to 2048 tokens), and the expert projections of a
mixture-of-experts FFN in both, over the weight types the backend takes.
Shapes are Llama-3-8B's and Qwen3-30B-A3B's, as the benchmark and the tests
use them.

Weights are N(0, 0.02) and activations N(0, 1).  Weights are quantized here by
plain round-to-nearest into the ggml block formats.  `exact` evaluates in f64
what the operation is defined to compute: the products of the stored weights
with the activations quantized to Q8_1 (blocks of 32: f16 scale d, f16 d * sum,
int8 codes).

Decode programs keep a captured graph of the step and replay it, since the
kernels last a few microseconds; prefill programs call the operations.
"""
import math
import os
import sys

import torch

_pkg = os.path.join(os.getcwd(), "llama.zig_amd")
if _pkg not in sys.path:
    sys.path.insert(0, _pkg)

import ggml_hip as G  # noqa: E402

DEV = "cuda:0"
BLOCK_BYTES = {"Q4_K": 144, "Q5_K": 176, "Q6_K": 210, "IQ4_XS": 136, "Q8_0": 34, "Q4_0": 18}
BLOCK_WEIGHTS = {"Q4_K": 256, "Q5_K": 256, "Q6_K": 256, "IQ4_XS": 256, "Q8_0": 32, "Q4_0": 32}
IQ4_LEVELS = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)

# A model file's weight mix: the type of most matrices, and of attn_v / ffn_down.
MIXES = {"Q4_K_M": ("Q4_K", "Q6_K"), "Q5_K_M": ("Q5_K", "Q6_K"), "Q8_0": ("Q8_0", "Q8_0"),
         "Q4_0": ("Q4_0", "Q4_0"), "IQ4_XS": ("IQ4_XS", "IQ4_XS")}


def listed():
    return [
        # The smallest call: one small projection of one token, where the call's
        # own latency counts.
        {"name": "attn_k_1", "kind": "mul_mat", "type": "Q4_K", "rows": 1024, "k": 4096, "cols": 1},
        # One decode step of one sequence over four layers' projections (a
        # model's weights do not stay in the caches from layer to layer).
        {"name": "decode_1", "kind": "decode", "mix": "Q4_K_M", "d": 4096, "kv": 1024, "ff": 14336, "layers": 4,
         "cols": 1},
        # The same with four sequences served together.
        {"name": "decode_4", "kind": "decode", "mix": "Q4_K_M", "d": 4096, "kv": 1024, "ff": 14336, "layers": 4,
         "cols": 4},
        # A speculative draft of 13 tokens verified at once.
        {"name": "verify_13", "kind": "decode", "mix": "Q5_K_M", "d": 4096, "kv": 1024, "ff": 14336, "layers": 2,
         "cols": 13},
        # A prompt batch through an FFN projection: the benchmark's prefill shape.
        {"name": "ffn_512", "kind": "mul_mat", "type": "Q4_K", "rows": 14336, "k": 4096, "cols": 512},
        # The long-row projection of the same batch, in its six-bit type.
        {"name": "down_512", "kind": "mul_mat", "type": "Q6_K", "rows": 4096, "k": 14336, "cols": 512},
        # A ragged prompt batch through attention's output projection.
        {"name": "attn_333", "kind": "mul_mat", "type": "Q5_K", "rows": 4096, "k": 4096, "cols": 333},
        # A short prompt, eight-bit weights.
        {"name": "short_100", "kind": "mul_mat", "type": "Q8_0", "rows": 4096, "k": 14336, "cols": 100},
        # A long batch through the fused key / query / value rows, table-coded weights.
        {"name": "qkv_1000", "kind": "mul_mat", "type": "IQ4_XS", "rows": 6144, "k": 4096, "cols": 1000},
        # The largest: gate, up and GLU of a full 2048-token batch.
        {"name": "glu_2048", "kind": "mul_mat_glu", "type": "Q4_K", "rows": 14336, "k": 4096, "cols": 2048},
        # Decode of one token through the experts of a layer: gate / up / GLU, then down.
        {"name": "moe_1", "kind": "moe", "type": "Q4_K", "experts": 128, "d": 2048, "ff": 768, "top": 8, "cols": 1},
        # A 512-token batch through the same experts, unevenly routed.
        {"name": "moe_512", "kind": "moe", "type": "Q4_K", "experts": 128, "d": 2048, "ff": 768, "top": 8,
         "cols": 512},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    types = ("Q4_K", "Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q4_0", "IQ4_XS")  # Q4_K is the usual one
    kind = rng.choice(("mul_mat", "mul_mat", "mul_mat", "mul_mat_glu", "decode", "moe"))
    if kind == "decode":
        d = 256 * rng.randint(4, 20)
        return {"kind": kind, "mix": rng.choice(sorted(MIXES)), "d": d, "kv": 128 * rng.randint(4, 16),
                "ff": 256 * rng.randint(d // 256, 56), "layers": rng.randint(1, 3), "cols": log_int(1, 32)}
    if kind == "moe":
        return {"kind": kind, "type": rng.choice(types), "experts": rng.choice((8, 32, 64, 128)),
                "d": 256 * rng.randint(4, 12), "ff": 256 * rng.randint(2, 8), "top": rng.choice((2, 4, 8)),
                "cols": log_int(1, 512)}
    return {"kind": kind, "type": rng.choice(types), "rows": log_int(512, 14336), "k": 256 * log_int(4, 28 if kind == "mul_mat_glu" else 56),
            "cols": log_int(1, 1024)}


# ---------------------------------------------------------------- weights


def _super_scale(s, top):
    """One f16 scale for rows of block scales, as f32, its largest block at `top`."""
    d = (s.amax(-1, keepdim=True) / top).half().float()
    return d, torch.where(d > 0, (s / d.clamp_min(1e-30)), torch.zeros_like(s)).round().clamp_(0, top)


def _f16_bytes(t):
    return t.half().contiguous().view(torch.uint8)


def _quantize(qtype, w):
    """f32 [rows, k] -> (blocks uint8 [rows, row bytes], values f64 parts).  The
    parts are (positive scale per block of n, integer codes, n, min term per
    block of 32 or None): weight = scale * code - min."""
    rows, k = w.shape
    if qtype in ("Q8_0", "Q4_0"):
        x = w.view(rows, k // 32, 32)
        top = 127.0 if qtype == "Q8_0" else 8.0
        d = (x.abs().amax(-1, keepdim=True) / top).half().float()
        q = (x / d.clamp_min(1e-30)).round()
        if qtype == "Q8_0":
            q = q.clamp_(-127, 127).to(torch.int8)
            body = q.view(torch.uint8)
        else:
            q = q.clamp_(-8, 7).to(torch.int8)
            u = (q + 8).view(torch.uint8)
            body = u[..., :16] | (u[..., 16:] << 4)
        blocks = torch.cat([_f16_bytes(d), body], -1)
        return blocks.reshape(rows, -1), (d.squeeze(-1), q.view(rows, k), 32, None)
    sb = 16 if qtype == "Q6_K" else 32
    x = w.view(rows, k // 256, 256 // sb, sb)
    if qtype in ("Q4_K", "Q5_K"):
        levels = 15 if qtype == "Q4_K" else 31
        lo = (-x.amin(-1)).clamp_min(0)
        s = (x.amax(-1) + lo) / levels
        d, sc = _super_scale(s, 63)
        dm, m = _super_scale(lo, 63)
        step, off = d * sc, dm * m
        q = ((x + off.unsqueeze(-1)) / step.clamp_min(1e-30).unsqueeze(-1)).round_().clamp_(0, levels).to(torch.uint8)
        scb, mb = sc.to(torch.uint8), m.to(torch.uint8)
        packed = torch.cat([scb[..., :4] | ((scb[..., 4:] >> 4) << 6), mb[..., :4] | ((mb[..., 4:] >> 4) << 6),
                            (scb[..., 4:] & 15) | ((mb[..., 4:] & 15) << 4)], -1)
        pair = q.view(rows, k // 256, 4, 2, 32)
        low = pair & 15
        body = (low[..., 0, :] | (low[..., 1, :] << 4)).reshape(rows, k // 256, 128)
        parts = [_f16_bytes(d), _f16_bytes(dm), packed]
        if qtype == "Q5_K":
            bit = torch.arange(8, dtype=torch.uint8, device=w.device).view(8, 1)
            parts.append(((q >> 4) << bit).sum(-2, dtype=torch.uint8))
        blocks = torch.cat(parts + [body], -1)
        return blocks.reshape(rows, -1), (step.reshape(rows, -1), q.reshape(rows, k), 32, off.reshape(rows, -1))
    if qtype == "Q6_K":
        d, sc = _super_scale(x.abs().amax(-1) / 31.0, 127)
        step = d * sc
        q = (x / step.clamp_min(1e-30).unsqueeze(-1)).round_().clamp_(-32, 31).to(torch.int8)
        u = (q + 32).view(torch.uint8).view(rows, k // 256, 2, 4, 32)
        low, high = u & 15, u >> 4
        ql = torch.cat([low[..., 0, :] | (low[..., 2, :] << 4), low[..., 1, :] | (low[..., 3, :] << 4)], -1)
        qh = high[..., 0, :] | (high[..., 1, :] << 2) | (high[..., 2, :] << 4) | (high[..., 3, :] << 6)
        blocks = torch.cat([ql.reshape(rows, -1, 128), qh.reshape(rows, -1, 64), sc.to(torch.uint8), _f16_bytes(d)], -1)
        return blocks.reshape(rows, -1), (step.reshape(rows, -1), q.reshape(rows, k), 16, None)
    d, sc = _super_scale(x.abs().amax(-1) / 127.0, 31)
    step = d * sc
    levels = torch.tensor(IQ4_LEVELS, dtype=torch.float32, device=w.device)
    idx = torch.bucketize(x / step.clamp_min(1e-30).unsqueeze(-1), (levels[1:] + levels[:-1]) / 2).to(torch.uint8)
    ls = sc.to(torch.int32) + 32
    high = ((ls >> 4) << (2 * torch.arange(8, device=w.device))).sum(-1, keepdim=True)
    nib = (ls & 15).to(torch.uint8).view(rows, k // 256, 4, 2)
    blocks = torch.cat([_f16_bytes(d), torch.cat([high & 255, high >> 8], -1).to(torch.uint8),
                        nib[..., 0] | (nib[..., 1] << 4),
                        (idx[..., :16] | (idx[..., 16:] << 4)).reshape(rows, k // 256, 128)], -1)
    q = levels.to(torch.int8)[idx.long()]
    return blocks.reshape(rows, -1), (step.reshape(rows, -1), q.reshape(rows, k), 32, None)


def _matrix(gen, qtype, rows, k):
    return _quantize(qtype, torch.randn((rows, k), generator=gen, device=DEV).mul_(0.02))


def _experts(gen, qtype, n, rows, k):
    parts = [_matrix(gen, qtype, rows, k) for _ in range(n)]
    return torch.stack([p[0] for p in parts]), [p[1] for p in parts]


def _columns(gen, cols, k):
    return torch.randn((cols, k), generator=gen, device=DEV)


# ---------------------------------------------------------------- inputs


def _inputs(case, seed):
    """Every call of one pass: (operation, quantized weights with their f64
    parts, activations, routing)."""
    gen = torch.Generator(DEV).manual_seed(seed)
    kind, n = case["kind"], case["cols"]
    if kind == "mul_mat":
        w = _matrix(gen, case["type"], case["rows"], case["k"])
        yield "mul_mat", case["type"], (w,), _columns(gen, n, case["k"]), None
    elif kind == "mul_mat_glu":
        w = [_matrix(gen, case["type"], case["rows"], case["k"]) for _ in range(2)]
        yield "mul_mat_glu", case["type"], w, _columns(gen, n, case["k"]), None
    elif kind == "decode":
        d, kv, ff = case["d"], case["kv"], case["ff"]
        most, some = MIXES[case["mix"]]
        for _ in range(case["layers"]):
            x = _columns(gen, n, d)
            for t, rows in ((most, d), (most, kv), (some, kv)):  # q, k, v
                yield "mul_mat", t, (_matrix(gen, t, rows, d),), x, None
            yield "mul_mat", most, (_matrix(gen, most, d, d),), _columns(gen, n, d), None  # o
            w = [_matrix(gen, most, ff, d) for _ in range(2)]
            yield "mul_mat_glu", most, w, _columns(gen, n, d), None
            yield "mul_mat", some, (_matrix(gen, some, d, ff),), _columns(gen, n, ff), None  # down
    else:
        d, ff, e, t = case["d"], case["ff"], case["experts"], case["type"]
        ids = torch.randn((n, e), generator=gen, device=DEV).topk(case["top"], -1).indices.int().contiguous()
        w = [_experts(gen, t, e, ff, d) for _ in range(2)]
        yield "mul_mat_id_glu", t, w, _columns(gen, n, d).view(n, 1, d), ids
        w = _experts(gen, t, e, d, ff)
        yield "mul_mat_id", t, (w,), _columns(gen, n * case["top"], ff).view(n, case["top"], ff), ids


def _captured(case):
    return case["kind"] == "decode" or (case["kind"] == "moe" and case["cols"] <= 8)


def _call(op, qtype, w, x, ids):
    if op == "mul_mat":
        return G.mul_mat(qtype, w[0], x)
    if op == "mul_mat_glu":
        return G.mul_mat_glu(qtype, w[0], w[1], x, glu="SWIGLU")
    if op == "mul_mat_id":
        return G.mul_mat_id(qtype, w[0], x, ids)
    return G.mul_mat_id_glu(qtype, w[0], w[1], x, ids, glu="SWIGLU")


def prepare(case, seed):
    calls = [(op, t, [m[0] for m in w], x, ids) for op, t, w, x, ids in _inputs(case, seed)]
    state = {"calls": calls, "graph": None, "out": None}
    if _captured(case):
        G.lib()
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["out"] = [_call(*c) for c in calls]
    return state


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
        return state["out"]
    return [_call(*c) for c in state["calls"]]


# ---------------------------------------------------------------- cost and values


def _products(case):
    """(type, rows, k, matrices read, columns computed, activation rows read,
    output rows written, products per column) of each call."""
    kind, n = case["kind"], case["cols"]
    if kind in ("mul_mat", "mul_mat_glu"):
        m = 2 if kind == "mul_mat_glu" else 1
        return [(case["type"], case["rows"], case["k"], m, n, n, n, m)]
    if kind == "decode":
        d, kv, ff = case["d"], case["kv"], case["ff"]
        most, some = MIXES[case["mix"]]
        one = [(most, d, d, 1, n, n, n, 1), (most, kv, d, 1, n, 0, n, 1), (some, kv, d, 1, n, 0, n, 1),
               (most, d, d, 1, n, n, n, 1), (most, ff, d, 2, n, n, n, 2), (some, d, ff, 1, n, n, n, 1)]
        return one * case["layers"]
    d, ff, e, top = case["d"], case["ff"], case["experts"], min(case["top"], case["experts"])
    used = e * (1.0 - (1.0 - top / e) ** n)  # experts that some token picks, on average
    return [(case["type"], ff, d, 2 * used, n * top, n, n * top, 2),
            (case["type"], d, ff, used, n * top, n * top, n * top, 1)]


def work(case):
    by = fl = 0.0
    for t, rows, k, mats, cols, xr, outs, per in _products(case):
        by += mats * rows * (k // BLOCK_WEIGHTS[t]) * BLOCK_BYTES[t] + 4.0 * (xr * k + outs * rows)
        fl += 2.0 * rows * k * cols * per
    return {"bytes": by, "flops": fl}


def tolerance(case):
    # Integer block products are exact; what differs between implementations is
    # the order of the f32 sums (and the exponential of the GLU): against the
    # f64 values at most 2.9e-7 and 4.2e-6 over these cases and 24 drawn ones.
    return {"rel": 1.2e-6, "max": 1.7e-5}


def _q8_1(x):
    """f32 [n, k] -> f64 (d * code [n, k], s [n, k / 32]) of the Q8_1 blocks: d and
    s = d * sum(codes) in f16, codes rounded half away from zero in f32 (the
    quotients go through f64, whose rounding to f32 is the f32 division's)."""
    n, k = x.shape
    b = x.view(n, k // 32, 32)
    d = (b.abs().amax(-1, keepdim=True).double() / 127.0).float()
    inv = torch.where(d > 0, 1.0 / d.double(), 0.0).float()
    v = (b * inv).double()
    q = torch.copysign((v.abs() + 0.5).floor_(), v).clamp_(-127, 127)
    s = (q.sum(-1, keepdim=True).float() * d).half().double()
    return (q * d.half().double()).view(n, k), s.view(n, -1)


def _product(parts, y, s):
    """f64 [n, rows] of one matrix's parts with Q8_1 columns."""
    step, q, nb, off = parts
    w = q.double() * step.double().repeat_interleave(nb, -1)
    out = y @ w.t()
    return out if off is None else out - s @ off.double().t()


def _glu(g, u):
    return g / (1.0 + torch.exp(-g)) * u


def exact(case, seed):
    out = []
    for op, t, w, x, ids in _inputs(case, seed):
        y, s = _q8_1(x.reshape(-1, x.shape[-1]))
        if ids is None:
            p = [_product(m[1], y, s) for m in w]
        else:
            n, top = ids.shape
            slot = torch.arange(n * top, device=DEV).view(n, top)
            src = slot if x.shape[1] == top else slot // top  # the activation row of each (token, slot)
            p = [torch.zeros((n * top, m[0].shape[1]), dtype=torch.float64, device=DEV) for m in w]
            for e in range(w[0][0].shape[0]):
                pick = (ids == e).nonzero(as_tuple=True)
                if pick[0].numel():
                    for i, m in enumerate(w):
                        p[i][slot[pick]] = _product(m[1][e], y[src[pick]], s[src[pick]])
            p = [v.view(n, top, -1) for v in p]
        out.append(_glu(p[1], p[0]) if len(p) == 2 else p[0])
    return out
