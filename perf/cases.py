"""The work that a program built on `candle_amd` has it do, as a list of measurable cases.

Every case goes through the public entry points: `QMatMul.forward` and its fused and shared-input forms, the grouped
expert calls, `QTensor.quantize` / `data` and `QTensor.dequantize[_f16]`.  A case is a dict of plain values; `kind`
says which of the five programs below it runs:

  forward     one projection on some activation rows: single-token decode (1 row), batched decode and draft
              verification (a few to some dozen rows), prompts (up to thousands of rows)
  step        the projections of a decode step over some decoder layers and the output head, either one call per
              projection (the model code as it stands) or with the fused and shared-input calls
  experts     the feed-forward block of a mixture-of-experts layer, two experts per token
  quantize    a checkpoint tensor quantized and brought back as GGML blocks, as a conversion program does
  dequantize  a quantized tensor brought back to f32 or f16 on the device

Weights are N(0, 0.02) with rows of unequal magnitude; activations are N(0, 1) with 1 % of the positions at eight
times that, the distribution of transformer activations that the prefill configuration is quoted on.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from candle_amd import qhip
from candle_amd.quantized import GgmlDType, QMatMul, QTensor

# block elements, bytes per block
BLOCKS = {"Q4_0": (32, 18), "Q4_1": (32, 20), "Q5_0": (32, 22), "Q5_1": (32, 24), "Q8_0": (32, 34),
          "Q2K": (256, 84), "Q3K": (256, 110), "Q4K": (256, 144), "Q5K": (256, 176), "Q6K": (256, 210)}
# how often the draws take each type: what checkpoints are mostly stored in first
OFTEN = {"Q4K": 5, "Q6K": 3, "Q8_0": 3, "Q4_0": 3, "Q5K": 2, "Q3K": 1, "Q2K": 1, "Q5_0": 1, "Q4_1": 1, "Q5_1": 1}
EPS = 1e-5
# no drawn projection costs more than the largest listed one
MOST_FLOPS = 2 * 4096 * 11008 * 4096


def listed():
    return [
        # one attention projection of a 7B-shaped model for one token: the smallest call there is in earnest
        {"name": "decode_q4k", "kind": "forward", "dtype": "Q4K", "n": 4096, "k": 4096, "rows": 1},
        # the projections of one token through 8 of the 32 layers and the output head, a call per projection
        {"name": "decode_step", "kind": "step", "layers": 8, "hidden": 4096, "kv": 4096, "ffn": 11008, "vocab": 32000,
         "dtype": "Q4K", "down": "Q6K", "head": "Q6K", "rows": 1, "fused": False},
        # the same for a grouped-query model with its norms and gates, four sequences at a time, fused calls
        {"name": "decode_step_fused", "kind": "step", "layers": 8, "hidden": 4096, "kv": 1024, "ffn": 14336,
         "vocab": 32000, "dtype": "Q4K", "down": "Q6K", "head": "Q6K", "rows": 4, "fused": True},
        # batched decode: eight sequences
        {"name": "batch_q4k_8", "kind": "forward", "dtype": "Q4K", "n": 11008, "k": 4096, "rows": 8},
        # verification of drafted tokens: an odd number of rows between the decode and the prompt sizes
        {"name": "verify_q8_0_21", "kind": "forward", "dtype": "Q8_0", "n": 14336, "k": 4096, "rows": 21},
        # the prefill configuration: 512 prompt tokens on the up-projection
        {"name": "prefill_q4k_512", "kind": "forward", "dtype": "Q4K", "n": 14336, "k": 4096, "rows": 512},
        # a prompt of odd length on the down-projection
        {"name": "prefill_q6k_1003", "kind": "forward", "dtype": "Q6K", "n": 4096, "k": 14336, "rows": 1003},
        # a long prompt: the largest projection
        {"name": "prefill_q4k_4096", "kind": "forward", "dtype": "Q4K", "n": 11008, "k": 4096, "rows": 4096},
        # a vocabulary and a row length that are no multiple of any tile, in a type whose blocks allow it
        {"name": "prefill_q4_0_ragged", "kind": "forward", "dtype": "Q4_0", "n": 32003, "k": 3200, "rows": 77},
        # the expert configuration: 8 experts, 64 tokens, top-2
        {"name": "experts_64", "kind": "experts", "experts": 8, "tokens": 64, "hidden": 4096, "ffn": 14336,
         "dtype": "Q4K", "down": "Q6K"},
        # conversion of a checkpoint tensor
        {"name": "quantize_q4k", "kind": "quantize", "dtype": "Q4K", "n": 11008, "k": 4096},
        # an output head brought back to f16
        {"name": "dequantize_q6k", "kind": "dequantize", "dtype": "Q6K", "n": 32000, "k": 4096, "f16": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _type(rng):
    return rng.choices(list(OFTEN), list(OFTEN.values()))[0]


def _whole(v, step):
    return max(step, v // step * step)


def _row_length(rng, dtype, hi=16384):
    """K-quants take rows of whole 256-element blocks; the 32-element types any even number of blocks, as
    their dot products over pairs of blocks want it."""
    k = _log(rng, 512, hi)
    return _whole(k, 256 if BLOCKS[dtype][0] == 256 or rng.random() < 0.5 else 64)


def _row_count(rng, hi=32768):
    """Mostly whole tiles as model dimensions are, a part of them odd as vocabularies are."""
    return _whole(_log(rng, 256, hi), rng.choice([256, 256, 32, 1]))


def draw(rng):
    kind = rng.choices(["forward", "step", "experts", "quantize", "dequantize"], [11, 2, 3, 2, 2])[0]
    dtype = _type(rng)
    if kind == "forward":
        n, k = _row_count(rng), _row_length(rng, dtype)
        return {"kind": kind, "dtype": dtype, "n": n, "k": k, "rows": min(_log(rng, 1, 4096), MOST_FLOPS // (2 * n * k))}
    if kind == "step":
        hidden = _whole(_log(rng, 1024, 5120), 256)
        return {"kind": kind, "layers": rng.randint(1, 8), "hidden": hidden, "kv": hidden // rng.choice([1, 2, 4]),
                "ffn": _whole(int(hidden * rng.uniform(2.5, 3.5)), 256), "vocab": rng.randint(1000, 32000),
                "dtype": dtype, "down": _type(rng), "head": _type(rng), "rows": _log(rng, 1, 8), "fused": rng.random() < 0.5}
    if kind == "experts":
        plain = [t for t in OFTEN if t not in ("Q4_1", "Q5_1", "Q2K")]   # the grouped calls take types without offsets
        hidden = _whole(_log(rng, 1024, 4096), 256)
        return {"kind": kind, "experts": 8, "tokens": _log(rng, 1, 256), "hidden": hidden,
                "ffn": _whole(int(hidden * rng.uniform(1.5, 3.5)), 256), "dtype": rng.choice(plain), "down": rng.choice(plain)}
    n, k = _row_count(rng, 16384), _row_length(rng, dtype, 8192)
    if kind == "quantize":
        return {"kind": kind, "dtype": dtype, "n": min(n, 11008 * 4096 // k), "k": k}
    return {"kind": kind, "dtype": dtype, "n": n, "k": k, "f16": rng.random() < 0.5}


# ---- inputs -------------------------------------------------------------------------------------------------------
def _dense(g, n, k):
    w = torch.randn(n, k, generator=g, device="cuda").mul_(0.02)
    return w.mul_(torch.rand(n, 1, generator=g, device="cuda").add_(0.5))


def _weight(g, dtype, n, k):
    return QTensor.quantize(_dense(g, n, k), GgmlDType[dtype])


def _matmul(g, dtype, n, k):
    return QMatMul.from_qtensor(_weight(g, dtype, n, k))


def _rows(g, *shape):
    x = torch.randn(*shape, generator=g, device="cuda")
    big = torch.rand(*shape, generator=g, device="cuda") < 0.01
    return torch.where(big, x.sign() * 8.0, x)


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "forward":
        s["w"] = _matmul(g, case["dtype"], case["n"], case["k"])
        s["x"] = _rows(g, 1, case["rows"], case["k"])
    elif kind == "step":
        h, kv, ffn, rows, dt = case["hidden"], case["kv"], case["ffn"], case["rows"], case["dtype"]
        s["layers"] = [{"q": _matmul(g, dt, h, h), "k": _matmul(g, dt, kv, h), "v": _matmul(g, dt, kv, h),
                        "o": _matmul(g, dt, h, h), "gate": _matmul(g, dt, ffn, h), "up": _matmul(g, dt, ffn, h),
                        "down": _matmul(g, case["down"], h, ffn),
                        "attn_norm": torch.rand(h, generator=g, device="cuda").add_(0.5),
                        "ffn_norm": torch.rand(h, generator=g, device="cuda").add_(0.5),
                        # what the attention and the residual stream leave for this layer's projections
                        "x": _rows(g, rows, 1, h), "attn": _rows(g, rows, 1, h), "mid": _rows(g, rows, 1, h),
                        "act": _rows(g, rows, 1, ffn)} for _ in range(case["layers"])]
        s["head"] = _matmul(g, case["head"], case["vocab"], h)
        s["norm"] = torch.rand(h, generator=g, device="cuda").add_(0.5)
        s["last"] = _rows(g, rows, 1, h)
    elif kind == "experts":
        e, t, h, ffn = case["experts"], case["tokens"], case["hidden"], case["ffn"]
        for name, dt, n, k in (("w1", case["dtype"], ffn, h), ("w3", case["dtype"], ffn, h), ("w2", case["down"], h, ffn)):
            s[name] = [_weight(g, dt, n, k).weight for _ in range(e)]
        s["x"] = _rows(g, t, h)
        p, chosen = torch.softmax(torch.randn(t, e, generator=g, device="cuda"), 1).topk(2, 1)
        p = p / p.sum(1, keepdim=True)
        order = chosen.reshape(-1).argsort(stable=True)   # token-major slots, sorted by expert
        s["row_ids"] = (order // 2).to(torch.int32)
        s["share"] = p.reshape(-1)[order].contiguous()
        count = torch.bincount(chosen.reshape(-1), minlength=e).cpu().numpy()
        s["offsets"] = np.concatenate([[0], count.cumsum()]).astype(np.int32)
        s["workspace"] = qhip.Workspace()
    elif kind == "quantize":
        s["dense"] = _dense(g, case["n"], case["k"])
    else:
        s["w"] = _weight(g, case["dtype"], case["n"], case["k"])
    return s


# ---- one pass -----------------------------------------------------------------------------------------------------
def _step(s):
    out = []
    for L in s["layers"]:
        out += [L["q"].forward(L["x"]), L["k"].forward(L["x"]), L["v"].forward(L["x"]), L["o"].forward(L["attn"]),
                L["gate"].forward(L["mid"]), L["up"].forward(L["mid"]), L["down"].forward(L["act"])]
    out.append(s["head"].forward(s["last"]))
    return out


def _step_fused(s):
    out = []
    for L in s["layers"]:
        out += QMatMul.forward_multi([L["q"], L["k"], L["v"]], L["x"], alpha=L["attn_norm"], eps=EPS)
        out.append(L["o"].forward(L["attn"]))
        gate, up = QMatMul.forward_multi([L["gate"], L["up"]], L["mid"], alpha=L["ffn_norm"], eps=EPS)
        out += [gate, up, L["down"].forward_silu_mul(gate, up)]
    out.append(s["head"].forward_rms_norm(s["last"], s["norm"], EPS))
    return out


def _experts(s):
    ws = s["workspace"]
    gate = qhip.qmatmul_grouped(s["w1"], s["x"], s["row_ids"], s["offsets"], workspace=ws)
    # the rows that w1's call quantized are still in the workspace
    up = qhip.qmatmul_grouped(s["w3"], s["x"], s["row_ids"], s["offsets"], flags=qhip.FLAG_REUSE_ACT, workspace=ws)
    y = qhip.qmatmul_grouped(s["w2"], gate, None, s["offsets"], workspace=ws, pre=qhip.PRE_SILU_MUL, aux=up)
    return qhip.moe_scatter_add(y, s["row_ids"], s["share"], s["case"]["tokens"])


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "forward":
        return state["w"].forward(state["x"])
    if kind == "step":
        return _step_fused(state) if case["fused"] else _step(state)
    if kind == "experts":
        return _experts(state)
    if kind == "quantize":
        return QTensor.quantize(state["dense"], GgmlDType[case["dtype"]]).data()
    return state["w"].dequantize_f16() if case["f16"] else state["w"].dequantize()


# ---- what a pass cannot do without ----------------------------------------------------------------------------------
def _ggml(dtype, n, k):
    block, size = BLOCKS[dtype]
    return n * k // block * size


def _projection(dtype, n, k, rows):
    return _ggml(dtype, n, k) + 4 * rows * (n + k), 2 * rows * n * k


def work(case):
    kind = case["kind"]
    if kind == "forward":
        b, f = _projection(case["dtype"], case["n"], case["k"], case["rows"])
    elif kind == "step":
        h, kv, ffn, rows, dt = case["hidden"], case["kv"], case["ffn"], case["rows"], case["dtype"]
        parts = [_projection(dt, n, h, rows) for n in (h, kv, kv, h, ffn, ffn)] + [_projection(case["down"], h, ffn, rows)]
        b0, f0 = _projection(case["head"], case["vocab"], h, rows)
        b = case["layers"] * sum(p[0] for p in parts) + b0
        f = case["layers"] * sum(p[1] for p in parts) + f0
    elif kind == "experts":
        e, t, h, ffn = case["experts"], case["tokens"], case["hidden"], case["ffn"]
        used = e * (1 - (1 - 2 / e) ** t)   # experts that some token chose, on average
        b = used * (2 * _ggml(case["dtype"], ffn, h) + _ggml(case["down"], h, ffn)) + 8 * t * h
        f = 2 * (2 * t) * 3 * h * ffn
    elif kind == "quantize":
        b, f = 4 * case["n"] * case["k"] + _ggml(case["dtype"], case["n"], case["k"]), 0
    else:
        b, f = (2 if case["f16"] else 4) * case["n"] * case["k"] + _ggml(case["dtype"], case["n"], case["k"]), 0
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Block integers are the same everywhere; the f32 sums over a row's blocks may be taken in another order.  A step
    in front of the quantizer (rms_norm, silu * mul) moves its input by rounding, which tips a few quants by one unit."""
    if case["kind"] in ("quantize", "dequantize"):
        return "exact"
    if case["kind"] == "experts" or case.get("fused"):
        return {"rel": 2e-3}
    return {"rel": 1e-5}
