"""Timed workloads of the matmul path: what each one is, its inputs, one pass through the public
API, the work it cannot do without, and the result in 64 bits.

A case is a dict of plain values with a ``kind``; ``listed()`` holds the fixed ones and ``draw``
makes more of the same kinds over the ranges that they stand for.  The sizes of the listed cases
are those of the repository's benchmark and shape sweep, or generic.
"""
from __future__ import annotations

import math

import torch

import metalblas_amd as mb

DEVICE = "cuda"

DTYPES = {
    "bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "c64": torch.complex64,
    "i8": torch.int8, "i16": torch.int16, "i32": torch.int32, "i64": torch.int64,
}
BYTES = {"bf16": 2, "f16": 2, "f32": 4, "c64": 8, "i8": 1, "i16": 2, "i32": 4, "i64": 8}

# The largest drawn case: 2 * 8192^3 bf16 operations, and for the types with slower matrix
# instructions the operations that take at most as long.
MAX_MNK = {"bf16": 8192 ** 3, "f16": 8192 ** 3, "f32": 2048 * 4096 * 4096, "c64": 2048 ** 3, "i8": 8192 * 4096 * 4096}


def listed():
    return [
        # integer bookkeeping (counts, index products): one small launch, all latency
        {"name": "i32_gemm_256", "kind": "gemm", "dtype": "i32", "M": 256, "N": 256, "K": 256, "layout": "rr"},
        # decoding one token: a square projection, weights stored (out, in)
        {"name": "bf16_mv_4096", "kind": "mv", "dtype": "bf16", "M": 4096, "K": 4096},
        # decoding one token: the vocabulary head, weights stored (in, out)
        {"name": "bf16_head_32000x4096", "kind": "gemm", "dtype": "bf16", "M": 1, "N": 32000, "K": 4096, "layout": "rr"},
        # decoding eight sequences at once against a large weight matrix
        {"name": "bf16_batch8_16384", "kind": "gemm", "dtype": "bf16", "M": 8, "N": 16384, "K": 16384, "layout": "rr"},
        # training step of a linear layer: forward with bias, gradient of the input, of the weights
        {"name": "bf16_linear_2048x4096x2048", "kind": "linear", "dtype": "bf16", "M": 2048, "N": 2048, "K": 4096},
        # large square product: prefill and training at full size
        {"name": "bf16_gemm_8192", "kind": "gemm", "dtype": "bf16", "M": 8192, "N": 8192, "K": 8192, "layout": "rr"},
        # sizes that no tile divides and rows that no vector load aligns with
        {"name": "bf16_odd_1023", "kind": "gemm", "dtype": "bf16", "M": 1023, "N": 1023, "K": 1023, "layout": "rr"},
        # attention's two batched products: scores = Q K^T, output = P V
        {"name": "f16_attention_32x1024x128", "kind": "attention", "dtype": "f16", "B": 32, "S": 1024, "D": 128},
        # Gram matrix / weight gradient of a narrow layer over a long sequence: deep K, small output
        {"name": "f16_deepk_128x128x65536", "kind": "gemm", "dtype": "f16", "M": 128, "N": 128, "K": 65536, "layout": "rr"},
        # single precision: numerical code, optimiser preconditioners
        {"name": "f32_gemm_2048", "kind": "gemm", "dtype": "f32", "M": 2048, "N": 2048, "K": 2048, "layout": "rr"},
        # complex: spectral operators, one operand conjugated
        {"name": "c64_gemm_2048", "kind": "gemm", "dtype": "c64", "M": 2048, "N": 2048, "K": 2048, "layout": "rr",
         "conj_a": True},
        # 8-bit integers, torch's wrapping result
        {"name": "i8_gemm_4096", "kind": "gemm", "dtype": "i8", "M": 4096, "N": 4096, "K": 4096, "layout": "rr"},
    ]


def _log_size(rng, lo, hi, odd=0.3):
    """A size spread over the logarithm of [lo, hi]: mostly multiples of 64 (or of 8 when small),
    a share of arbitrary, odd ones among them."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    if rng.random() < odd:
        return max(lo, min(hi, int(v) | 1))
    unit = 64 if v >= 256 else 8
    return max(lo, min(hi, int(round(v / unit)) * unit))


def draw(rng):
    kind = rng.choice(["small_int", "mv", "head", "thin", "linear", "gemm", "odd", "attention", "deepk", "f32", "c64", "i8"])
    layout = rng.choice(["rr", "rr", "rc", "cr", "cc"])
    half = rng.choice(["bf16", "bf16", "f16"])
    if kind == "small_int":
        return {"kind": "gemm", "dtype": rng.choice(["i16", "i32", "i32", "i64"]), "M": _log_size(rng, 64, 512),
                "N": _log_size(rng, 64, 512), "K": _log_size(rng, 64, 512), "layout": layout}
    if kind == "mv":
        return {"kind": "mv", "dtype": half, "M": _log_size(rng, 1024, 16384, 0.2), "K": _log_size(rng, 1024, 16384, 0.2)}
    if kind == "head":
        return {"kind": "gemm", "dtype": half, "M": 1, "N": _log_size(rng, 4096, 65536, 0.2),
                "K": _log_size(rng, 1024, 8192, 0.2), "layout": "rr"}
    if kind == "thin":
        return {"kind": "gemm", "dtype": half, "M": rng.randint(2, 32), "N": _log_size(rng, 2048, 16384, 0.2),
                "K": _log_size(rng, 2048, 16384, 0.2), "layout": rng.choice(["rr", "rr", "rc"])}
    if kind == "linear":
        return {"kind": "linear", "dtype": half, "M": _log_size(rng, 256, 4096), "N": _log_size(rng, 1024, 4096, 0),
                "K": _log_size(rng, 1024, 4096, 0)}
    if kind == "odd":
        return {"kind": "gemm", "dtype": half, "M": _log_size(rng, 257, 4097, 1), "N": _log_size(rng, 257, 4097, 1),
                "K": _log_size(rng, 257, 4097, 1), "layout": "rr"}
    if kind == "attention":
        s = _log_size(rng, 128, 1024)
        return {"kind": "attention", "dtype": half, "B": min(rng.choice([8, 16, 32, 48, 96, 192]), 32 * 1024 * 1024 // (s * s)),
                "S": s, "D": rng.choice([64, 128])}
    if kind == "deepk":
        return {"kind": "gemm", "dtype": half, "M": _log_size(rng, 32, 256), "N": _log_size(rng, 32, 256),
                "K": _log_size(rng, 8192, 65536), "layout": rng.choice(["rr", "cr"])}
    dtype = {"gemm": half, "f32": "f32", "c64": "c64", "i8": "i8"}[kind]
    lo, hi = {"gemm": (128, 8192), "f32": (512, 4096), "c64": (256, 2048), "i8": (512, 8192)}[kind]
    case = {"kind": "gemm", "dtype": dtype, "layout": layout}
    for d in "MNK":
        case[d] = _log_size(rng, lo, hi)
    while case["M"] * case["N"] * case["K"] > MAX_MNK[dtype]:
        big = max("MNK", key=lambda d: case[d])
        case[big] = max(lo, case[big] // 2)
    if dtype == "c64":
        case["conj_a"], case["conj_b"] = rng.random() < 0.5, rng.random() < 0.3
    return case


def _values(shape, dtype, g, scale=1.0):
    """Operand values: N(0, scale^2), or for the integer types the full 8-bit range, 15-bit values
    for the wider ones (their sums wrap in 16 bits and stay exact in double)."""
    if dtype == torch.int8:
        return torch.randint(-128, 128, shape, dtype=dtype, device=DEVICE, generator=g)
    if not (dtype.is_floating_point or dtype.is_complex):
        return torch.randint(-16384, 16384, shape, dtype=dtype, device=DEVICE, generator=g)
    t = torch.randn(shape, dtype=torch.float32 if dtype.is_floating_point else dtype, device=DEVICE, generator=g)
    return (t * scale).to(dtype)


def _matrix(rows, cols, dtype, g, layout, scale=1.0):
    """A rows x cols matrix stored row-major ("r") or as the transposed view of a row-major one."""
    if layout == "r":
        return _values((rows, cols), dtype, g, scale)
    return _values((cols, rows), dtype, g, scale).t()


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    dtype, kind = DTYPES[case["dtype"]], case["kind"]
    state = {"case": case}
    if kind == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        state["a"] = _matrix(M, K, dtype, g, case["layout"][0])
        state["b"] = _matrix(K, N, dtype, g, case["layout"][1], 1.0 if M > 32 else K ** -0.5)
    elif kind == "mv":
        state["w"] = _values((case["M"], case["K"]), dtype, g, case["K"] ** -0.5)
        state["x"] = _values((case["K"],), dtype, g)
    elif kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        state["x"] = _values((M, K), dtype, g)
        state["w"] = _values((K, N), dtype, g, K ** -0.5)
        state["bias"] = _values((N,), dtype, g)
        state["dy"] = _values((M, N), dtype, g)
    else:
        B, S, D = case["B"], case["S"], case["D"]
        state["q"] = _values((B, S, D), dtype, g, D ** -0.5)
        state["k"] = _values((B, S, D), dtype, g)
        state["v"] = _values((B, S, D), dtype, g)
        state["p"] = torch.softmax(torch.randn((B, S, S), device=DEVICE, generator=g), dim=-1).to(dtype)
    return state


def _operands(state):
    """A and B of a plain product, with the lazy conjugations that the case asks for."""
    a, b, case = state["a"], state["b"], state["case"]
    return a.conj() if case.get("conj_a") else a, b.conj() if case.get("conj_b") else b


def run(state):
    kind = state["case"]["kind"]
    if kind == "gemm":
        a, b = _operands(state)
        return mb.matmul(a, b)
    if kind == "mv":
        return mb.mv(state["w"], state["x"])
    if kind == "linear":
        x, w, dy = state["x"], state["w"], state["dy"]
        return {"y": mb.addmm(state["bias"], x, w), "dx": mb.matmul(dy, w.t()), "dw": mb.matmul(x.t(), dy)}
    return {"scores": mb.bmm(state["q"], state["k"].transpose(1, 2)), "out": mb.bmm(state["p"], state["v"])}


def work(case):
    es, kind = BYTES[case["dtype"]], case["kind"]
    if kind == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": es * (M * K + K * N + M * N), "flops": (8 if case["dtype"] == "c64" else 2) * M * N * K}
    if kind == "mv":
        M, K = case["M"], case["K"]
        return {"bytes": es * (M * K + K + M), "flops": 2 * M * K}
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": es * (2 * M * K + 2 * K * N + 2 * M * N + N), "flops": 6 * M * N * K}
    B, S, D = case["B"], case["S"], case["D"]
    return {"bytes": es * B * (4 * S * D + 2 * S * S), "flops": 4 * B * S * S * D}


def tolerance(case):
    """Four times the distance from the 64-bit result: one rounding of the output for the 16-bit
    types (2^-9 and 2^-12 at most, 1.7e-3 and 2.1e-4 in the 2-norm), the rounding of the sums for
    the 32-bit ones (1.2e-6 at K = 4096, growing with its square root)."""
    dtype = case["dtype"]
    if dtype in ("bf16", "f16"):
        return {"rel": 7e-3 if dtype == "bf16" else 9e-4}
    if dtype in ("f32", "c64"):
        return {"rel": 5e-6}
    return "exact"


def _wide(t):
    return t.to(torch.complex128 if t.is_complex() else torch.float64).contiguous()


def exact(case, seed):
    state, kind = prepare(case, seed), case["kind"]
    if kind == "gemm":
        a, b = _operands(state)
        r = torch.matmul(_wide(a.resolve_conj()), _wide(b.resolve_conj()))
        if r.is_complex() or state["a"].is_floating_point():
            return r
        # integer sums are below 2^53, so exact in double; the result wraps to the operand type
        return r.to(torch.int64).to(state["a"].dtype)
    if kind == "mv":
        return torch.mv(_wide(state["w"]), _wide(state["x"]))
    if kind == "linear":
        x, w, dy = _wide(state["x"]), _wide(state["w"]), _wide(state["dy"])
        return {"y": torch.addmm(_wide(state["bias"]), x, w), "dx": torch.matmul(dy, w.t().contiguous()),
                "dw": torch.matmul(x.t().contiguous(), dy)}
    q, k, v, p = (_wide(state[n]) for n in ("q", "k", "v", "p"))
    return {"scores": torch.bmm(q, k.transpose(1, 2).contiguous()), "out": torch.bmm(p, v)}
