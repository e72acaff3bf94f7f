"""The work that users of this library have it do, as cases that can be timed.

Every case is `calls` calls of one public entry point (aiehlc_amd.Context over
the C ABI of include/miaie.h) on buffers that are already on the GPU: one
call, or, where a call is so short that a program issues several in a row (the
harness over its tiles, a server over its waiting requests), a few back to
back, each with operands of its own.  Operands are torch tensors; the context
launches on torch's current stream, as a program that mixes the two does.

A case is a dict of plain values with an "op":
  window     mm_window_i32     n x n int32 NT product of one packed A||B window
  gemm_i8    gemm_i8_rq        int8 GEMM, fused round / shift / saturate, optional
                               ReLU; acc: also the int32 accumulators
  gemm_i32   gemm_i8_i32       int8 GEMM, int32 result
  gemm_bf16  gemm_bf16_f32     bf16 GEMM, fp32 result
  mlp        mlp_i8            two chained int8 GEMMs with requant and ReLU between
  conv       conv2d_i8_nhwc    int8 NHWC convolution, per-channel requant
"""
from __future__ import annotations

import math

import torch

import aiehlc_amd as mi


# ------------------------------------------------------------------ the cases
def listed() -> list[dict]:
    return [
        # the reference harness's own call, a 16 x 16 int32 tile, on four tiles (the smallest work there is: latency)
        {"name": "window_16", "op": "window", "n": 16, "calls": 4},
        # one 64^3 int8 tile to int32, B row-major: the single-tile configuration, four requests
        {"name": "gemm_tile_64", "op": "gemm_i32", "M": 64, "N": 64, "K": 64, "nt": False, "calls": 4},
        # the headline: a large square quantized layer
        {"name": "gemm_4096", "op": "gemm_i8", "M": 4096, "N": 4096, "K": 4096, "nt": False, "shift": 10,
         "relu": False, "acc": False, "calls": 1},
        # one of eight row shards of that layer, a mid-size grid
        {"name": "gemm_shard_512", "op": "gemm_i8", "M": 512, "N": 4096, "K": 4096, "nt": False, "shift": 10,
         "relu": False, "acc": False, "calls": 1},
        # a layer whose sizes divide by no tile, weights stored [N][K], ReLU
        {"name": "gemm_ragged_nt", "op": "gemm_i8", "M": 1000, "N": 2050, "K": 1000, "nt": True, "shift": 9,
         "relu": True, "acc": False, "calls": 1},
        # the bf16 benchmark: the largest work
        {"name": "bf16_8192", "op": "gemm_bf16", "M": 8192, "N": 8192, "K": 8192, "calls": 1},
        # an ordinary bf16 layer of round decimal sizes (no tile divides them)
        {"name": "bf16_1000", "op": "gemm_bf16", "M": 1000, "N": 1000, "K": 1000, "calls": 1},
        # the chained MLP over a long batch (prefill) ...
        {"name": "mlp_prefill_2048", "op": "mlp", "M": 2048, "K": 4096, "F": 11008, "N": 4096, "s1": 11, "s2": 12,
         "calls": 1},
        # ... and over the few rows of one decoding step, where the weights are the work
        {"name": "mlp_decode_16", "op": "mlp", "M": 16, "K": 4096, "F": 11008, "N": 4096, "s1": 11, "s2": 12, "calls": 1},
        # a body layer of a convolutional network: the conv benchmark, two batches
        {"name": "conv_56", "op": "conv", "N": 8, "H": 56, "W": 56, "Cin": 64, "Cout": 64, "R": 3, "stride": 1, "pad": 1,
         "calls": 2},
        # its first layer: three input channels, a 7x7 filter, stride 2
        {"name": "conv_stem_224", "op": "conv", "N": 8, "H": 224, "W": 224, "Cin": 3, "Cout": 64, "R": 7, "stride": 2,
         "pad": 3, "calls": 1},
        # a deep layer that halves the image
        {"name": "conv_down_28", "op": "conv", "N": 8, "H": 28, "W": 28, "Cin": 256, "Cout": 256, "R": 3, "stride": 2,
         "pad": 1, "calls": 1},
    ]


# Sizes of a draw: spread over the logarithm of [lo, hi], a third of them
# multiples of 128, a third multiples of 16, the rest as they fall (odd ones
# among them).
def _size(rng, lo: int, hi: int) -> int:
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + 0.999)))
    unit = rng.choice((128, 16, 1))
    n = max(1, round(v / unit)) * unit if v >= unit else int(v)
    return min(hi, max(lo, n))


# Products of a drawn GEMM stay below those of the largest listed one of its kind.
_MAX_MACS = {"gemm_i8": 4096**3, "gemm_i32": 4096**3, "gemm_bf16": 8192**3, "mlp": 2048 * 4096 * 11008}


def draw(rng) -> dict:
    case = _draw(rng)
    # several calls in a pass where one is little more than its launch
    macs = work({**case, "calls": 1})["flops"] / 2
    case["calls"] = 4 if macs < 5e7 else 2 if macs < 2e9 else 1
    return case


def _draw(rng) -> dict:
    op = rng.choice(("window", "gemm_i8", "gemm_i8", "gemm_i32", "gemm_bf16", "gemm_bf16", "mlp", "conv", "conv", "conv"))
    if op == "window":
        return {"op": op, "n": int(math.exp(rng.uniform(math.log(17), math.log(513))))}
    if op in ("gemm_i8", "gemm_i32", "gemm_bf16"):
        while True:
            M, N, K = _size(rng, 1, 8192), _size(rng, 16, 8192), _size(rng, 16, 8192)
            if M * N * K <= _MAX_MACS[op]:
                break
        case = {"op": op, "M": M, "N": N, "K": K}
        if op != "gemm_bf16":
            case["nt"] = rng.random() < 0.5
        if op == "gemm_i8":
            # (mostly the shifts that keep the result in range, now and then any other)
            case["shift"] = rng.randint(8, 12) if rng.random() < 0.75 else rng.randint(0, 16)
            case["relu"] = rng.random() < 0.5
            case["acc"] = rng.random() < 0.2
        return case
    if op == "mlp":
        while True:
            M, K, F, N = _size(rng, 1, 2048), _size(rng, 256, 4096), _size(rng, 256, 11008), _size(rng, 256, 4096)
            if M * F * max(K, N) <= _MAX_MACS[op]:
                break
        return {"op": op, "M": M, "K": K, "F": F, "N": N, "s1": rng.randint(8, 12), "s2": rng.randint(8, 12)}
    while True:
        case = {"op": "conv", "N": rng.choice((1, 2, 4, 8, 8, 16)), "H": _size(rng, 7, 224), "Cin": 0, "Cout": 0,
                "R": rng.choice((1, 3, 3, 3, 5, 7)), "stride": rng.choice((1, 1, 2))}
        case["W"] = case["H"] if rng.random() < 0.7 else _size(rng, 7, 224)
        # image channels, channel counts of the usual multiples, and uneven ones
        case["Cin"] = rng.choice((1, 3, 3, 16, 32, 48, 64, 64, 96, 128, 128, 192, 256, 512, rng.randint(1, 256)))
        case["Cout"] = rng.choice((16, 32, 64, 64, 96, 128, 128, 192, 256, 512, rng.randint(1, 256)))
        case["pad"] = rng.choice((0, case["R"] // 2, case["R"] // 2))
        # no more than a large body layer of a batch
        if 2 * _conv_macs(case) <= 4e10 and case["H"] + 2 * case["pad"] >= case["R"] and case["W"] + 2 * case["pad"] >= case["R"]:
            return case


def _conv_out(c: dict) -> tuple[int, int]:
    return tuple((c[d] + 2 * c["pad"] - c["R"]) // c["stride"] + 1 for d in ("H", "W"))


def _conv_macs(c: dict) -> int:
    Ho, Wo = _conv_out(c)
    return c["N"] * Ho * Wo * c["Cout"] * c["R"] * c["R"] * c["Cin"]


# ------------------------------------------------------------------ inputs
def _inputs(case: dict, seed: int) -> list[dict]:
    """Operands of each call, on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return [_operands(case, g) for _ in range(case["calls"])]


def _operands(case: dict, g: torch.Generator) -> dict:

    def i8(*shape):  # the benchmark's operands: int8 uniform over the whole range
        return torch.randint(-128, 128, shape, dtype=torch.int8, device="cuda", generator=g)

    op = case["op"]
    if op == "window":  # the harness's windows hold small non-negative integers
        n = case["n"]
        return {"win": torch.randint(0, 512, (2, n, n), dtype=torch.int32, device="cuda", generator=g)}
    if op in ("gemm_i8", "gemm_i32"):
        M, N, K = case["M"], case["N"], case["K"]
        return {"A": i8(M, K), "B": i8(N, K) if case["nt"] else i8(K, N)}
    if op == "gemm_bf16":  # N(0, 1) / sqrt(K), as the benchmark draws them
        M, N, K = case["M"], case["N"], case["K"]
        s = 1.0 / math.sqrt(K)
        return {k: (torch.randn(shape, device="cuda", generator=g) * s).to(torch.bfloat16)
                for k, shape in (("A", (M, K)), ("B", (K, N)))}
    if op == "mlp":
        M, K, F, N = case["M"], case["K"], case["F"], case["N"]
        return {"X": i8(M, K), "W1": i8(K, F), "W2": i8(F, N)}
    return {"X": i8(case["N"], case["H"], case["W"], case["Cin"]),
            "W": i8(case["Cout"], case["R"], case["R"], case["Cin"]),
            "shifts": torch.randint(8, 13, (case["Cout"],), dtype=torch.uint8, device="cuda", generator=g)}


_contexts: dict[int, mi.Context] = {}


def _context() -> mi.Context:
    """The program's one context per stream."""
    stream = torch.cuda.current_stream().cuda_stream
    if stream not in _contexts:
        _contexts[stream] = mi.Context(torch.cuda.current_device(), stream=stream)
    return _contexts[stream]


def prepare(case: dict, seed: int) -> dict:
    return {"case": dict(case), "ctx": _context(), "calls": [_with_outputs(case, s) for s in _inputs(case, seed)]}


def _with_outputs(case: dict, s: dict) -> dict:
    def out(dtype, *shape):
        return torch.empty(shape, dtype=dtype, device="cuda")

    op = case["op"]
    if op == "window":
        s["C"] = out(torch.int32, case["n"], case["n"])
    elif op == "gemm_i8":
        s["Y"] = out(torch.int8, case["M"], case["N"])
        if case["acc"]:
            s["C"] = out(torch.int32, case["M"], case["N"])
    elif op == "gemm_i32":
        s["C"] = out(torch.int32, case["M"], case["N"])
    elif op == "gemm_bf16":
        s["C"] = out(torch.float32, case["M"], case["N"])
    elif op == "mlp":
        s["Hid"] = out(torch.int8, case["M"], case["F"])
        s["Y"] = out(torch.int8, case["M"], case["N"])
    else:
        Ho, Wo = _conv_out(case)
        s["Y"] = out(torch.int8, case["N"], Ho, Wo, case["Cout"])
    return s


# ------------------------------------------------------------------ one pass
def run(state: dict):
    return [_call(state["ctx"], state["case"], s) for s in state["calls"]]


def _call(ctx: mi.Context, c: dict, s: dict):
    op = c["op"]
    if op == "window":
        ctx.mm_window_i32(s["win"].data_ptr(), s["C"].data_ptr(), c["n"])
        return s["C"]
    if op == "gemm_i8":
        acc = s.get("C")
        ctx.gemm_i8_rq(s["A"].data_ptr(), s["B"].data_ptr(), s["Y"].data_ptr(), c["M"], c["N"], c["K"], c["shift"],
                       c["relu"], None if acc is None else acc.data_ptr(), mi.B_NT if c["nt"] else mi.B_NN)
        return s["Y"] if acc is None else (s["Y"], acc)
    if op == "gemm_i32":
        ctx.gemm_i8_i32(s["A"].data_ptr(), s["B"].data_ptr(), s["C"].data_ptr(), c["M"], c["N"], c["K"],
                        b_layout=mi.B_NT if c["nt"] else mi.B_NN)
        return s["C"]
    if op == "gemm_bf16":
        ctx.gemm_bf16_f32(s["A"].data_ptr(), s["B"].data_ptr(), s["C"].data_ptr(), c["M"], c["N"], c["K"])
        return s["C"]
    if op == "mlp":
        ctx.mlp_i8(s["X"].data_ptr(), s["W1"].data_ptr(), s["W2"].data_ptr(), s["Hid"].data_ptr(), s["Y"].data_ptr(),
                   c["M"], c["K"], c["F"], c["N"], c["s1"], c["s2"])
        return s["Hid"], s["Y"]
    ctx.conv2d_i8_nhwc(s["X"].data_ptr(), s["W"].data_ptr(), s["shifts"].data_ptr(), s["Y"].data_ptr(), c["N"], c["H"],
                       c["W"], c["Cin"], c["Cout"], c["R"], c["R"], c["stride"], c["pad"])
    return s["Y"]


# ------------------------------------------------------------------ what a pass cannot do without
def work(case: dict) -> dict:
    return {k: case["calls"] * v for k, v in _work(case).items()}


def _work(case: dict) -> dict:
    op = case["op"]
    if op == "window":
        n = case["n"]
        return {"bytes": 12 * n * n, "flops": 2 * n**3}
    if op in ("gemm_i8", "gemm_i32", "gemm_bf16"):
        M, N, K = case["M"], case["N"], case["K"]
        inb = 2 if op == "gemm_bf16" else 1
        outb = 5 if case.get("acc") else 1 if op == "gemm_i8" else 4
        return {"bytes": inb * (M * K + K * N) + outb * M * N, "flops": 2 * M * N * K}
    if op == "mlp":  # H is an output of the call
        M, K, F, N = case["M"], case["K"], case["F"], case["N"]
        return {"bytes": M * K + K * F + F * N + M * F + M * N, "flops": 2 * M * F * (K + N)}
    Ho, Wo = _conv_out(case)
    macs = _conv_macs(case)
    return {"bytes": case["N"] * case["H"] * case["W"] * case["Cin"] + case["Cout"] * (case["R"]**2 * case["Cin"] + 1) +
            case["N"] * Ho * Wo * case["Cout"], "flops": 2 * macs}


def tolerance(case: dict):
    """Integer paths are exact.  bf16 products are exact in fp32, so what
    differs is the fp32 sums: at K = 8192 this library's are 5.7e-7 off the
    64-bit ones (rms; 5.1e-6 at most), an fp32 library product's 9.6e-7
    (9.0e-6), and the two differ by 1.1e-6 (1.1e-5); all less at smaller K.
    About four times that is stated."""
    return {"rel": 4e-6, "max": 4e-5} if case["op"] == "gemm_bf16" else "exact"


# ------------------------------------------------------------------ the same in 64 bits
def _requant(acc: torch.Tensor, shift, relu: bool = False) -> torch.Tensor:
    """sat_int8(floor((acc + 2^(shift-1)) / 2^shift)), then ReLU; acc holds
    whole numbers below 2^53 in float64, so every step is exact."""
    shift = torch.as_tensor(shift, dtype=torch.float64, device=acc.device)
    half = torch.where(shift > 0, torch.exp2(shift - 1), torch.zeros_like(shift))
    q = torch.floor((acc + half) / torch.exp2(shift))
    return q.clamp_(0 if relu else -128, 127).to(torch.int8)


def exact(case: dict, seed: int):
    return [_exact(case, s) for s in _inputs(case, seed)]


def _exact(case: dict, s: dict):
    op = case["op"]
    if op == "window":
        return (s["win"][0].double() @ s["win"][1].double().t().contiguous()).to(torch.int32)
    if op in ("gemm_i8", "gemm_i32"):
        B = s["B"].double()
        acc = s["A"].double() @ (B.t().contiguous() if case["nt"] else B)
        if op == "gemm_i32":
            return acc.to(torch.int32)
        Y = _requant(acc, case["shift"], case["relu"])
        return (Y, acc.to(torch.int32)) if case["acc"] else Y
    if op == "gemm_bf16":
        return s["A"].double() @ s["B"].double()
    if op == "mlp":
        H = _requant(s["X"].double() @ s["W1"].double(), case["s1"], True)
        return H, _requant(H.double() @ s["W2"].double(), case["s2"])
    Ho, Wo = _conv_out(case)
    p, st = case["pad"], case["stride"]
    X = torch.nn.functional.pad(s["X"].double(), (0, 0, p, p, p, p))
    W = s["W"].double()
    acc = torch.zeros(case["N"] * Ho * Wo, case["Cout"], dtype=torch.float64, device="cuda")
    for r in range(case["R"]):
        for c in range(case["R"]):
            px = X[:, r:r + (Ho - 1) * st + 1:st, c:c + (Wo - 1) * st + 1:st, :]
            acc += px.reshape(-1, case["Cin"]) @ W[:, r, c, :].t().contiguous()
    return _requant(acc, s["shifts"].double()).reshape(case["N"], Ho, Wo, case["Cout"])
