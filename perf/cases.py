"""The work that users of moye_hip have it do, as timed cases: `gemm!` from a 256-cube with the reference's arithmetic to an
fp8 8192-cube and a linear layer's training step, `copyto!` as transposition, permutation and conversion, and the
element-wise operations around them.  Everything goes through the package's public entry points.

A case is a dict of plain values; its "op" says which of the families below it belongs to.  `listed()` names the cases that
are always looked at, `draw()` gives more of the same ranges.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "moye.jl_amd"))  # the package of the working folder, whose root this runs in

import moye_hip as mh  # noqa: E402
from moye_hip import _lib  # noqa: E402
from moye_hip.torch_interop import current_stream, tensor_of  # noqa: E402

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "fp8": torch.float8_e4m3fn}
BYTES = {"f32": 4, "f16": 2, "bf16": 2, "fp8": 1}
ATOM = {"f32": mh.MFMA_F32_16x16x4_F32, "f16": mh.MFMA_F32_16x16x32_F16, "bf16": mh.MFMA_F32_16x16x32_BF16,
        "fp8": mh.MFMA_F32_16x16x32_FP8}


def listed():
    return [
        # The reference's own arithmetic (UniversalFMA) on column-major arrays, a 32x32x8 tile: the smallest configuration
        # of the benchmark, what a user checks a layout or a kernel against.  Latency and launch count.
        {"name": "fma_f32_256", "op": "fma", "M": 256, "N": 256, "K": 256, "dtype": "f32"},
        # A small matrix-core product with everything left to the library: attention-sized or test-sized calls that come in
        # great numbers.  Latency, host work.
        {"name": "gemm_f16_384x640x512", "op": "gemm", "M": 384, "N": 640, "K": 512, "dtype": "f16", "out": "f16"},
        # Decoding with a batch of 16: the benchmark's short-M problem, bound by reading the weight.
        {"name": "decode_bf16_16x8192x8192", "op": "gemm", "M": 16, "N": 8192, "K": 8192, "dtype": "bf16", "out": "f32"},
        # Decoding with a larger, uneven batch against a wide weight.
        {"name": "decode_bf16_50x14336x4096", "op": "gemm", "M": 50, "N": 14336, "K": 4096, "dtype": "bf16", "out": "bf16"},
        # Prefill of one prompt: a number of rows that is no multiple of any tile.
        {"name": "prefill_bf16_1000x6144x4096", "op": "gemm", "M": 1000, "N": 6144, "K": 4096, "dtype": "bf16", "out": "bf16"},
        # The benchmark's headline.
        {"name": "gemm_f16_4096", "op": "gemm", "M": 4096, "N": 4096, "K": 4096, "dtype": "f16", "out": "f16"},
        # Its largest fp8 configuration, per-tensor scales folded into alpha.
        {"name": "gemm_fp8_8192", "op": "gemm", "M": 8192, "N": 8192, "K": 8192, "dtype": "fp8", "out": "bf16"},
        # One linear layer of a training step: forward with a bias, the gradient of the input, the gradient of the weight,
        # over a packed batch whose number of tokens is no multiple of any tile.
        {"name": "train_bf16_6000x4096x14336", "op": "train", "T": 6000, "I": 4096, "O": 14336, "dtype": "bf16"},
        # The benchmark's tiled copy: column-major to row-major, 1 GiB each way.
        {"name": "transpose_f32_16384", "op": "transpose", "R": 16384, "C": 16384, "dtype": "f32"},
        # Keys of a batch of sequences brought to the form a product with queries reads: [B,S,H,D] -> [B,H,D,S].
        {"name": "permute_f16_4x2000x32x128", "op": "permute", "kind": "bshd_bhds", "B": 4, "S": 2000, "H": 32, "D": 128, "dtype": "f16"},
        # A master weight written out transposed in the compute type.
        {"name": "cast_f32_bf16_5000x3000", "op": "cast", "kind": "transposed", "R": 5000, "C": 3000, "src": "f32", "dst": "bf16"},
        # What surrounds a layer's product when it is not fused: a bias that repeats over the columns, a ReLU, a residual
        # (axpby!) and a masked overwrite (copyto_if!), on activations with one column per token.
        {"name": "pointwise_bf16_4096x3000", "op": "pointwise", "F": 4096, "T": 3000, "dtype": "bf16"},
    ]


# ---- more cases of the same ranges ---------------------------------------------------------------------------------
def _log(rng, lo, hi, step=1):
    """A whole multiple of `step` in lo..hi, spread over its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    family = rng.choice(["fma", "small", "decode", "decode", "prefill", "prefill", "large", "train", "transpose", "permute",
                         "permute", "cast", "pointwise"])
    if family == "fma":
        # any sizes: the kernels predicate their edges
        return {"op": "fma", "M": _log(rng, 64, 768), "N": _log(rng, 64, 768), "K": _log(rng, 64, 768), "dtype": rng.choice(["f32", "f16"])}
    if family == "small":
        return {"op": "gemm", "M": _log(rng, 96, 1024, 8), "N": _log(rng, 96, 1024, 8), "K": _log(rng, 64, 1024, 8),
                "dtype": rng.choice(["f16", "bf16"]), "out": rng.choice(["f16", "bf16", "f32"])}
    if family == "decode":
        return {"op": "gemm", "M": _log(rng, 1, 64), "N": _log(rng, 1024, 28672, 8), "K": _log(rng, 1024, 16384, rng.choice([16, 64, 128])),
                "dtype": rng.choice(["bf16", "f16", "fp8"]), "out": rng.choice(["bf16", "f32"])}
    if family == "prefill":
        # any number of rows; weights in the usual multiples of 128, now and then only of 8
        step = rng.choice([128, 128, 8])
        return {"op": "gemm", "M": _log(rng, 65, 4096), "N": _log(rng, 1024, 14336, step), "K": _log(rng, 1024, 8192, rng.choice([128, 128, 16])),
                "dtype": rng.choice(["bf16", "f16", "fp8"]), "out": "bf16"}
    if family == "large":
        dtype = rng.choice(["f16", "bf16", "fp8", "f32"])
        hi = 4096 if dtype == "f32" else 8192
        return {"op": "gemm", "M": _log(rng, 2048, hi, 64), "N": _log(rng, 2048, hi, 64), "K": _log(rng, 2048, hi, 64), "dtype": dtype,
                "out": "f32" if dtype == "f32" else rng.choice(["bf16", "f32"])}
    if family == "train":
        return {"op": "train", "T": _log(rng, 256, 6000, 8), "I": _log(rng, 1024, 4096, 64), "O": _log(rng, 1024, 14336, 64),
                "dtype": rng.choice(["bf16", "f16"])}
    if family == "transpose":
        return {"op": "transpose", "R": _log(rng, 256, 16384, rng.choice([1, 8, 64])), "C": _log(rng, 256, 16384, rng.choice([1, 8, 64])),
                "dtype": rng.choice(["f32", "f32", "f16", "fp8"])}
    if family == "permute":
        if rng.random() < 0.5:
            hw = rng.choice([7, 14, 28, 56])
            return {"op": "permute", "kind": rng.choice(["nchw_nhwc", "nhwc_nchw"]), "B": _log(rng, 1, 64), "H": hw, "W": hw,
                    "C": 64 * rng.choice([1, 2, 4, 8]), "dtype": rng.choice(["f16", "f32"])}
        return {"op": "permute", "kind": rng.choice(["bshd_bhds", "bshd_bhsd"]), "B": rng.randint(1, 8), "S": _log(rng, 128, 4096, rng.choice([1, 8])),
                "H": rng.choice([8, 16, 32]), "D": rng.choice([64, 128]), "dtype": rng.choice(["f16", "bf16"])}
    if family == "cast":
        src, dst = rng.choice([("f32", "bf16"), ("f32", "f16"), ("bf16", "f32"), ("f32", "fp8"), ("bf16", "fp8")])
        return {"op": "cast", "kind": rng.choice(["transposed", "dense", "window"]), "R": _log(rng, 256, 12288, rng.choice([1, 8, 128])),
                "C": _log(rng, 256, 12288, rng.choice([1, 8, 128])), "src": src, "dst": dst}
    return {"op": "pointwise", "F": _log(rng, 256, 16384, rng.choice([1, 8, 128])), "T": _log(rng, 64, 8192), "dtype": rng.choice(["bf16", "f16", "f32"])}


# ---- inputs and what a program keeps beside them --------------------------------------------------------------------
def _randn(shape, dtype, g, scale=1.0):
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * scale).to(DT[dtype])


def _col(t, shape):
    """A column-major MoYeArray over t's buffer (the reference's arrays are column-major)."""
    return mh.MoYeArray.from_torch(t, mh.Layout(shape, tuple(math.prod(shape[:i]) for i in range(len(shape)))))


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return {"case": case, **_PREPARE[case["op"]](case, g)}


def _prepare_fma(c, g):
    M, N, K, dt = c["M"], c["N"], c["K"], c["dtype"]
    a, b = _randn(M * K, dt, g), _randn(K * N, dt, g)
    d, acc = torch.empty(M * N, device="cuda", dtype=torch.float32), _randn(M * N, "f32", g)
    # C (M,N) += A (M,K) times a column-major (K,N) matrix, handed over as (N,K)
    return {"mma": mh.make_tiled_mma(mh.MMA_UNIVERSAL_FMA, cta_tile=(32, 32, 8)), "d": d, "A": _col(a, (M, K)),
            "B": mh.MoYeArray.from_torch(b, mh.Layout((N, K), (K, 1))), "C": _col(acc, (M, N)), "D": _col(d, (M, N))}


def _prepare_gemm(c, g):
    M, N, K, dt = c["M"], c["N"], c["K"], c["dtype"]
    alpha = 1.0
    if dt == "fp8":
        a, b = _randn((M, K), "f32", g), _randn((N, K), "f32", g)
        sa, sb = 4.5 / 448, 4.5 / 448  # per-tensor scales as a calibration leaves them: the largest of a normal sample near the top of the range
        a, b = (a / sa).clamp_(-448, 448).to(DT[dt]), (b / sb).clamp_(-448, 448).to(DT[dt])
        alpha = sa * sb / math.sqrt(K)
    else:
        a, b = _randn((M, K), dt, g), _randn((N, K), dt, g, 1.0 / math.sqrt(K))
    d = torch.empty((M, N), device="cuda", dtype=DT[c["out"]])
    # tile, waves and K ranges are left to the library
    return {"mma": mh.tiled_mma_desc(ATOM[dt], split_k=-1), "alpha": alpha, "d": d, "A": mh.MoYeArray.from_torch(a),
            "B": mh.MoYeArray.from_torch(b), "D": mh.MoYeArray.from_torch(d)}


def _prepare_train(c, g):
    T, I, O, dt = c["T"], c["I"], c["O"], c["dtype"]
    x, w = _randn((T, I), dt, g), _randn((O, I), dt, g, 1.0 / math.sqrt(I))
    dy, bias = _randn((T, O), dt, g), _randn((O,), "f32", g)
    y, dx = (torch.empty(s, device="cuda", dtype=DT[dt]) for s in ((T, O), (T, I)))
    dw = torch.empty((O, I), device="cuda", dtype=torch.float32)
    mma = mh.tiled_mma_desc(ATOM[dt])
    tx, tw, tdy = tensor_of(x), tensor_of(w), tensor_of(dy)
    # Y = X W' + bias;  dX = dY W;  dW = dY' X: the second operand is (N,K), so W and X come as transposed views
    calls = [(tensor_of(y), tx, tw, mh.gemm_epilogue(op=_lib.MAP_ADD, operand=tensor_of(bias, (T, O), (0, 1)))),
             (tensor_of(dx), tdy, tensor_of(w, (I, O), (1, I)), mh.gemm_epilogue()),
             (tensor_of(dw), tensor_of(dy, (O, T), (1, O)), tensor_of(x, (I, T), (1, I)), mh.gemm_epilogue())]
    need = max(mh.gemm_workspace_size(mma, D, A, B, ep) for D, A, B, ep in calls)
    ws = torch.empty(max(need, 256), dtype=torch.uint8, device="cuda")
    return {"mma": mma, "calls": calls, "ws": ws, "need": need, "keep": (x, w, dy, bias), "out": (y, dx, dw)}


def _prepare_transpose(c, g):
    R, C, dt = c["R"], c["C"], c["dtype"]
    src = torch.randint(0, 256, (R * C * BYTES[dt],), generator=g, device="cuda", dtype=torch.uint8).view(
        {4: torch.int32, 2: torch.int16, 1: torch.uint8}[BYTES[dt]])
    dst = torch.empty_like(src)
    # (R,C) column-major -> row-major
    return {"dst": dst, "S": _col(src, (R, C)), "T": mh.MoYeArray.from_torch(dst, mh.Layout((R, C), (C, 1)))}


def _prepare_permute(c, g):
    dt, kind = c["dtype"], c["kind"]
    if kind in ("nchw_nhwc", "nhwc_nchw"):
        shape = (c["B"], c["C"], c["H"], c["W"]) if kind == "nchw_nhwc" else (c["B"], c["H"], c["W"], c["C"])
        order = (0, 2, 3, 1) if kind == "nchw_nhwc" else (0, 3, 1, 2)
    else:
        shape = (c["B"], c["S"], c["H"], c["D"])
        order = (0, 2, 3, 1) if kind == "bshd_bhds" else (0, 2, 1, 3)
    src = _randn(shape, dt, g)
    dst = torch.empty([shape[i] for i in order], device="cuda", dtype=DT[dt])
    return {"dst": dst, "S": mh.MoYeArray.from_torch(src.permute(order)), "T": mh.MoYeArray.from_torch(dst)}


def _prepare_cast(c, g):
    R, C, kind = c["R"], c["C"], c["kind"]
    if kind == "window":  # a block of columns of a wider array (one projection of a fused one)
        src = _randn((R, 2 * C), c["src"], g)[:, C:]
    else:
        src = _randn((R, C), c["src"], g)
    dst = torch.empty((C, R) if kind == "transposed" else (R, C), device="cuda", dtype=DT[c["dst"]])
    return {"dst": dst, "keep": src, "S": mh.MoYeArray.from_torch(src.t() if kind == "transposed" else src), "T": mh.MoYeArray.from_torch(dst)}


def _prepare_pointwise(c, g):
    F, T, dt = c["F"], c["T"], c["dtype"]
    x, resid, pad, bias = (_randn(n, dt, g) for n in (F * T, F * T, F * T, F))
    # whole tokens (columns) are masked, as padding is
    mask = (torch.rand((T, 1), generator=g, device="cuda") < 0.25).expand(T, F).contiguous().to(torch.uint8)
    h, y = torch.empty_like(x), torch.empty_like(x)
    return {"X": _col(x, (F, T)), "bias": _col(bias, (F,)), "resid": _col(resid, (F, T)), "pad": _col(pad, (F, T)),
            "mask": _col(mask, (F, T)), "H": _col(h, (F, T)), "Y": _col(y, (F, T)), "out": (h, y)}


_PREPARE = {"fma": _prepare_fma, "gemm": _prepare_gemm, "train": _prepare_train, "transpose": _prepare_transpose,
            "permute": _prepare_permute, "cast": _prepare_cast, "pointwise": _prepare_pointwise}


# ---- one pass -------------------------------------------------------------------------------------------------------
def run(s):
    op, st = s["case"]["op"], current_stream()
    if op == "fma":
        mh.gemm_(s["mma"], s["D"], s["A"], s["B"], s["C"], stream=st)
        return s["d"]
    if op == "gemm":
        mh.gemm_(s["mma"], s["D"], s["A"], s["B"], alpha=s["alpha"], stream=st)
        return s["d"]
    if op == "train":
        for D, A, B, ep in s["calls"]:
            mh.gemm_ex_(s["mma"], D, A, B, None, ep, s["ws"].data_ptr() if s["need"] else None, s["need"], st)
        return s["out"]
    if op in ("transpose", "permute", "cast"):
        mh.copyto_(s["T"], s["S"], stream=st)
        return s["dst"]
    mh.map_("add", s["H"], s["X"], s["bias"], stream=st)
    mh.map_("max", s["H"], s["H"], scalar=0.0, stream=st)
    mh.copyto_(s["Y"], s["resid"], stream=st)
    mh.axpby_(0.5, s["H"], 1.0, s["Y"], stream=st)
    mh.copyto_if_(s["Y"], s["pad"], s["mask"], stream=st)
    return s["out"]


# ---- what a pass cannot do without ----------------------------------------------------------------------------------
def work(c):
    op = c["op"]
    if op in ("fma", "gemm"):
        M, N, K, eb = c["M"], c["N"], c["K"], BYTES[c["dtype"]]
        out = 2 * M * N * 4 if op == "fma" else M * N * BYTES[c["out"]]
        return {"bytes": (M + N) * K * eb + out, "flops": 2 * M * N * K}
    if op == "train":
        T, I, O = c["T"], c["I"], c["O"]
        return {"bytes": 2 * (T * I + O * I + T * O) + 4 * O + 2 * (T * O + T * I) + 4 * O * I, "flops": 6 * T * I * O}
    if op == "transpose":
        return {"bytes": 2 * c["R"] * c["C"] * BYTES[c["dtype"]], "flops": 0}
    if op == "permute":
        n = c["B"] * c["H"] * (c["W"] * c["C"] if "C" in c else c["S"] * c["D"])
        return {"bytes": 2 * n * BYTES[c["dtype"]], "flops": 0}
    if op == "cast":
        return {"bytes": c["R"] * c["C"] * (BYTES[c["src"]] + BYTES[c["dst"]]), "flops": 0}
    F, T, eb = c["F"], c["T"], BYTES[c["dtype"]]
    # read x, bias, residual, pad and mask; write h and y
    return {"bytes": 5 * F * T * eb + F * T + F * eb, "flops": 4 * F * T}


def tolerance(c):
    """Copies, conversions, element-wise operations and UniversalFMA have one right answer.  A matrix-core product sums in an
    order of its own and rounds once: against the product in 64 bits 1.66e-3 with bf16 results and 2.08e-4 with f16 ones
    whatever the sizes (the rounding itself), and with f32 results 1.1e-7 to 4.9e-7 from narrower operands (K up to 12000),
    up to 1.1e-6 from f32 operands.  Four times that."""
    if c["op"] == "train":
        return {"rel": 7e-3 if c["dtype"] == "bf16" else 8.5e-4}
    if c["op"] != "gemm":
        return "exact"
    return {"rel": {"bf16": 7e-3, "f16": 8.5e-4, "f32": 4e-6 if c["dtype"] == "f32" else 2e-6}[c["out"]]}
