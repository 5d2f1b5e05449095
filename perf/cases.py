"""The work that users of this framework have it do, as cases that can be timed.

Every case goes through the public entry points (`computelibrary_amd.capi`, the binding of include/mi355_gemmlowp.h)
with device-resident tensors. Handles are created and static weights prepared in `prepare`, as a program does once;
`run` is what the program does for every new input.

A GEMM case has M, N, K, batch, the operand types (`a`, `b`: u8 = QASYMM8, s8 = QASYMM8_SIGNED / QSYMM8), the destination
type (`out`) and `per_channel` requantisation; a decode case the rows M and the two sizes of a transformer's block; a
convolution case its geometry, types and layout. u8 operands have zero points near the middle of their range that are
not exactly 128, as calibrated tensors have, so both offset terms count.
"""
import math

import numpy as np
import torch

from computelibrary_amd import capi

_TORCH = {"u8": torch.uint8, "s8": torch.int8, "s32": torch.int32, "f32": torch.float32, "f16": torch.float16}
_CODE = {"u8": capi.U8, "s8": capi.S8, "s32": capi.S32, "f32": capi.F32, "f16": capi.F16}
_BYTES = {"u8": 1, "s8": 1, "s32": 4, "f32": 4, "f16": 2}

# the most that a drawn case may cost: below the largest listed case (prefill_long)
_MOST_OPS = 6.0e11
_MOST_BYTES = 4.0e8


def _gemm(kind, M, N, K, a, b, out, per_channel, batch=1):
    return {"kind": kind, "M": M, "N": N, "K": K, "batch": batch, "a": a, "b": b, "out": out, "per_channel": per_channel}


def _conv(batch, H, W, C, OFM, k, stride, src, weights, per_channel, layout):
    return {"kind": "conv", "batch": batch, "H": H, "W": W, "C": C, "OFM": OFM, "k": k, "stride": stride, "src": src,
            "weights": weights, "per_channel": per_channel, "layout": layout}


def listed():
    return [
        # the smallest call: one QASYMM8 product of the size of the reference's example program. Latency is what counts.
        dict(_gemm("gemm", 256, 256, 256, "u8", "u8", "u8", False), name="gemm_u8_256"),
        # one projection of a prompt of 2048 tokens: the headline workload
        dict(_gemm("gemm", 2048, 4096, 4096, "s8", "s8", "s8", True), name="prefill_projection"),
        # the widest projection of a feed-forward block for a batch of prompts: the largest call
        dict(_gemm("gemm", 8192, 11008, 4096, "s8", "s8", "s8", True), name="prefill_long"),
        # one decode step of a batch of 8: the four projections of a transformer block, each with its own weights
        # (157 MB of them, so a step over several blocks reads them from HBM)
        {"kind": "decode", "M": 8, "hidden": 4096, "ffn": 11008, "name": "decode_block_m8"},
        # the two-function form with a shape in which nothing is aligned (K odd: rows of A start on any byte): an S32 GEMM
        # followed by the stand-alone output stage
        dict(_gemm("two_step", 973, 783, 1021, "u8", "u8", "u8", False), name="two_step_u8_ragged"),
        # batched products dequantised to float, K not a multiple of a matrix-core step
        dict(_gemm("gemm", 1024, 1024, 1000, "s8", "s8", "f32", False, 16), name="batched_f32_k1000"),
        # a product of two activations (attention scores of 32 heads): B is not constant, so it is packed before every run
        dict(_gemm("dynamic", 512, 512, 128, "s8", "s8", "f32", False, 32), name="dynamic_b_heads"),
        # a projection whose result goes on in half precision
        dict(_gemm("gemm", 512, 4096, 4096, "s8", "s8", "f16", False), name="projection_f16"),
        # 3x3 layer of an early stage, symmetric per-channel weights
        dict(_conv(32, 56, 56, 64, 64, 3, 1, "s8", "s8", True, "nhwc"), name="conv_56_s8_per_channel"),
        # 3x3 layer of a late stage in the fully asymmetric scheme: QASYMM8 weights with a zero point
        dict(_conv(32, 14, 14, 256, 256, 3, 1, "u8", "u8", False, "nhwc"), name="conv_14_u8_asymmetric"),
        # first layer on RGB images
        dict(_conv(32, 224, 224, 3, 64, 7, 2, "u8", "s8", True, "nhwc"), name="conv_rgb_7x7_s2"),
        # 3x3 layer of a middle stage in the other data layout
        dict(_conv(32, 28, 28, 128, 128, 3, 1, "s8", "s8", True, "nchw"), name="conv_28_nchw"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size over the logarithm of its range: two in five whole multiples of 64 (or 16), the others whatever comes."""
    v = _log(rng, lo, hi)
    how = rng.random()
    step = 64 if how < 0.25 else 16 if how < 0.4 else 1
    return max(lo, v // step * step) if v >= step else v


def draw(rng):
    while True:
        which = rng.choice(["gemm", "gemm", "gemm", "decode", "two_step", "batched", "dynamic", "f16", "conv", "conv", "rgb", "nchw"])
        if which == "gemm":
            a, b, out, pc = rng.choice([("u8", "u8", "u8", False), ("s8", "s8", "s8", True), ("s8", "s8", "s8", False), ("u8", "s8", "u8", True)])
            case = _gemm("gemm", _size(rng, 1, 8192), _size(rng, 16, 11008), _size(rng, 16, 11008), a, b, out, pc)
        elif which == "decode":
            hidden = 64 * _log(rng, 12, 96)
            case = {"kind": "decode", "M": _log(rng, 1, 64), "hidden": hidden, "ffn": 16 * int(round(hidden * rng.uniform(2.5, 4.0) / 16))}
        elif which == "two_step":
            a, b, out = rng.choice([("u8", "u8", "u8"), ("s8", "s8", "s8")])
            case = _gemm("two_step", _size(rng, 16, 2048), _size(rng, 16, 2048), _size(rng, 16, 4096), a, b, out, False)
        elif which == "batched":
            case = _gemm("gemm", _size(rng, 16, 1024), _size(rng, 16, 1024), _size(rng, 16, 2048), "s8", "s8", rng.choice(["f32", "f32", "s32"]), False,
                         rng.randint(2, 32))
        elif which == "dynamic":
            case = _gemm("dynamic", _size(rng, 16, 1024), _size(rng, 16, 1024), _size(rng, 16, 512), "s8", "s8", rng.choice(["f32", "s32"]), False,
                         _log(rng, 1, 64))
        elif which == "f16":
            case = _gemm("gemm", _size(rng, 1, 2048), _size(rng, 64, 8192), _size(rng, 64, 8192), "s8", "s8", "f16", False)
        elif which == "rgb":
            k = rng.choice([3, 5, 7])
            hw = rng.randint(64, 224)
            case = _conv(_log(rng, 1, 32), hw, hw, rng.choice([1, 3, 3, 3, 4]), rng.choice([16, 24, 32, 64, 96]), k, rng.choice([1, 2, 2]),
                         rng.choice(["u8", "s8"]), "s8", True, "nhwc")
        else:
            hw = _log(rng, 7, 112)
            src, weights, pc = rng.choice([("s8", "s8", True), ("u8", "u8", False), ("u8", "s8", True)])
            case = _conv(_log(rng, 1, 32), hw, hw + rng.choice([0, 0, 1, 3]), 8 * _log(rng, 2, 64), 8 * _log(rng, 2, 64), rng.choice([1, 3, 3, 5]),
                         rng.choice([1, 1, 1, 2]), src, weights, pc, "nchw" if which == "nchw" else "nhwc")
        w = work(case)
        if w["flops"] <= (_MOST_OPS if case["kind"] == "gemm" else _MOST_OPS / 6) and w["bytes"] <= _MOST_BYTES:
            return case


def _decode_shapes(case):
    h, f = case["hidden"], case["ffn"]
    return [(3 * h, h), (h, h), (f, h), (h, f)]  # (N, K): queries, keys and values; attention output; up; down


def _out_hw(case):
    pad = case["k"] // 2
    return tuple((case[d] + 2 * pad - case["k"]) // case["stride"] + 1 for d in ("H", "W"))


def work(case):
    if case["kind"] == "decode":
        M = case["M"]
        return {"bytes": sum(N * K + M * K + M * N + 12 * N for N, K in _decode_shapes(case)),
                "flops": sum(2 * M * N * K for N, K in _decode_shapes(case))}
    if case["kind"] == "conv":
        OH, OW = _out_hw(case)
        K = case["k"] * case["k"] * case["C"]
        return {"bytes": case["batch"] * (case["H"] * case["W"] * case["C"] + OH * OW * case["OFM"]) + case["OFM"] * (K + 12),
                "flops": 2 * case["batch"] * OH * OW * case["OFM"] * K}
    M, N, K, batch = case["M"], case["N"], case["K"], case["batch"]
    # (two functions: the S32 matrix between them is an output of the first and an input of the second)
    out = M * N * (4 + 4 + 1 if case["kind"] == "two_step" else _BYTES[case["out"]])
    return {"bytes": batch * (M * K + K * N + out) + 12 * N, "flops": 2 * batch * M * N * K}


def tolerance(case):
    # Integers and bytes are exact. The float of a dequantised product is an exact integer times one float, rounded: against
    # the same in 64 bits it is off by 2.5e-8 (2-norm) at depths of 128, 1000 and 4096, at most 6e-8 of a value. Half
    # precision rounds that once more: 2.1e-4, at most 4.9e-4.
    out = case.get("out")
    if out == "f32":
        return {"rel": 1e-7, "max": 2.4e-7}
    if out == "f16":
        return {"rel": 8e-4, "max": 2e-3}
    return "exact"


def _multipliers(scales):
    """(multiplier, shift) of real = multiplier * 2^-31 * 2^-shift, multiplier in [2^30, 2^31), as int32 tensors"""
    q, e = np.frexp(np.asarray(scales, dtype=np.float64))
    m = np.floor(q * float(1 << 31) + 0.5).astype(np.int64)
    e, m = np.where(m == 1 << 31, e + 1, e), np.where(m == 1 << 31, m // 2, m)
    return m.astype(np.int32), (-e).astype(np.int32)


class _Inputs:
    """What a calibrated quantised network holds, made on the GPU from the seed alone"""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.rng = np.random.default_rng(seed)

    def normal(self, shape, std):
        return torch.randn(shape, device="cuda", generator=self.gen).mul_(std).round_()

    def activations(self, shape, dtype):
        """The whole 8-bit range, as calibration leaves it: uniform, which is also the headline workload's distribution"""
        lo, hi = (0, 256) if dtype == "u8" else (-128, 128)
        return torch.randint(lo, hi, shape, device="cuda", generator=self.gen, dtype=_TORCH[dtype])

    def weights(self, shape, dtype, zero_point=0):
        x = self.normal(shape, 32.0)
        return (x.add_(zero_point).clamp_(0, 255) if dtype == "u8" else x.clamp_(-127, 127)).to(_TORCH[dtype])

    def zero_point(self, dtype):
        return int(self.rng.integers(110, 146)) if dtype == "u8" else int(self.rng.integers(-10, 11))

    def requant(self, K, N, out, per_channel):
        """(descriptor, multipliers, shifts, bias) that spread the results of a K-deep product over the output's range"""
        base = 40.0 / (math.sqrt(K) * 74.0 * 32.0)
        scales = base * self.rng.uniform(0.5, 2.0, size=N if per_channel else 1)
        m, s = _multipliers(scales)
        lo, hi = (0, 255) if out == "u8" else (-128, 127)
        offset = self.zero_point(out)
        rq = capi.requant(0 if per_channel else m[0], 0 if per_channel else s[0], offset, lo, hi, per_channel)
        bias = self.normal((N,), 20.0 / base / 40.0).to(torch.int32)
        if not per_channel:
            return rq, None, None, bias
        return rq, torch.from_numpy(m).cuda(), torch.from_numpy(s).cuda(), bias


def _prepare_gemm(case, x, stream, M, N, K):
    """One static-weights product: (handle, A, D)"""
    batch, a, b, out = case.get("batch", 1), case.get("a", "s8"), case.get("b", "s8"), case.get("out", "s8")
    # (the offsets that go into the library are negated zero points; symmetric weights and both operands of a dequantised
    # product have none)
    dequantised = out in ("f32", "f16")
    a_zp = 0 if dequantised else x.zero_point(a)
    b_zp = x.zero_point(b) if b == "u8" else 0
    A = x.activations((batch, M, K), a)
    B = x.weights((batch, K, N), b, b_zp)
    D = torch.empty((batch, M, N), dtype=_TORCH[out], device="cuda")
    if out in ("u8", "s8"):
        rq, mult, shift, bias = x.requant(K, N, out, case.get("per_channel", True))
        g = capi.Gemm(M, N, K, _CODE[a], _CODE[b], _CODE[out], capi.EPI_FIXEDPOINT, -a_zp, -b_zp, rq, batch=batch, b_batched=batch > 1)
        g.prepare(B, bias, mult, shift, stream)
    else:
        epi = capi.EPI_S32 if out == "s32" else capi.EPI_F32
        g = capi.Gemm(M, N, K, _CODE[a], _CODE[b], _CODE[out], epi, -a_zp, -b_zp, scale=0.02 * 0.005, batch=batch, b_batched=batch > 1)
        g.prepare(B, stream=stream)
    return g, A, D


def prepare(case, seed):
    x = _Inputs(seed)
    stream = torch.cuda.current_stream().cuda_stream
    state = {"kind": case["kind"], "stream": stream}
    if case["kind"] == "decode":
        state["calls"] = [_prepare_gemm(case, x, stream, case["M"], N, K) for N, K in _decode_shapes(case)]
        return state
    if case["kind"] == "conv":
        return _prepare_conv(case, x, state)
    M, N, K, batch = case["M"], case["N"], case["K"], case["batch"]
    if case["kind"] == "gemm":
        state["calls"] = [_prepare_gemm(case, x, stream, M, N, K)]
    elif case["kind"] == "two_step":
        g, A, acc = _prepare_gemm(dict(case, out="s32"), x, stream, M, N, K)
        rq, _, _, bias = x.requant(K, N, case["out"], False)
        state.update(gemm=g, A=A, acc=acc, rq=rq, bias=bias, D=torch.empty((M, N), dtype=_TORCH[case["out"]], device="cuda"))
    else:  # dynamic: both operands are new in every pass
        epi = capi.EPI_S32 if case["out"] == "s32" else capi.EPI_F32
        state.update(gemm=capi.Gemm(M, N, K, _CODE[case["a"]], _CODE[case["b"]], _CODE[case["out"]], epi, scale=0.02 * 0.02, batch=batch,
                                    b_batched=batch > 1),
                     A=x.activations((batch, M, K), case["a"]), B=x.activations((batch, K, N), case["b"]),
                     D=torch.empty((batch, M, N), dtype=_TORCH[case["out"]], device="cuda"))
    return state


def _prepare_conv(case, x, state):
    n, H, W, C, OFM, k, src, weights = (case[f] for f in ("batch", "H", "W", "C", "OFM", "k", "src", "weights"))
    OH, OW = _out_hw(case)
    nchw = case["layout"] == "nchw"
    src_zp, w_zp = x.zero_point(src), x.zero_point(weights) if weights == "u8" else 0
    rq, mult, shift, bias = x.requant(k * k * C, OFM, src, case["per_channel"])
    p = k // 2
    desc = capi.conv_desc(n, H, W, C, OFM, k, k, (case["stride"],) * 2, (p, p, p, p), (1, 1), _CODE[src], _CODE[weights], _CODE[src], -src_zp, -w_zp,
                          src_zp, rq, layout=capi.NCHW if nchw else capi.NHWC)
    w = x.weights((OFM, C, k, k) if nchw else (OFM, k, k, C), weights, w_zp)
    conv = capi.Conv(desc)
    conv.prepare(w, bias, mult, shift, state["stream"])
    state.update(conv=conv, src=x.activations((n, C, H, W) if nchw else (n, H, W, C), src),
                 D=torch.empty((n, OFM, OH, OW) if nchw else (n, OH, OW, OFM), dtype=_TORCH[src], device="cuda"))
    return state


def run(state):
    kind, stream = state["kind"], state["stream"]
    if kind == "conv":
        state["conv"].run(state["src"], state["D"], stream)
        return state["D"]
    if kind == "two_step":
        state["gemm"].run(state["A"], state["acc"], None, stream)
        capi.output_stage(state["acc"][0], state["bias"], state["D"], state["rq"], stream)
        return {"acc": state["acc"], "out": state["D"]}
    if kind == "dynamic":
        state["gemm"].prepare(state["B"], stream=stream)
        state["gemm"].run(state["A"], state["D"], None, stream)
        return state["D"]
    for g, A, D in state["calls"]:
        g.run(A, D, None, stream)
    return [D for _, _, D in state["calls"]]
