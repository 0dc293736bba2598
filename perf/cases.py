"""The work that users of this package give it, as cases that can be timed and compared.

A case is a dict with an ``op`` (which operator, through its public Python entry point) and its sizes and options:

``w4a16``    dequant_gemm_fp16_wrapper: activations x packed int4 weights with per-group scales and zero points.  One row is
             the decode step of one sequence, up to some tens a decode batch, hundreds a chunk of a prompt, thousands prefill.
``w8a8``     the quantised (batch) matmuls: int8 weights [K, N] as the reference lays them out, one scale per channel, or per
             token and per channel; one to eight matrices in a call.
``linear8``  an int8 linear layer as an inference program runs it: quantise the activations per token, then the GEMM with
             weights [N, K] and the two-scale epilogue.
``w4a8``     w4a8_gemm_cv: int8 activations x packed int4 weights with the caller's workspace, exact int32 results.
``plain``    the 16-bit GEMM (one matrix: fp16_gemm; more: batch_matmul) that the quantised operators stand beside.
``weights``  a weight matrix on its way into the package and out again: quantised to int4 with scales, packed, dequantised.
"""
import torch

from tilelang_ascend_amd import ops
from tilelang_ascend_amd.quantize import gpu as quantize_gpu

_T = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}
_BYTES = {"float16": 2, "bfloat16": 2, "float32": 4}
# the most that one case may cost: the largest listed one (8192 rows on a 14336 x 4096 matrix)
_MOST = 8192 * 14336 * 4096


def listed():
    return [
        # the smallest call there is a use for: a 256 x 256 x 256 problem, one scalar zero point
        {"name": "w4a16 small", "op": "w4a16", "M": 256, "N": 256, "K": 256, "group": 128, "dtype": "float16", "zeros": "scalar"},
        # one sequence being decoded: one row against an up projection
        {"name": "w4a16 decode", "op": "w4a16", "M": 1, "N": 11008, "K": 4096, "group": 128, "dtype": "float16", "zeros": "tensor"},
        # sixteen sequences being decoded together
        {"name": "w4a16 decode batch", "op": "w4a16", "M": 16, "N": 14336, "K": 4096, "group": 128, "dtype": "bfloat16", "zeros": "tensor"},
        # a short prompt, of a length that is no multiple of anything, against a down projection with 86 groups in a row
        {"name": "w4a16 short prompt", "op": "w4a16", "M": 211, "N": 4096, "K": 11008, "group": 128, "dtype": "float16", "zeros": "tensor"},
        # prefill of 4096 tokens
        {"name": "w4a16 prefill", "op": "w4a16", "M": 4096, "N": 4096, "K": 4096, "group": 128, "dtype": "bfloat16", "zeros": "scalar"},
        # prefill of several prompts at once against an up projection: the largest
        {"name": "w4a16 long prefill", "op": "w4a16", "M": 8192, "N": 14336, "K": 4096, "group": 64, "dtype": "float16", "zeros": "tensor"},
        # eight matrices of int8 products with per-token and per-channel scales
        {"name": "w8a8 batch", "op": "w8a8", "B": 8, "M": 2048, "N": 4096, "K": 4096, "scale": "token", "dtype": "float16"},
        # an int8 down projection in a decode batch
        {"name": "linear8 decode", "op": "linear8", "M": 32, "N": 4096, "K": 14336, "dtype": "bfloat16"},
        # the same kind of layer over a prompt of an odd length
        {"name": "linear8 prefill", "op": "linear8", "M": 4099, "N": 4096, "K": 4096, "dtype": "bfloat16"},
        # int8 activations on int4 weights, a batch of requests
        {"name": "w4a8", "op": "w4a8", "M": 128, "N": 4096, "K": 11008},
        # the 16-bit GEMM on weights that were not quantised
        {"name": "plain", "op": "plain", "B": 1, "M": 1000, "N": 4096, "K": 4096, "dtype": "float16"},
        # one matrix of a checkpoint quantised, packed and dequantised
        {"name": "weights", "op": "weights", "N": 14336, "K": 4096, "group": 128, "dtype": "float16"},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    op = rng.choice(["w4a16"] * 5 + ["w8a8", "linear8", "linear8", "w4a8", "plain", "weights"])
    while True:
        N = 16 * _log(rng, 16, 14336 // 16)
        if rng.random() < 0.6:
            N = max(256, N // 128 * 128)
        K = 128 * _log(rng, 2, 14336 // 128)
        M = _log(rng, 1, 8192)
        dtype = rng.choice(["float16", "bfloat16"])
        B = 1
        if op == "w4a16":
            c = {"M": M, "N": N, "K": K, "group": rng.choice([64, 128, 128]), "dtype": dtype, "zeros": rng.choice(["tensor", "scalar"])}
        elif op == "w8a8":
            B = rng.choice([1, 1, 2, 4, 8])
            c = {"B": B, "M": M, "N": N, "K": K, "scale": rng.choice(["token", "channel"]), "dtype": dtype}
        elif op == "linear8":
            c = {"M": M, "N": N, "K": K, "dtype": rng.choice(["bfloat16", "float32"])}
        elif op == "w4a8":
            c = {"M": M, "N": N, "K": K}
        elif op == "plain":
            B = rng.choice([1, 1, 2, 4, 8])
            c = {"B": B, "M": M, "N": N, "K": K, "dtype": "float16" if B == 1 else dtype}
        else:
            c = {"N": N, "K": K, "group": rng.choice([64, 128, 128]), "dtype": dtype}
        if op == "weights" or 2 * B * M * N * K <= _MOST:
            return {"op": op, **c}


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    op, N, K = case["op"], case["N"], case["K"]

    def normal(*shape, dtype):
        return torch.randn(*shape, generator=g, device="cuda", dtype=_T[dtype])

    def uniform(lo, hi, *shape, dtype="float32"):
        return (torch.rand(*shape, generator=g, device="cuda") * (hi - lo) + lo).to(_T[dtype])

    def whole(lo, hi, *shape, dtype):  # lo .. hi - 1
        return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=dtype)

    s = {"op": op, "case": case}
    if op == "w4a16":
        group, dtype, M = case["group"], case["dtype"], case["M"]
        s["gemm"] = ops.dequant_gemm_fp16_wrapper(M, N, K, 128, 256, 64, dtype, dtype, group)
        s["args"] = [normal(M, K, dtype=dtype), whole(0, 256, N, K // 2, dtype=torch.uint8),
                     uniform(0.005, 0.02, N, K // group, dtype=dtype),
                     whole(6, 10, N, K // group, dtype=torch.int32).to(_T[dtype]) if case["zeros"] == "tensor" else 8]
    elif op == "w8a8":
        B, M, dtype = case["B"], case["M"], case["dtype"]
        lead = (B,)
        if case["scale"] == "token":
            s["gemm"] = ops.quant_batch_matmul_per_token(B, M, N, K, out_dtype=dtype)
        elif B > 1:
            s["gemm"] = ops.simple_quant_batch_matmul(B, M, N, K, "N", 128, 256, 64, out_dtype=dtype)
        else:
            s["gemm"] = ops.simple_quant_matmul(M, N, K, "N", 128, 256, 64, out_dtype=dtype)
            lead = ()
        s["args"] = [whole(-127, 128, *lead, M, K, dtype=torch.int8), whole(-127, 128, *lead, K, N, dtype=torch.int8)]
        if case["scale"] == "token":
            s["args"].append(uniform(0.01, 0.05, B, M))
        s["args"].append(uniform(0.001, 0.01, N))
    elif op == "linear8":
        s["quantise"] = ops.act_quant_kernel_int8_optimized(K)
        s["gemm"] = ops.int8_gemm_kernel_corrected(N, K, out_dtype=case["dtype"])
        s["args"] = [normal(case["M"], K, dtype="bfloat16"), whole(-127, 128, N, K, dtype=torch.int8), uniform(0.001, 0.01, N)]
    elif op == "w4a8":
        s["gemm"] = ops.w4a8_gemm_cv(case["M"], N, K)
        s["args"] = [whole(-127, 128, case["M"], K, dtype=torch.int8), whole(0, 256, N, K // 2, dtype=torch.uint8),
                     torch.empty(N, K, dtype=torch.int8, device="cuda")]
    elif op == "plain":
        B, M, dtype = case["B"], case["M"], case["dtype"]
        lead = (B,) if B > 1 else ()
        s["gemm"] = ops.batch_matmul(B, M, N, K, 128, 256, 64, dtype) if B > 1 else ops.fp16_gemm(M, N, K, 128, 256, 64)
        s["args"] = [normal(*lead, M, K, dtype=dtype), normal(*lead, K, N, dtype=dtype)]
    else:
        s["args"] = [normal(N, K, dtype=case["dtype"]) * 0.02]
    return s


def run(state):
    args = state["args"]
    if state["op"] == "linear8":
        x, weight, scale = args
        q, scale_x = state["quantise"](x)
        return q, scale_x, state["gemm"](q, weight, scale_x, scale)
    if state["op"] == "weights":
        case = state["case"]
        q, scales = quantize_gpu.quantize_sym4(args[0], case["group"])
        # the positive maximum of a group becomes q = 16, which four bits do not hold: stored as 15
        packed = quantize_gpu.pack_int4((q + 8).clamp_(max=15), None, torch.uint8)
        return packed, scales, ops.dequantize_w4(packed, scales, 8, case["group"], _T[case["dtype"]])
    return state["gemm"](*args)


def work(case):
    op, N, K, M, B = case["op"], case["N"], case["K"], case.get("M", 0), case.get("B", 1)
    flops = 2 * B * M * N * K
    if op == "w4a16":
        values = N * (K // case["group"]) * 2
        moved = N * K // 2 + values * (2 if case["zeros"] == "tensor" else 1) + 2 * M * K + 2 * M * N
    elif op == "w8a8":
        moved = B * (M * K + N * K + 2 * M * N) + 4 * N + (4 * B * M if case["scale"] == "token" else 0)
    elif op == "linear8":
        # the quantised activations and their scales are outputs too
        moved = 2 * M * K + M * K + 4 * M + N * K + 4 * N + M * N * _BYTES[case["dtype"]]
    elif op == "w4a8":
        moved = M * K + N * K // 2 + 4 * M * N
    elif op == "plain":
        moved = 2 * B * (M * K + N * K + M * N)
    else:
        moved = 2 * N * K + N * K // 2 + 2 * N * (K // case["group"]) + 2 * N * K
        flops = 4 * N * K
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    if case["op"] in ("w4a16", "plain"):
        # sums of exactly rounded products in 32 bits, in any order: what is left is the rounding of the result to its type,
        # where two orders of summation may fall on neighbouring values (2^-10 and 2^-7 of a value apart)
        return {"rel": 1e-3, "max": 4e-3} if case["dtype"] == "float16" else {"rel": 4e-3, "max": 2e-2}
    # integer sums are exact, and the rescaling of each value and the quantisers are functions of single values
    return "exact"
