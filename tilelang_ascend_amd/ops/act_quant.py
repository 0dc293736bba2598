"""Per-token int8 activation quantiser.

Surface of examples/deepseek_v4/act_quant.py: ``act_quant_kernel_int8_optimized(N, block_M=32,
block_N=32, round_scale=False)`` (:25-92) -> ``kernel(X bfloat16 [M, N]) -> [Y int8 [M, N],
S float32 [M]]`` with ``out_idx=[-2, -1]`` and a symbolic M (:37).

    amax = max(max_n |X[m, n]|, 1e-4)
    S[m] = amax / 127                 (round_scale: 2 ** ceil(log2(amax / 127)), :95-109)
    Y    = int8( rint( clamp(X / S[m], -127, 127) ) )

The arithmetic is that of the reference's golden ``act_quant_torch`` (:112-142): the 1e-4 floor
keeps an all-zero row finite, and the scale always covers the whole row (the reference kernel
only does so when block_N == N, which is how its own test calls it, :171-172).  The block sizes
are accepted for compatibility and do not change the result.  ``in_dtype`` widens the input
type beyond the reference's bfloat16.
"""
from __future__ import annotations

from typing import Literal

from ..jit import ABI_DTYPE, TORCH_DTYPES, KernelSpec, NativeCall, Param, PassConfigKey, jit

_PASS_CONFIGS = {
    PassConfigKey.TL_ASCEND_AUTO_SYNC: True,
    PassConfigKey.TIR_MERGE_STATIC_SMEM: True,
    PassConfigKey.TL_ASCEND_MEMORY_PLANNING: True,
}


@jit(out_idx=[-2, -1], pass_configs=_PASS_CONFIGS)
def act_quant_kernel_int8_optimized(N: int, block_M: int = 32, block_N: int = 32, round_scale: bool = False,
                                    in_dtype: Literal["bfloat16", "float16", "float32"] = "bfloat16"):
    if N <= 0:
        raise ValueError("N must be positive")
    tin = ABI_DTYPE[TORCH_DTYPES[in_dtype]]
    return KernelSpec("act_quant_kernel_int8_optimized",
                      [Param("X", ("M", N), in_dtype), Param("Y", ("M", N), "int8"), Param("S", ("M",), "float32")],
                      NativeCall("act_quant", (N, tin, bool(round_scale))), {"block": (block_M, block_N), "round_scale": bool(round_scale)})
