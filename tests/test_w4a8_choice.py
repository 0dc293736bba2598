"""W4A8 with two's complement weights: where the choice between the small-tile kernel and what would run in its place was wrong while both
ways of multiplying four bits shared an estimate, and on either side of the row count up to which the workspace is scratch."""
import ctypes

import pytest
import torch

from helpers import assert_bit_equal, gen
from tilelang_ascend_amd import _abi


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [_abi.S4_TWOS, _abi.S4_OFFSET8, _abi.U4])
@pytest.mark.parametrize("M,N,K", [(1, 6336, 11520), (25, 4432, 10112), (49, 2304, 12160), (64, 1040, 384), (65, 1040, 384), (186, 1408, 7168), (256, 1040, 128)])
def test_exact(mode, M, N, K):
    g = gen(M + N)
    A = torch.randint(-128, 128, (M, K), dtype=torch.int8, generator=g)
    Wp = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, generator=g)
    u = torch.stack([Wp & 15, Wp >> 4], dim=-1).reshape(N, K).to(torch.float32)
    W = u if mode == _abi.U4 else u - 8 if mode == _abi.S4_OFFSET8 else torch.where(u >= 8, u - 16, u)
    Ad, Wd = A.cuda(), Wp.cuda()
    want = (Ad.double() @ W.double().cuda().T.contiguous()).to(torch.int32).cpu()  # (sums below 2^53: exact)
    lib, st = _abi.load(), torch.cuda.current_stream().cuda_stream
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    C, ws = torch.full((M, N), 7, dtype=torch.int32, device="cuda"), torch.empty(N, K, dtype=torch.int8, device="cuda")
    lib.tlq_debug_launch_log(1)
    rc = lib.tlq_gemm_w4a8_ws(P(Ad), P(Wd), P(ws), ws.numel(), P(C), M, N, K, mode, st)
    log = lib.tlq_debug_launch_log_text().decode()
    lib.tlq_debug_launch_log(0)
    _abi.check(rc)
    assert mode == _abi.U4 or "gemm_small_kernel" in log or lib.tlq_device_cu_count() != 256, log
    assert_bit_equal(C.cpu(), want, f"W4A8 mode {mode} {M}x{N}x{K}")
