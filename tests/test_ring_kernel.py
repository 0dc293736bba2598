"""The ring kernel (csrc/gemm_ring.h) at the stage counts where its loops change hands: fewer stages than slots, as many, one to three more, odd and
even, a partial stage behind each.  int8, so that every sum is exact and a stage read too early or twice shows."""
import pytest
import torch

from helpers import gen
from tilelang_ascend_amd import _abi

SLOTS = {2: 5, 3: 6, 4: 6, 5: 10}  # 160 KB / one stage of both operand tiles


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [2, 3, 4, 5])
@pytest.mark.parametrize("more", [-1, 0, 1, 2, 3, 17, 18])
@pytest.mark.parametrize("tail", [0, 80])
def test_stage_counts(variant, more, tail):
    lib, P, st = _abi.load(), _abi.ptr, torch.cuda.current_stream().cuda_stream
    M, N, K = 130, 208, (SLOTS[variant] + more) * 128 + tail
    print(f"ring variant={variant} stages={SLOTS[variant] + more} tail={tail}", flush=True)
    A = torch.randint(-127, 128, (M, K), dtype=torch.int8, generator=gen(K))
    W = torch.randint(-127, 128, (K, N), dtype=torch.int8, generator=gen(K + 1))
    want = (A.double() @ W.double()).to(torch.int32)
    dA = A.cuda()
    lib.tlq_tune_gemm_groups(variant), lib.tlq_tune_i8_tile(128)
    try:
        for layout, dW in ((_abi.B_KN, W.cuda()), (_abi.B_NK, W.t().contiguous().cuda())):
            for _ in range(3):
                C = torch.full((M, N), -1, dtype=torch.int32, device="cuda")
                lib.tlq_debug_launch_log(1)
                rc = lib.tlq_gemm_i8(P(dA), P(dW), P(C), 1, M, N, K, layout, st)
                log = lib.tlq_debug_launch_log_text().decode()
                lib.tlq_debug_launch_log(0)
                _abi.check(rc)
                assert "ring_gemm_mfma_kernel" in log and torch.equal(C.cpu(), want)
    finally:
        lib.tlq_tune_gemm_groups(0), lib.tlq_tune_i8_tile(0)
