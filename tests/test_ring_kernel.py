"""The ring kernel (csrc/gemm_ring.h) at the stage counts where its loops change hands: the fewest, one to four more, around the bound of its loads' lead, odd and
even, a partial stage behind each.  int8, so that every sum is exact and a stage read too early or twice shows."""
import pytest
import torch

from helpers import gen
from tilelang_ascend_amd import _abi

STAGES = [4, 5, 6, 7, 8, 15, 16, 17, 18, 19, 20, 33]  # loads three stages ahead up to 16, four beyond; every way through the last ones


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [2, 3, 4, 5])
@pytest.mark.parametrize("stages", STAGES)
@pytest.mark.parametrize("tail", [0, 80])
def test_stage_counts(variant, stages, tail):
    lib, P, st = _abi.load(), _abi.ptr, torch.cuda.current_stream().cuda_stream
    M, N, K = 130, 208, stages * 128 + tail
    print(f"ring variant={variant} stages={stages} tail={tail}", flush=True)
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


def test_schedule():
    """Walked on the host: every stage is waited for and published by a barrier before it is read, nothing is overwritten that someone may still read, and
    no more than four stages are asked for ahead of the first product, whatever LDS would hold; one load more left in flight and the walk fails."""
    lib = _abi.load()
    for stages in [*range(1, 41), 224]:
        for loads in (2, 3, 4):
            assert lib.tlq_debug_check_ring_schedule(stages, loads, 0) == 0, _abi.last_error()
            assert lib.tlq_debug_check_ring_schedule(stages, loads, 1) != 0
            assert "before its loads were waited for" in _abi.last_error()
