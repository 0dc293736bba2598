"""129 .. 512 rows on large matrices: the panel kernels take row counts that are no multiple of four in the automatic choice, and the streaming kernel runs where its
estimate is ahead of theirs."""
import pytest
import torch

from helpers import check_float_output, gen, make_w4
from oracle import ref


# (M, N, K, group, kernel): the last of one, two, three rows of a block of four, with K slices and without; a streaming plan in the place of either panel kernel
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,group,kernel", [(495, 24320, 384, 128, "panel256"), (421, 30336, 768, 32, "panel256"), (426, 28032, 384, 64, "panel256"),
                                                (445, 9088, 9984, 64, "panel256"), (488, 4240, 10240, 128, "stream"), (308, 14720, 4096, 128, "stream")])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("zeros", ["int", "frac"])
def test_automatic_choice(M, N, K, group, kernel, dtype, zeros):
    from tilelang_ascend_amd import _abi

    lib, P = _abi.load(), _abi.ptr
    print(f"rows up to 512 M={M} N={N} K={K} g={group} {dtype} zeros={zeros}", flush=True)
    A = torch.randn(M, K, generator=gen(M)).to(dtype)
    Wp, s, z = make_w4(N, K, group, dtype, zeros, seed=M + 1)
    dA, dW, dS, dZ = A.cuda(), Wp.cuda(), s.cuda(), z.cuda()
    code = _abi.F16 if dtype is torch.float16 else _abi.BF16
    full = lib.tlq_w4a16_workspace_bytes(M, N, K)
    rows = torch.cat([torch.arange(0, 4), torch.arange(M - 6, M)])
    want = ref.ref_program_w4a16(A[rows], Wp, s, z, group, "float32")
    for size in (full, 0):  # (without a workspace: a kernel that needs none)
        ws = torch.empty(max(16, size), dtype=torch.uint8, device="cuda")
        C = torch.full((M + 4, N), 3.0, dtype=dtype, device="cuda")
        lib.tlq_debug_launch_log(1)
        rc = lib.tlq_gemm_w4a16_ws(P(dA), P(dW), P(dS), P(dZ), P(C), M, N, K, group, 0.0, code, code, _abi.ALGO_AUTO, P(ws) if size else None, size,
                                   torch.cuda.current_stream().cuda_stream)
        log = lib.tlq_debug_launch_log_text().decode()
        lib.tlq_debug_launch_log(0)
        _abi.check(rc)
        torch.cuda.synchronize()
        assert size == 0 or kernel in log or lib.tlq_device_cu_count() != 256, log
        assert bool((C[M:] == 3.0).all())  # nothing behind the result
        check_float_output(C[:M].cpu()[rows], want, f"{M} x {N} x {K}, workspace {size}")
