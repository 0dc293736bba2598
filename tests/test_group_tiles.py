"""The ring kernel (csrc/gemm_ring.h) in the place of 128-row tiles: every tile, both weight layouts, even and odd stages of K, a partial last stage, ragged rows and columns, batches, every epilogue -- integers bit for bit, 16-bit results against fp64; the estimate's choice."""
import pytest
import torch

from helpers import assert_bit_equal, gen
from tilelang_ascend_amd import _abi

CODE = {torch.float16: _abi.F16, torch.bfloat16: _abi.BF16, torch.float32: _abi.F32}
# (batch, M, N, 128-byte stages of K, bytes of K in a partial stage behind them): parts of 2 / 3 / 4 stages and uneven ones, tiles cut on both sides
SHAPES = [(1, 128, 128, 4, 0), (1, 130, 144, 5, 0), (2, 63, 272, 6, 64), (1, 300, 48, 7, 32), (3, 129, 64, 9, 0), (1, 65, 400, 16, 96)]


@pytest.fixture
def lib():
    lib = _abi.load()
    yield lib
    lib.tlq_tune_gemm_groups(0), lib.tlq_tune_gemm_tile(0), lib.tlq_tune_i8_tile(0)


def called(lib, rc, groups=True):
    log = lib.tlq_debug_launch_log_text().decode()
    lib.tlq_debug_launch_log(0)
    _abi.check(rc)
    torch.cuda.synchronize()
    assert "gemm_mfma_kernel" in log and ("groups of wavefronts" in log) == groups and log.count("[") == 1, log


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [2, 3, 4, 5])
@pytest.mark.parametrize("B,M,N,stages,tail", SHAPES)
def test_int8(lib, variant, B, M, N, stages, tail):
    print(f"groups int8 variant={variant} B={B} M={M} N={N} stages={stages}+{tail}", flush=True)
    P, st, K = _abi.ptr, torch.cuda.current_stream().cuda_stream, stages * 128 + tail
    lib.tlq_tune_gemm_groups(variant), lib.tlq_tune_i8_tile(128)
    A = torch.randint(-127, 128, (B, M, K), dtype=torch.int8, generator=gen(1))
    W = torch.randint(-127, 128, (B, K, N), dtype=torch.int8, generator=gen(2))
    sa, sb = torch.rand(B, M, generator=gen(3)), torch.rand(N, generator=gen(4))
    acc = torch.bmm(A.double(), W.double()).to(torch.int32)
    dA, dsa, dsb = A.cuda(), sa.cuda(), sb.cuda()
    for layout, dW in ((_abi.B_KN, W.cuda()), (_abi.B_NK, W.transpose(1, 2).contiguous().cuda())):
        C = torch.full((B, M, N), -1, dtype=torch.int32, device="cuda")
        lib.tlq_debug_launch_log(1)
        called(lib, lib.tlq_gemm_i8(P(dA), P(dW), P(C), B, M, N, K, layout, st))
        assert torch.equal(C.cpu(), acc)
        for dt in CODE:
            out = torch.full((B, M, N), float("nan"), dtype=dt, device="cuda")
            lib.tlq_debug_launch_log(1)
            called(lib, lib.tlq_gemm_w8a8(P(dA), P(dW), P(dsa), P(dsb), P(out), B, M, N, K, N, layout, CODE[dt], st))
            assert_bit_equal(out.cpu(), ((acc.float() * sa[:, :, None]) * sb).to(dt), f"rescaled {dt}")


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [2, 3, 4, 5])
@pytest.mark.parametrize("B,M,N,stages,tail", SHAPES)
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_float(lib, variant, B, M, N, stages, tail, dt):
    print(f"groups {dt} variant={variant} B={B} M={M} N={N} stages={stages}+{tail}", flush=True)
    P, st, K = _abi.ptr, torch.cuda.current_stream().cuda_stream, stages * 64 + tail // 2
    lib.tlq_tune_gemm_groups(variant), lib.tlq_tune_gemm_tile(128)
    A, W = torch.randn(B, M, K, generator=gen(1)).to(dt), torch.randn(B, K, N, generator=gen(2)).to(dt)
    want = torch.bmm(A.double(), W.double())
    # fp32 sums of K exact products: at most K * 2^-24 of the sum of their magnitudes
    bound = K * 2.0**-24 * torch.bmm(A.double().abs(), W.double().abs())
    dA = A.cuda()
    for layout, dW in ((_abi.B_KN, W.cuda()), (_abi.B_NK, W.transpose(1, 2).contiguous().cuda())):
        for out_dt, half_ulp in ((torch.float32, 2.0**-24), (dt, 2.0**-11 if dt is torch.float16 else 2.0**-8)):
            C = torch.full((B, M, N), float("nan"), dtype=out_dt, device="cuda")
            lib.tlq_debug_launch_log(1)
            called(lib, lib.tlq_gemm_f16_batched(P(dA), P(dW), P(C), B, M, N, K, CODE[dt], CODE[out_dt], layout, st))
            assert bool(((C.cpu().double() - want).abs() <= bound + half_ulp * (want.abs() + bound) + 2.0**-25).all())


@pytest.mark.gpu
def test_taken_where_tiles_leave_one_work_group_to_a_cu(lib):
    P, st = _abi.ptr, torch.cuda.current_stream().cuda_stream
    for M, N, K, groups in ((1000, 4096, 4096, True), (2000, 4096, 4096, False)):
        A, W = torch.randn(M, K, generator=gen(1)).half(), torch.randn(K, N, generator=gen(2)).half()
        C, dA, dW = torch.empty(M, N, dtype=torch.float16, device="cuda"), A.cuda(), W.cuda()
        lib.tlq_debug_launch_log(1)
        called(lib, lib.tlq_gemm_f16(P(dA), P(dW), P(C), M, N, K, _abi.F16, _abi.F16, _abi.B_KN, st), groups)
    # (280 tiles of 128 x 128; 504 of 128 x 64 would be two rounds)
    A, W = torch.randn(8, 780, 1024, generator=gen(1)).half().cuda(), torch.randn(8, 1024, 528, generator=gen(2)).half().cuda()
    C = torch.empty(8, 780, 528, dtype=torch.float16, device="cuda")
    lib.tlq_debug_launch_log(1)
    called(lib, lib.tlq_gemm_f16_batched(P(A), P(W), P(C), 8, 780, 528, 1024, _abi.F16, _abi.F16, _abi.B_KN, st), False)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,launches", [(4099, 4096, 1024, 2), (4096, 4096, 1024, 1), (7314, 2384, 384, 1), (7314, 2384, 768, 2)])
def test_rows_of_full_rounds_and_the_rest(lib, M, N, K, launches):
    """One tile row too many for a round of the machine: the rest of the rows is a launch of its own (checked on a machine of 256 CUs), at the
    right rows of the activations, the scales and the result.  Not on rows of fewer than six 128-byte stages, where it is behind one launch."""
    print(f"full rounds M={M} N={N} K={K}", flush=True)
    P, st = _abi.ptr, torch.cuda.current_stream().cuda_stream
    A = torch.randint(-127, 128, (M, K), dtype=torch.int8, generator=gen(1)).cuda()
    W = torch.randint(-127, 128, (N, K), dtype=torch.int8, generator=gen(2)).cuda()
    sa, sb = torch.rand(M, generator=gen(3)).cuda(), torch.rand(N, generator=gen(4)).cuda()
    acc = (A.double() @ W.double().T).to(torch.int32)  # exact

    def count(rc):
        log = lib.tlq_debug_launch_log_text().decode()
        lib.tlq_debug_launch_log(0)
        _abi.check(rc)
        torch.cuda.synchronize()
        assert lib.tlq_device_cu_count() != 256 or log.count("[") == launches, log

    C = torch.full((M, N), -1, dtype=torch.int32, device="cuda")
    lib.tlq_debug_launch_log(1)
    count(lib.tlq_gemm_i8(P(A), P(W), P(C), 1, M, N, K, _abi.B_NK, st))
    assert torch.equal(C, acc)
    for dt in CODE:
        for scale in (sa, None):
            out = torch.full((M, N), float("nan"), dtype=dt, device="cuda")
            lib.tlq_debug_launch_log(1)
            count(lib.tlq_gemm_w8a8(P(A), P(W), None if scale is None else P(scale), P(sb), P(out), 1, M, N, K, N, _abi.B_NK, CODE[dt], st))
            want = ((acc.float() if scale is None else acc.float() * scale[:, None]) * sb).to(dt)
            assert_bit_equal(out.cpu(), want.cpu(), f"rescaled {dt}")


@pytest.mark.gpu
@pytest.mark.parametrize("op,B,M,N,K,kernel", [
    ("w8a8 NK", 1, 180, 1456, 512, "gemm_small_kernel"), ("w8a8 NK", 1, 226, 1232, 512, "gemm_small_kernel"),
    ("f16 KN", 2, 77, 3312, 512, "ring_gemm"), ("f16 KN", 4, 215, 896, 512, "ring_gemm"), ("f16 KN", 4, 210, 720, 640, "ring_gemm")])
def test_small_tiles_or_the_ring_kernel_on_short_rows(op, B, M, N, K, kernel):
    """Problems where one of the two is ahead by 15 to 40 % and the choice had it the other way round when it compared the small tiles with another kernel."""
    lib, P, st = _abi.load(), _abi.ptr, torch.cuda.current_stream().cuda_stream
    if lib.tlq_device_cu_count() != 256:
        pytest.skip("the estimates are of 256 compute units")
    lay = _abi.B_KN if op.endswith("KN") else _abi.B_NK
    print(f"choice {op} B={B} M={M} N={N} K={K}", flush=True)
    lib.tlq_debug_launch_log(1)
    if op.startswith("f16"):
        A, W, C = torch.zeros(B, M, K, dtype=torch.float16, device="cuda"), torch.zeros(B, K, N, dtype=torch.float16, device="cuda"), torch.empty(B, M, N, dtype=torch.float16, device="cuda")
        rc = lib.tlq_gemm_f16_batched(P(A), P(W), P(C), B, M, N, K, _abi.F16, _abi.F16, lay, st)
    else:
        A, W, C = torch.zeros(B, M, K, dtype=torch.int8, device="cuda"), torch.zeros(B, K, N, dtype=torch.int8, device="cuda"), torch.empty(B, M, N, dtype=torch.bfloat16, device="cuda")
        sa, sb = torch.ones(B, M, device="cuda"), torch.ones(N, device="cuda")
        rc = lib.tlq_gemm_w8a8(P(A), P(W), P(sa), P(sb), P(C), B, M, N, K, N, lay, _abi.BF16, st)
    log = lib.tlq_debug_launch_log_text().decode()
    lib.tlq_debug_launch_log(0)
    _abi.check(rc)
    assert kernel in log, log
