"""W4A16 above 512 rows: where the automatic choice takes the two passes by estimate (row counts that are no multiple of four, many rounds of short
rows, few output tiles), with room for them and -- the kernels that ran before -- without."""
import pytest
import torch

from helpers import gen
from tilelang_ascend_amd import _abi

# 639: three rows over; 4868: short rows in a round and a sixteenth; 614 / 667: few output tiles; 1037: one row over, two stages of K per step
SHAPES = [(639, 5680, 896, 128), (4868, 3152, 384, 128), (614, 1392, 2304, 128), (667, 256, 12288, 128), (1037, 3488, 384, 64)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,group", SHAPES)
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tensor", [True, False])
def test_two_passes_by_estimate(M, N, K, group, dt, tensor):
    print(f"two passes M={M} N={N} K={K} g={group} {dt} tensor={tensor}", flush=True)
    lib, P, st = _abi.load(), _abi.ptr, torch.cuda.current_stream().cuda_stream
    code = _abi.F16 if dt is torch.float16 else _abi.BF16
    A = torch.randn(M, K, generator=gen(1)).to(dt).cuda()
    W = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, generator=gen(2)).cuda()
    S = (torch.rand(N, K // group, generator=gen(3)) * 0.015 + 0.005).to(dt).cuda()
    Z = torch.randint(6, 10, (N, K // group), generator=gen(4)).to(dt).cuda() if tensor else None
    u = torch.stack([W & 15, W >> 4], -1).reshape(N, K // group, group).to(dt)
    w = ((u - (Z[:, :, None] if tensor else torch.tensor(8, dtype=dt, device="cuda"))) * S[:, :, None]).reshape(N, K)  # each operation rounded to dt
    want, size = A.double() @ w.double().T, A.double().abs() @ w.double().abs().T
    # fp32 sums of K exact products (partial sums in any order), then the result's own rounding
    tol = K * 2.0**-24 * size + (2.0**-11 if dt is torch.float16 else 2.0**-8) * (want.abs() + K * 2.0**-24 * size) + 2.0**-25
    # the last one or two fp16 rows go to the GEMV, which applies scale and zero point to the group's sum: its weights are not rounded to fp16,
    # half an ulp each
    bound = tol.clone()
    if dt is torch.float16 and M % 4 in (1, 2):
        bound[M & ~3:] += 2.0**-11 * size[M & ~3:]
    full = lib.tlq_w4a16_workspace_bytes(M, N, K)
    for size_ws in (full, N * K * 2, 0):
        ws = torch.empty(size_ws + 16, dtype=torch.uint8, device="cuda")
        C = torch.full((M, N), float("nan"), dtype=dt, device="cuda")
        lib.tlq_debug_launch_log(1)
        rc = lib.tlq_gemm_w4a16_ws(P(A), P(W), P(S), P(Z) if tensor else None, P(C), M, N, K, group, 0.0 if tensor else 8.0, code, code, _abi.ALGO_AUTO,
                                   P(ws) if size_ws else None, size_ws, st)
        log = lib.tlq_debug_launch_log_text().decode()
        lib.tlq_debug_launch_log(0)
        _abi.check(rc)
        torch.cuda.synchronize()
        assert ("dequant_w4" in log) == (size_ws > 0) or lib.tlq_device_cu_count() != 256, log
        assert bool(((C.double() - want).abs() <= bound).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,group", [(1037, 3488, 384, 64), (637, 5680, 896, 128), (513, 256, 384, 128), (601, 272, 1280, 64), (1030, 8192, 256, 64),
                                         (614, 1392, 2304, 128)])
@pytest.mark.parametrize("tensor", [True, False])
def test_last_fp16_rows_keep_the_gemv_kernels_precision(M, N, K, group, tensor):
    """The last one or two fp16 rows of a row count that is no multiple of four, where they belong to the GEMV kernels: those apply scale and
    zero point to fp32 sums, so their rows agree with the product of UNROUNDED weights to fp32 sums and the result's own rounding --
    whatever kernel runs the rows above, with room for two passes and without."""
    print(f"last rows M={M} N={N} K={K} g={group} tensor={tensor}", flush=True)
    lib, P, st = _abi.load(), _abi.ptr, torch.cuda.current_stream().cuda_stream
    A = torch.randn(M, K, generator=gen(5)).half().cuda()
    W = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, generator=gen(6)).cuda()
    S = (torch.rand(N, K // group, generator=gen(7)) * 0.015 + 0.005).half().cuda()
    Z = (torch.rand(N, K // group, generator=gen(8)) * 3 + 6).half().cuda() if tensor else None
    zs = 0.0 if tensor else 7.5
    head = M & ~3

    def run(fn, a, rows, *ws):
        C = torch.full((rows, N), float("nan"), dtype=torch.float16, device="cuda")
        _abi.check(fn(P(a), P(W), P(S), P(Z), P(C), rows, N, K, group, zs, _abi.F16, _abi.F16, _abi.ALGO_AUTO, *ws, st))
        return C

    last = run(lib.tlq_gemm_w4a16, A[head:], M - head)
    lib.tlq_debug_launch_log(1)
    run(lib.tlq_gemm_w4a16, A[head:], M - head)
    gemv = "gemv" in lib.tlq_debug_launch_log_text().decode().lower()
    lib.tlq_debug_launch_log(0)
    assert gemv or lib.tlq_device_cu_count() != 256
    u = torch.stack([W & 15, W >> 4], -1).reshape(N, K // group, group).double()
    exact = ((u - (Z.double()[:, :, None] if tensor else zs)) * S.double()[:, :, None]).reshape(N, K)
    a = A[head:].double()
    # fp32: s (sum a u - z sum a) per chunk, sums of K products of up to (u + |z|) s |a| in any order; then the result's rounding
    size = a.abs() @ ((u + (Z.double()[:, :, None].abs() if tensor else zs)) * S.double()[:, :, None]).reshape(N, K).T
    want = a @ exact.T
    bound = K * 2.0**-24 * size + 2.0**-11 * (want.abs() + K * 2.0**-24 * size) + 2.0**-25
    for size_ws in (lib.tlq_w4a16_workspace_bytes(M, N, K), N * K * 2, 0):
        ws = torch.empty(size_ws + 16, dtype=torch.uint8, device="cuda")
        C = run(lib.tlq_gemm_w4a16_ws, A, M, P(ws) if size_ws else None, size_ws)
        torch.cuda.synchronize()
        assert torch.equal(C[head:], last)
        assert not gemv or bool(((C[head:].double() - want).abs() <= bound).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,group,dt", [(8192, 4096, 4096, 64, torch.float16), (4907, 256, 2048, 64, torch.bfloat16), (881, 528, 3968, 128, torch.bfloat16), (1237, 2912, 2688, 128, torch.bfloat16)])
def test_two_passes_take_all_rows(M, N, K, group, dt):
    """Large products, many rows on few weights, and row counts that are no multiple of four where no panel kernel would run: the dequantisation pass and
    one product over all rows; the same bits as the two passes by name."""
    lib, P, st = _abi.load(), _abi.ptr, torch.cuda.current_stream().cuda_stream
    print(f"two passes for all rows M={M} N={N} K={K} g={group} {dt}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M)
    A = torch.randn(M, K, device="cuda", generator=g).to(dt)
    Wp = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, device="cuda", generator=g)
    s = (torch.rand(N, K // group, device="cuda", generator=g) * 0.015 + 0.005).to(dt)
    z = torch.randint(6, 10, (N, K // group), device="cuda", generator=g).to(dt)
    size = lib.tlq_w4a16_workspace_bytes_for(M, N, K, _abi.ALGO_AUTO)
    ws = torch.empty(size, dtype=torch.uint8, device="cuda")
    t, C = (_abi.F16 if dt == torch.float16 else _abi.BF16), [torch.empty(M, N, dtype=dt, device="cuda") for _ in range(2)]
    for c, algo in zip(C, (_abi.ALGO_AUTO, _abi.ALGO_TWO_PASS)):
        lib.tlq_debug_launch_log(1)
        rc = lib.tlq_gemm_w4a16_ws(P(A), P(Wp), P(s), P(z), P(c), M, N, K, group, 0.0, t, t, algo, P(ws), size, st)
        log = lib.tlq_debug_launch_log_text().decode()
        lib.tlq_debug_launch_log(0)
        _abi.check(rc)
        assert ("dequant_w4" in log and log.count("tlq_gemm_w4a16") == 0) or lib.tlq_device_cu_count() != 256, log
    assert torch.equal(C[0], C[1])
