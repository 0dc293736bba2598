"""W4A16 on 129 to 512 rows: where the automatic choice, in both word layouts, takes the streaming kernel and where one of the others, at problems where
the prices that the rules put on the streaming kernel were those of another geometry.  Seen in the launch log and, bit for bit, in the named
kernel's result.  The times beside the problems: the kernel that is to run, then the one that ran."""
import ctypes

import pytest
import torch

from helpers import assert_bit_equal
from tilelang_ascend_amd import _abi

KERNEL = {_abi.ALGO_STREAM: "w4a16_stream_kernel", _abi.ALGO_PANEL256: "w4a16_panel256_kernel", _abi.ALGO_PANELM: "w4a16_panelm_kernel"}


def run(M, N, K, group, layout, algo, dtype=torch.float16):
    lib, P, st = _abi.load(), _abi.ptr, torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randn(M, K, generator=g, device="cuda", dtype=dtype)
    W = torch.randint(0, 256, (N, K // 2), generator=g, device="cuda", dtype=torch.uint8)
    S = (torch.rand(N, K // group, generator=g, device="cuda") * 0.015 + 0.005).to(dtype)
    Z = torch.randint(6, 10, (N, K // group), generator=g, device="cuda").to(dtype)
    need = int(lib.tlq_w4a16_workspace_bytes(M, N, K) if algo == _abi.ALGO_AUTO else lib.tlq_w4a16_workspace_bytes_for(M, N, K, algo))
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    C = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
    code = _abi.F16 if dtype is torch.float16 else _abi.BF16
    print(f"stream choice M={M} N={N} K={K} g={group} layout={layout} algo={algo} {dtype}", flush=True)
    lib.tlq_debug_launch_log(1)
    rc = lib.tlq_gemm_w4a16_layout_ws(P(A), P(W), P(S), P(Z), P(C), M, N, K, group, 0.0, code, code, algo, layout, P(ws) if need else None, need, st)
    log = lib.tlq_debug_launch_log_text().decode()
    lib.tlq_debug_launch_log(0)
    _abi.check(rc)
    torch.cuda.synchronize()
    return C, log


def check(M, N, K, group, layout, algo, dtype=torch.float16):
    got, log = run(M, N, K, group, layout, _abi.ALGO_AUTO, dtype)
    if _abi.load().tlq_device_cu_count() != 256:
        pytest.skip("the choices are those of 256 compute units")
    assert KERNEL[algo] in log, log
    assert_bit_equal(got.cpu(), run(M, N, K, group, layout, algo, dtype)[0].cpu(), f"{M}x{N}x{K} g{group} layout {layout}: automatic choice vs the named kernel")


@pytest.mark.gpu
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("M,N,K,group,algo", [
    # against the 256-row panel kernel: plans of four groups of wavefronts (blocks of 128 weight rows)
    (256, 11008, 5504, 128, _abi.ALGO_STREAM),   # 45.4, 71.2 us
    (384, 8192, 6912, 128, _abi.ALGO_STREAM),    # 53.2, 69.8
    (512, 4096, 11008, 64, _abi.ALGO_STREAM),    # 61.0, 72.3
    (256, 5120, 13824, 128, _abi.ALGO_STREAM),   # 49.4, 65.4
    (512, 6144, 14720, 128, _abi.ALGO_PANEL256), # 87.7 (the streaming kernel 105.1)
    (448, 18944, 3584, 64, _abi.ALGO_PANEL256),  # 82.7 (100.4), two groups
    (472, 20352, 1152, 32, _abi.ALGO_PANEL256),  # 32.0 (39.7), short rows of a wide matrix
    (316, 24960, 256, 128, _abi.ALGO_PANEL256),  # 16.8 (20.2)
])
def test_against_the_256_row_kernel(M, N, K, group, layout, algo):
    check(M, N, K, group, layout, algo)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("M,N,K,group,dtype", [
    # against the tile kernel over K slices and the two passes: more work-groups than compute units, group counts that the panel kernels do not take
    (318, 24192, 8576, 128, torch.float16),   # 213, 300 and 333 us
    (295, 23424, 3968, 128, torch.bfloat16),  # 93, 129, 142
    (407, 19968, 2048, 256, torch.float16),   # 50, 80, 64
    (319, 3200, 12800, 32, torch.float16),    # 51, 89, 74
    (384, 20480, 1920, 32, torch.bfloat16),   # 38, 92, 53
    (446, 8192, 7680, 32, torch.float16),     # 61, 108, 105
])
def test_against_k_slices_and_two_passes(M, N, K, group, layout, dtype):
    if layout and dtype is torch.bfloat16:
        pytest.skip("repacked words are for float16")
    check(M, N, K, group, layout, _abi.ALGO_STREAM, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,group,dtype,algo", [
    # against the middle-M kernel in whole rounds of its work-groups
    (224, 8192, 4096, 128, torch.float16, _abi.ALGO_STREAM),   # 27.9, 31.6 us: the second tile of 128 rows partly filled
    (232, 8192, 6656, 64, torch.float16, _abi.ALGO_STREAM),    # 39.4, 46.3
    (252, 2048, 16384, 128, torch.float16, _abi.ALGO_STREAM),  # 30.1, 33.1
    (256, 8192, 4096, 128, torch.bfloat16, _abi.ALGO_STREAM),  # 28.1, 31.9
    (256, 4096, 8192, 64, torch.bfloat16, _abi.ALGO_STREAM),
    (256, 8192, 5120, 64, torch.float16, _abi.ALGO_STREAM),    # 34.4, 40.4: K slices of 12 steps
    (256, 8192, 4096, 128, torch.float16, _abi.ALGO_PANELM),
])
def test_against_whole_rounds_of_the_middle_m_kernel(M, N, K, group, dtype, algo):
    check(M, N, K, group, 0, algo, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,dtype", [
    # against small tiles, groups of 32 with zero points
    (154, 6016, 3200, torch.float16),   # 25.5, 34.5 us
    (44, 12224, 3584, torch.bfloat16),  # 20.0, 24.0
    (213, 4304, 2304, torch.bfloat16),  # 19.8, 23.2
])
def test_against_small_tiles_in_groups_of_32(M, N, K, dtype):
    check(M, N, K, 32, 0, _abi.ALGO_STREAM, dtype)


@pytest.mark.parametrize("M,N,K,group", [
    (188, 18128, 3200, 64),  # 284 work-groups of 96 x 128 rows 49.6 us, 142 of 96 x 256 35.0
    (133, 18432, 1920, 32),  # 288 35.7, 144 25.4
    (223, 17408, 5248, 32),  # 272 96.6, 204 69.0
    (472, 8352, 4992, 32),   # 264 92.1, 165 70.0
    (69, 23296, 8064, 64),   # 364 in four K slices 80.2, 182 in two 61.4
    (47, 32896, 3840, 64),   # 257 51.9, 129 39.7
])
def test_plans_leave_no_few_work_groups_for_a_second_round(M, N, K, group):
    plan = (ctypes.c_int64 * 5)()
    assert _abi.load().tlq_debug_stream_plan(M, N, K, group, 256, plan) == 1
    rows, weight_rows, slices, steps, _ = plan
    assert -(-M // rows) * -(-N // weight_rows) * slices <= 256 and slices * steps >= K // 128


def test_the_workspace_size_follows_the_switch():
    """Above 512 rows the size counts the streaming kernel's K slices: one asked for with the kernel off is not handed out once it is on again."""
    lib = _abi.load()
    M, N, K = 640, 12, 1664
    lib.tlq_tune_w4a16_stream(1)
    on = lib.tlq_w4a16_workspace_bytes(M, N, K)
    try:
        lib.tlq_tune_w4a16_stream(0)
        off = lib.tlq_w4a16_workspace_bytes(M, N, K)
    finally:
        lib.tlq_tune_w4a16_stream(1)
    plan = (ctypes.c_int64 * 5)()
    assert lib.tlq_debug_stream_plan(M, N, K, 32, lib.tlq_device_cu_count() or 256, plan) == 1
    assert on >= plan[2] * M * N * 4 > off
    assert lib.tlq_w4a16_workspace_bytes(M, N, K) == on


@pytest.mark.parametrize("M,N,K", [(512, 4096, 14336), (400, 8192, 8192), (64, 4096, 14336), (200, 4096, 4096), (96, 20480, 2048)])
def test_the_size_by_name_is_the_most_slices_of_any_plan(M, N, K):
    """No slices that no plan cuts: in the size by name, which is what a call by name needs for the group size that cuts most."""
    lib = _abi.load()
    plan = (ctypes.c_int64 * 5)()
    slices = []
    for shift in range(5, 14):
        if K % (1 << shift) == 0 and lib.tlq_debug_stream_plan(M, N, K, 1 << shift, lib.tlq_device_cu_count() or 256, plan) == 1:
            slices.append(plan[2])
    most = max(slices)
    assert lib.tlq_w4a16_workspace_bytes_for(M, N, K, _abi.ALGO_STREAM) == (most * M * N * 4 if most > 1 else 0)
    assert lib.tlq_w4a16_workspace_bytes(M, N, K) >= most * M * N * 4 or most == 1
