"""Row counts above 512 that are no multiple of four, bfloat16: the last one to three rows lie in the last tile of the four-wavefront panel kernels
or the streaming kernel and go along with them, or -- where they would need a tile row of their own -- run as before in a launch of their own."""
import pytest
import torch

from helpers import check_float_output, gen, make_w4
from oracle import ref


@pytest.mark.parametrize("rows", [1, 2, 3, 5, 511, 513, 514, 515, 767, 769, 1021])
@pytest.mark.parametrize("N,K,group", [(272, 1024, 128), (16, 1024, 64)])
def test_loads_of_a_partial_block_of_rows_stay_inside_the_matrix(rows, N, K, group):
    from tilelang_ascend_amd import _abi

    lib = _abi.load()
    assert lib.tlq_debug_check_panel256_addressing(rows, N, K, group, K // 128) == 0, _abi.last_error()
    for tile in (64, 128):
        assert lib.tlq_debug_check_panelm_addressing(rows, N, K, group, tile, K // 128) == 0, _abi.last_error()


# (M, N, K, group): in the last tile of the 256-row kernel; of the 128-row one; a tile row of their own; in a block of the streaming kernel, with K slices and without
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,group,along", [(1002, 8960, 1152, 64, True), (1023, 8960, 1152, 64, True), (1025, 8960, 1152, 64, False),
                                               (601, 11008, 4096, 128, True), (639, 11008, 4096, 128, True), (641, 11008, 4096, 128, False),
                                               (2209, 14224, 1536, 128, True), (839, 6144, 2048, 64, True), (641, 7936, 4224, 128, True),
                                               (590, 1664, 5120, 128, True), (1207, 1024, 6144, 64, True)])
@pytest.mark.parametrize("zeros", ["int", "frac", None])
def test_last_bfloat16_rows_go_along(M, N, K, group, along, zeros):
    from tilelang_ascend_amd import _abi

    lib, P = _abi.load(), _abi.ptr
    print(f"rows behind M={M} N={N} K={K} g={group} zeros={zeros}", flush=True)
    A = torch.randn(M, K, generator=gen(M)).bfloat16()
    Wp, s, z = make_w4(N, K, group, torch.bfloat16, zeros or "int", seed=M + 1)
    z = z if zeros else None
    dA, dW, dS, dZ = A.cuda(), Wp.cuda(), s.cuda(), z.cuda() if zeros else None
    ws = torch.empty(max(16, lib.tlq_w4a16_workspace_bytes(M, N, K)), dtype=torch.uint8, device="cuda")
    C = torch.full((M + 4, N), 3.0, dtype=torch.bfloat16, device="cuda")
    lib.tlq_debug_launch_log(1)
    rc = lib.tlq_gemm_w4a16_ws(P(dA), P(dW), P(dS), P(dZ) if zeros else None, P(C), M, N, K, group, 0.0 if zeros else 8.0, _abi.BF16, _abi.BF16, _abi.ALGO_AUTO,
                               P(ws), ws.numel(), torch.cuda.current_stream().cuda_stream)
    log = lib.tlq_debug_launch_log_text().decode().strip()
    lib.tlq_debug_launch_log(0)
    _abi.check(rc)
    torch.cuda.synchronize()
    if lib.tlq_device_cu_count() == 256 and "dequant" not in log:
        assert (len([l for l in log.split(" + ") if "reduce" not in l]) == 1) == along, log
    assert bool((C[M:] == 3.0).all())  # nothing behind the result
    head = M - M % 4 - 4
    rows = torch.cat([torch.arange(0, 8), torch.arange(head, M)])
    check_float_output(C[:M].cpu()[rows], ref.ref_program_w4a16(A[rows], Wp, s, z if zeros else 8, group, "float32"), "rows behind")
