"""The small-tile W4A16 kernel (csrc/gemm_w4a16_small.hip: 16 .. 64 activation rows x 16 .. 64 weight rows per work-group, wavefronts split
K) against the oracle: every tile, ragged rows and columns, one to all k-blocks per wavefront, group sizes from a quarter of a k-block to
the whole row, every kind of zero point -- also one whose fractions start in the middle of a wavefront's slice -- and both word layouts."""
import ctypes
import re
import subprocess

import pytest
import torch

from helpers import DT, assert_bit_equal, check_float_output, gen, make_w4, w4a16_reference
from oracle import ref
from tilelang_ascend_amd import _abi, build

CODE = {torch.float16: _abi.F16, torch.bfloat16: _abi.BF16, torch.float32: _abi.F32}


def run(A, Wp, s, z, group, algo, out_dtype=None, layout=_abi.W_PLAIN, workspace=0):
    lib, P = _abi.load(), _abi.ptr
    (M, K), N = A.shape, Wp.shape[0]
    out_dtype = out_dtype or A.dtype
    zt = z.cuda() if torch.is_tensor(z) else None
    dA, dW, dS = A.cuda(), Wp.cuda(), s.cuda()
    C = torch.full((M, N), float("nan"), dtype=out_dtype, device="cuda")
    ws = torch.empty(workspace, dtype=torch.uint8, device="cuda") if workspace else None
    print(f"small tiles M={M} N={N} K={K} g={group} algo={algo} layout={layout}", flush=True)
    lib.tlq_debug_launch_log(1)
    rc = lib.tlq_gemm_w4a16_layout_ws(P(dA), P(dW), P(dS), P(zt), P(C), M, N, K, group, 0.0 if zt is not None or z is None else float(z),
                                      CODE[A.dtype], CODE[out_dtype], algo, layout, P(ws), workspace, torch.cuda.current_stream().cuda_stream)
    run.log = lib.tlq_debug_launch_log_text().decode().strip()
    lib.tlq_debug_launch_log(0)
    _abi.check(rc)
    torch.cuda.synchronize()
    return C.cpu()


@pytest.mark.gpu
@pytest.mark.parametrize("in_dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("rows,cols", [(1, 1), (1, 2), (1, 4), (2, 1), (2, 2), (2, 4), (4, 1), (4, 2), (4, 4)])
@pytest.mark.parametrize("M,N,K,group,zeros_kind,waves", [
    (1, 16, 128, 128, None, 1), (17, 36, 256, 32, "frac", 2), (33, 100, 640, 64, "mixed", 3), (64, 68, 1152, 128, "int", 4),
    (50, 1000, 2048, 2048, "scalar8", 8), (7, 260, 4224, 32, "mixed", 16),
])
def test_every_tile_against_the_oracle(in_dtype, rows, cols, M, N, K, group, zeros_kind, waves):
    dt, lib = DT[in_dtype], _abi.load()
    A = torch.randn(M, K, generator=gen(M + K)).to(dt)
    Wp, s, z = make_w4(N, K, group, dt, "int" if zeros_kind == "mixed" else zeros_kind, seed=K)
    if zeros_kind == "mixed":  # integral zero points first, fractional ones later: the dequantiser changes on the way
        z = z.clone()
        z[:, K // group // 3:] = make_w4(N, K, group, dt, "frac", seed=K + 1)[2][:, K // group // 3:]
    lib.tlq_tune_w4a16_skinny(waves, 100 * rows + 20 + cols)
    try:
        got = run(A, Wp, s, z, group, _abi.ALGO_SKINNY)
        assert "w4a16_small_kernel" in run.log, run.log
        wide = run(A, Wp, s, z, group, _abi.ALGO_SKINNY, torch.float32)
    finally:
        lib.tlq_tune_w4a16_skinny(0, 0)
    check_float_output(got, w4a16_reference(A, Wp, s, z, group), f"{rows}x{cols} tiles")
    assert_bit_equal(got, wide.to(dt), "the same sums, rounded once")


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,group", [(40, 1024, 3072, 128), (200, 300, 1024, 64), (130, 528, 512, 32), (700, 256, 384, 128), (603, 272, 1280, 64),
                                         (9, 336, 8320, 128)])
def test_automatic_choice_runs_it_on_small_problems(M, N, K, group):
    """Where its estimate is lower; the same bits by its own name, and on repacked words."""
    A = torch.randn(M, K, generator=gen(M)).half()
    Wp, s, z = make_w4(N, K, group, torch.float16, "int", seed=N)
    got = run(A, Wp, s, z, group, _abi.ALGO_AUTO)
    assert "w4a16_small_kernel" in run.log, run.log
    check_float_output(got, w4a16_reference(A, Wp, s, z, group), f"{M}x{N}x{K}")
    assert_bit_equal(run(A, Wp, s, z, group, _abi.ALGO_SMALL), got, "by name")
    Wi = ref.interleave_weight(Wp.view(torch.int8), 4, "float16").view(torch.uint8).contiguous()
    assert_bit_equal(run(A, Wi, s, z, group, _abi.ALGO_SMALL, layout=_abi.W_INTERLEAVED_F16), got, "interleaved words")


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,group", [(3952, 1120, 128, 128), (6980, 912, 128, 128), (2140, 3408, 128, 32), (7256, 480, 256, 64), (358, 13600, 128, 128),
                                         (640, 13248, 128, 64)])
def test_automatic_choice_leaves_many_results_of_short_rows_to_larger_tiles(M, N, K, group):
    """The store of the result and the activations bound these: up to 2.7 x slower in small tiles (on a machine of 256 CUs)."""
    A = torch.randn(M, K, generator=gen(M)).half()
    Wp, s, z = make_w4(N, K, group, torch.float16, "int", seed=N)
    got = run(A, Wp, s, z, group, _abi.ALGO_AUTO, workspace=_abi.load().tlq_w4a16_workspace_bytes(M, N, K))
    assert "w4a16_small_kernel" not in run.log or _abi.load().tlq_device_cu_count() != 256, run.log
    check_float_output(got, w4a16_reference(A, Wp, s, z, group), f"{M}x{N}x{K}")


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,kernel", [(64, 4096, 14336, "w4a16_stream_kernel"), (48, 4096, 4096, "w4a16_small_kernel"), (24, 8192, 10368, "w4a16_small_kernel")])
def test_long_shares_of_large_matrices_go_to_the_streaming_kernel(M, N, K, kernel):
    """Small tiles are level there while a cache holds the weights and 1.2 x slower from memory (on a machine of 256 CUs)."""
    A = torch.randn(M, K, generator=gen(M)).half()
    Wp, s, z = make_w4(N, K, 128, torch.float16, "int", seed=N)
    got = run(A, Wp, s, z, 128, _abi.ALGO_AUTO, workspace=_abi.load().tlq_w4a16_workspace_bytes(M, N, K))
    assert kernel in run.log or _abi.load().tlq_device_cu_count() != 256, run.log
    check_float_output(got, w4a16_reference(A, Wp, s, z, 128), f"{M}x{N}x{K}")


@pytest.mark.gpu
@pytest.mark.parametrize("layout", [_abi.W_PLAIN, _abi.W_INTERLEAVED_F16])
@pytest.mark.parametrize("M,N,K,group,algo,kernel", [
    (40, 1024, 768, 128, "STREAM", "w4a16_stream_kernel"), (200, 300, 256, 64, "STREAM", "w4a16_stream_kernel"), (130, 528, 512, 32, "MFMA", "tlq_gemm_w4a16(mfma)"),
    (256, 256, 256, 128, "MFMA", "tlq_gemm_w4a16(mfma)"), (40, 1024, 768, 128, "SKINNY", "w4a16_skinny_kernel"), (64, 512, 512, 64, "SKINNY", "w4a16_skinny_kernel"),
    (130, 528, 512, 32, "SMALL", "w4a16_small_kernel")])
def test_families_asked_for_by_name_run_themselves(layout, M, N, K, group, algo, kernel):
    """Also on problems that the automatic choice gives to the small-tile kernel."""
    if layout != _abi.W_PLAIN and algo in ("MFMA", "SKINNY"):
        pytest.skip("does not read repacked words")
    A = torch.randn(M, K, generator=gen(M)).half()
    Wp, s, z = make_w4(N, K, group, torch.float16, "int", seed=N)
    Wl = Wp if layout == _abi.W_PLAIN else ref.interleave_weight(Wp.view(torch.int8), 4, "float16").view(torch.uint8).contiguous()
    workspace = _abi.load().tlq_w4a16_workspace_bytes_for(M, N, K, getattr(_abi, "ALGO_" + algo)) if algo == "STREAM" else 0
    got = run(A, Wl, s, z, group, getattr(_abi, "ALGO_" + algo), layout=layout, workspace=workspace)
    assert kernel in run.log and (algo == "SMALL") == ("w4a16_small_kernel" in run.log), run.log
    check_float_output(got, w4a16_reference(A, Wp, s, z, group), f"{algo} {M}x{N}x{K}")


@pytest.mark.gpu
@pytest.mark.parametrize("layout", [_abi.W_PLAIN, _abi.W_INTERLEAVED_F16])
def test_streaming_kernel_by_name_is_refused_without_room_for_its_slices(layout):
    M, N, K, group = 64, 1024, 4096, 128
    assert _abi.load().tlq_w4a16_workspace_bytes_for(M, N, K, _abi.ALGO_STREAM) > 0
    A, (Wp, s, z) = torch.zeros(M, K).half(), make_w4(N, K, group, torch.float16, "int", seed=1)
    with pytest.raises(RuntimeError, match="streaming kernel"):
        run(A, Wp, s, z, group, _abi.ALGO_STREAM, layout=layout)
    assert run.log == ""


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,group,layout,error", [
    (700, 258, 384, 128, _abi.W_PLAIN, "N % 4"), (2420, 85, 256, 32, _abi.W_PLAIN, "N % 4"),  # rows over a multiple of four of weights: with the packed result's room only
    (40, 1024, 3072, 128, _abi.W_INTERLEAVED_F16, "workspace"), (364, 512, 3840, 32, _abi.W_INTERLEAVED_F16, "workspace")])
def test_automatic_choice_refuses_without_a_workspace_what_wants_one(M, N, K, group, layout, error):
    """Calls that the other kernels refuse for lack of room are not accepted because the small-tile kernel needs none."""
    A, (Wp, s, z) = torch.zeros(M, K).half(), make_w4(N, K, group, torch.float16, "int", seed=1)
    with pytest.raises(RuntimeError, match=error):
        run(A, Wp, s, z, group, _abi.ALGO_AUTO, layout=layout)
    assert run.log == ""
    need = max(_abi.load().tlq_w4a16_workspace_bytes(M, N, K), N * K * 2)
    run(A, Wp, s, z, group, _abi.ALGO_AUTO, layout=layout, workspace=need)
    assert "w4a16_small_kernel" in run.log, run.log


def test_small_family_refuses_what_its_kernel_does_not_read():
    lib, fake = _abi.load(), ctypes.c_void_p(1 << 20)
    for N, K, group in ((64, 192, 64), (64, 384, 96), (1, 128, 128)):  # K in whole k-blocks, power-of-two groups, an even number of scales
        rc = lib.tlq_gemm_w4a16(fake, fake, fake, None, fake, 40, N, K, group, 8.0, _abi.F16, _abi.F16, _abi.ALGO_SMALL, None)
        assert rc != 0 and "small-tile kernel needs" in _abi.last_error()
        rc = lib.tlq_gemm_w4a16_layout_ws(fake, fake, fake, None, fake, 40, N, K, group, 8.0, _abi.F16, _abi.F16, _abi.ALGO_SMALL, _abi.W_INTERLEAVED_F16, None, 0, None)
        assert rc != 0 and "small-tile kernel needs" in _abi.last_error()


def test_plan_keeps_to_the_machine():
    o = (ctypes.c_int64 * 4)()
    for M in (1, 16, 17, 40, 64, 130, 512, 5000):
        for N in (16, 100, 1024, 14336):
            for K in (128, 1024, 11008, 28672):
                assert _abi.load().tlq_debug_small_plan(M, N, K, 128, o) == 1
                bm, bn, waves, ns = o
                assert bm in (16, 32, 64) and bn in (16, 32, 64) and 1 <= waves <= min(K // 128, 16) and ns >= 5000
                assert waves * (2 * (bn * 64 + bm * 256) + 64 * bn) <= 160 * 1024 and (bm == 16 or waves <= 8)
    for bad in ((0, 16, 128, 128), (1, 16, 192, 64), (1, 16, 128, 96), (1, 16, 384, 256)):
        assert _abi.load().tlq_debug_small_plan(*bad, o) == 0


def test_no_register_spills(tmp_path):
    cmd = [build.hipcc_path(), *build.HIPCC_FLAGS, "-Rpass-analysis=kernel-resource-usage", "-c", f"{build.CSRC_DIR}/gemm_w4a16_small.hip",
           "-o", str(tmp_path / "out.o")]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout[-2000:]
    blocks = [b for b in re.split(r"remark: Function Name: ", res.stdout)[1:] if "w4a16_small_kernel" in b.split()[0]]
    assert len(blocks) == 72
    for b in blocks:
        assert re.search(r"ScratchSize \[bytes/lane\]: 0\b", b) and re.search(r"VGPRs Spill: 0\b", b), b[:300]
