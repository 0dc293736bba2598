"""The kernel of four wavefronts on 256 x 256 tiles (csrc/gemm_quad.h): the fewest stages, ragged tiles, one tile, several rounds of tiles for each
work-group with ragged ones among them, and batches; int8 exact, 16-bit bit for bit what the two-stage kernel gives (the same products in
the same order) and against 64 bits."""
import os
import re
import subprocess

import pytest
import torch

from helpers import gen
from tilelang_ascend_amd import _abi, build

# 289 and 3 x 100 tiles are more than one round of 256 CUs; stages of 128 bytes of K
SHAPES = [(1, 256, 256, 2), (1, 257, 272, 3), (1, 40, 1040, 4), (2, 300, 528, 5), (1, 4330, 4240, 2), (1, 4352, 4336, 3), (3, 2500, 2448, 2), (1, 8200, 4112, 7)]


def run(mode, call):
    lib = _abi.load()
    lib.tlq_tune_gemm_tile(256), lib.tlq_tune_i8_tile(256), lib.tlq_tune_gemm_slots(mode)
    lib.tlq_debug_launch_log(1)
    try:
        rc = call(lib)
        log = lib.tlq_debug_launch_log_text().decode()
        _abi.check(rc)
    finally:
        lib.tlq_debug_launch_log(0)
        lib.tlq_tune_gemm_tile(0), lib.tlq_tune_i8_tile(0), lib.tlq_tune_gemm_slots(1)
    assert ("quad_gemm_mfma_kernel" in log) == (mode == 3), log


@pytest.mark.gpu
@pytest.mark.parametrize("B,M,N,stages", SHAPES)
@pytest.mark.parametrize("layout", ["KN", "NK"])
def test_int8(layout, B, M, N, stages):
    P, st, K = _abi.ptr, torch.cuda.current_stream().cuda_stream, 128 * stages
    print(f"quad int8 {layout} B={B} M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N)
    A = torch.randint(-127, 128, (B, M, K), dtype=torch.int8, device="cuda", generator=g)
    W = torch.randint(-127, 128, (B, K, N), dtype=torch.int8, device="cuda", generator=g)
    want = torch.stack([a.float() @ w.float() for a, w in zip(A, W)])  # (sums below 2^24: exact)
    Wd, code = (W, _abi.B_KN) if layout == "KN" else (W.transpose(1, 2).contiguous(), _abi.B_NK)
    C = torch.full((B, M, N), -1, dtype=torch.int32, device="cuda")
    run(3, lambda lib: lib.tlq_gemm_i8(P(A), P(Wd), P(C), B, M, N, K, code, st))
    assert torch.equal(C, want.to(torch.int32))
    # row scales or none, a scale per column (from a 16-byte boundary and 4 bytes behind one) or one for all, every result type
    sa, sb = torch.rand(B, M, device="cuda", generator=g) * 0.04 + 0.01, torch.rand(N + 1, device="cuda", generator=g) * 0.009 + 0.001
    for rows in (sa, None):
        for scale, n in ((sb[:N], N), (sb[1:], N), (sb[:1], 1)):
            for dtype, t in ((torch.bfloat16, _abi.BF16), (torch.float16, _abi.F16), (torch.float32, _abi.F32)):
                out = torch.full((B, M, N), -1, dtype=dtype, device="cuda")
                run(3, lambda lib: lib.tlq_gemm_w8a8(P(A), P(Wd), None if rows is None else P(rows), P(scale), P(out), B, M, N, K, n, code, t, st))
                scaled = (want if rows is None else want * rows[:, :, None]) * scale
                assert torch.equal(out, scaled.to(dtype)), (rows is None, n, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("B,M,N,stages", SHAPES)
@pytest.mark.parametrize("layout", ["KN", "NK"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_16_bit(dtype, layout, B, M, N, stages):
    P, st, K = _abi.ptr, torch.cuda.current_stream().cuda_stream, 64 * stages
    print(f"quad {dtype} {layout} B={B} M={M} N={N} K={K}", flush=True)
    A = torch.randn(B, M, K, generator=gen(M)).to(dtype).cuda()
    W = torch.randn(B, K, N, generator=gen(N)).to(dtype).cuda()
    Wd, code = (W, _abi.B_KN) if layout == "KN" else (W.transpose(1, 2).contiguous(), _abi.B_NK)
    t = _abi.F16 if dtype == torch.float16 else _abi.BF16
    for out_dtype, out in ((torch.float32, _abi.F32), (dtype, t)):
        C = [torch.full((B, M, N), -1, dtype=out_dtype, device="cuda") for _ in range(2)]
        for c, mode in zip(C, (3, 0)):
            run(mode, lambda lib: lib.tlq_gemm_f16_batched(P(A), P(Wd), P(c), B, M, N, K, t, out, code, st))
        assert torch.equal(C[0], C[1])
        if out_dtype == torch.float32:  # products are exact: what is left is the rounding of K sums in fp32, K 2^-24 of the sum of magnitudes at most
            want, size = A[-1].double() @ W[-1].double(), A[-1].double().abs() @ W[-1].double().abs()
            assert bool(((C[0][-1].double() - want).abs() <= K * 2.0 ** -24 * size).all())


@pytest.mark.gpu
def test_in_a_graph():
    """More tiles than work-groups, captured and replayed with other inputs, eager work in between."""
    B, M, N, K = 1, 8192, 4096, 1088
    A, W = torch.randn(M, K, generator=gen(1)).to(torch.bfloat16).cuda(), torch.randn(N, K, generator=gen(2)).to(torch.bfloat16).cuda()
    C, D, lib, P = torch.empty(M, N, dtype=torch.bfloat16, device="cuda"), torch.empty(M, N, dtype=torch.bfloat16, device="cuda"), _abi.load(), _abi.ptr

    def call(out):
        _abi.check(lib.tlq_gemm_f16_batched(P(A), P(W), P(out), B, M, N, K, _abi.BF16, _abi.BF16, _abi.B_NK, torch.cuda.current_stream().cuda_stream))

    lib.tlq_debug_launch_log(1)
    call(C)
    log = lib.tlq_debug_launch_log_text().decode()
    lib.tlq_debug_launch_log(0)
    assert "quad_gemm_mfma_kernel" in log or lib.tlq_device_cu_count() != 256, log
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(C)
    for seed in (3, 4, 5):
        A.copy_(torch.randn(M, K, generator=gen(seed)).to(torch.bfloat16))
        C.fill_(-1)
        torch.cuda.synchronize()
        graph.replay()
        call(D)
        torch.cuda.synchronize()
        assert torch.equal(C, D)


def test_schedule():
    """Walked on the host over several tiles of a work-group: every stage is waited for and published before it is read, loads and outputs overwrite nothing
    that someone may still read; one load more left in flight by any wait and the walk fails."""
    lib = _abi.load()
    for stages in (2, 3, 4, 5, 6, 7, 16, 33):
        for tiles in (1, 2, 3, 7):
            assert lib.tlq_debug_check_quad_schedule(stages, tiles, 0, 0) == 0, _abi.last_error()
            assert lib.tlq_debug_check_quad_schedule(stages, tiles, 1, 0) != 0
            assert "before its loads were waited for" in _abi.last_error()
            if stages * tiles > 2:
                assert lib.tlq_debug_check_quad_schedule(stages, tiles, 0, 1) != 0
                assert "before its loads were waited for" in _abi.last_error()


def code_object(tmp_path, source):
    obj, llvm = os.path.join(build.OBJ_DIR, source + ".o"), "/opt/rocm/llvm/bin"
    if not (os.path.exists(obj) and os.path.exists(f"{llvm}/clang-offload-bundler")):
        pytest.skip("objects of a build and ROCm's LLVM tools wanted")
    bundle, code = tmp_path / "bundle", tmp_path / "code"
    subprocess.run([f"{llvm}/llvm-objcopy", "--dump-section", f".hip_fatbin={bundle}", obj, str(tmp_path / "copy.o")], check=True)
    subprocess.run([f"{llvm}/clang-offload-bundler", "--unbundle", "--type=o", f"--input={bundle}", f"--targets=hipv4-amdgcn-amd-amdhsa--{build.ARCH}",
                    f"--output={code}"], check=True)
    return code, llvm


@pytest.mark.parametrize("source", ["gemm_f16", "gemm_int8"])
def test_no_spills(tmp_path, source):
    """The waits of the main loop count its loads: nothing may go through scratch memory there."""
    code, llvm = code_object(tmp_path, source)
    notes = subprocess.run([f"{llvm}/llvm-readelf", "--notes", str(code)], capture_output=True, text=True, check=True).stdout
    kernels = [(re.search(r"\.name:\s+(\S+)", k), k) for k in re.split(r"\n  - \.a(?:gpr_count|rgs)", notes)[1:]]
    quads = [(n[1], k) for n, k in kernels if n and "quad_gemm_mfma_kernel" in n[1]]
    assert len(quads) == 4
    for name, k in quads:
        assert re.search(r"\.vgpr_spill_count: (\d+)", k)[1] == "0" and re.search(r"\.private_segment_fixed_size: (\d+)", k)[1] == "0", name


def test_nothing_is_drained_for_the_scales(tmp_path):
    """A tile's scales are asked for at its start, when the tile before is still being stored and the loads of its own next stages are under way, and
    have arrived with its first stage: no wait for vector memory stands between the loop's head and its first product, nor ahead of the
    first output, where the next tile's loads are under way."""
    code, llvm = code_object(tmp_path, "gemm_int8")
    listing = subprocess.run([f"{llvm}/llvm-objdump", "-d", "--no-show-raw-insn", str(code)], capture_output=True, text=True, check=True).stdout
    kernels = [k for k in re.split(r"\n[0-9a-f]{16} (?=<)", listing) if k.startswith("<_ZN3tlq21quad_gemm_mfma_kernel") and "EpiRescale" in k.split("\n", 1)[0]]
    assert len(kernels) == 2
    for k in kernels:
        ops = [line.split("//")[0].strip() for line in k.split("\n")[1:]]

        def at(start, *names):
            return next(i for i in range(start, len(ops)) if ops[i].startswith(names))

        head, first = at(0, "s_barrier"), at(0, "v_mfma")  # (the tile loop's head lies between them)
        out = at(first, "v_accvgpr_read")
        for lo, hi in ((head, first), (out, at(out, "ds_write"))):
            assert hi > lo and not [op for op in ops[lo:hi] if "vmcnt" in op], ops[lo:hi]
