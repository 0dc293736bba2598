"""The kernel of four wavefronts (csrc/gemm_quad.h) on its tiles other than 256 x 256: the fewest stages, ragged tiles, more tiles than one round of the
machine, batches; int8 exact, 16-bit bit for bit what the two-stage kernel gives (the same products in the same order) and against 64 bits."""
import os
import re
import subprocess

import pytest
import torch

from helpers import gen
from tilelang_ascend_amd import _abi, build

VARIANTS = {7: (192, 256), 8: (128, 256), 9: (256, 128), 10: (192, 128), 11: (128, 128)}
# stages of 128 bytes of K; the last two are more than one round of 256 CUs in every tile (512 work-groups of 128 x 128)
SHAPES = [(1, 128, 128, 2), (1, 193, 272, 3), (1, 40, 1040, 4), (2, 300, 144, 5), (3, 2500, 3088, 2), (1, 4330, 4240, 7)]


def run(variant, call):
    lib = _abi.load()
    lib.tlq_tune_gemm_quad(variant), lib.tlq_tune_gemm_tile(256), lib.tlq_tune_i8_tile(256), lib.tlq_tune_gemm_slots(0 if variant == 1 else 1)
    lib.tlq_debug_launch_log(1)
    try:
        rc = call(lib)
        log = lib.tlq_debug_launch_log_text().decode()
        _abi.check(rc)
    finally:
        lib.tlq_debug_launch_log(0)
        lib.tlq_tune_gemm_quad(0), lib.tlq_tune_gemm_tile(0), lib.tlq_tune_i8_tile(0), lib.tlq_tune_gemm_slots(1)
    assert variant == 1 or "quad_gemm_mfma_kernel %dx%d" % VARIANTS[variant] in log, log


@pytest.mark.gpu
@pytest.mark.parametrize("B,M,N,stages", SHAPES)
@pytest.mark.parametrize("variant", VARIANTS)
def test_int8(variant, B, M, N, stages):
    P, st, K = _abi.ptr, torch.cuda.current_stream().cuda_stream, 128 * stages
    print(f"quad tiles int8 variant={variant} B={B} M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N)
    A = torch.randint(-127, 128, (B, M, K), dtype=torch.int8, device="cuda", generator=g)
    W = torch.randint(-127, 128, (B, K, N), dtype=torch.int8, device="cuda", generator=g)
    want = torch.stack([a.float() @ w.float() for a, w in zip(A, W)])  # (sums below 2^24: exact)
    sa, sb = torch.rand(B, M, device="cuda", generator=g) * 0.04 + 0.01, torch.rand(N + 1, device="cuda", generator=g) * 0.009 + 0.001
    for Wd, code in ((W, _abi.B_KN), (W.transpose(1, 2).contiguous(), _abi.B_NK)):
        C = torch.full((B, M, N), -1, dtype=torch.int32, device="cuda")
        run(variant, lambda lib: lib.tlq_gemm_i8(P(A), P(Wd), P(C), B, M, N, K, code, st))
        assert torch.equal(C, want.to(torch.int32))
        for rows, scale, n, dtype, t in ((sa, sb[1:], N, torch.bfloat16, _abi.BF16), (None, sb[:1], 1, torch.float16, _abi.F16), (sa, sb[:N], N, torch.float32, _abi.F32)):
            out = torch.full((B, M, N), -1, dtype=dtype, device="cuda")
            run(variant, lambda lib: lib.tlq_gemm_w8a8(P(A), P(Wd), None if rows is None else P(rows), P(scale), P(out), B, M, N, K, n, code, t, st))
            scaled = (want if rows is None else want * rows[:, :, None]) * scale
            assert torch.equal(out, scaled.to(dtype)), (rows is None, n, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("B,M,N,stages", SHAPES)
@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_16_bit(dtype, variant, B, M, N, stages):
    P, st, K = _abi.ptr, torch.cuda.current_stream().cuda_stream, 64 * stages
    print(f"quad tiles {dtype} variant={variant} B={B} M={M} N={N} K={K}", flush=True)
    A = torch.randn(B, M, K, generator=gen(M)).to(dtype).cuda()
    W = torch.randn(B, K, N, generator=gen(N)).to(dtype).cuda()
    t = _abi.F16 if dtype == torch.float16 else _abi.BF16
    for Wd, code in ((W, _abi.B_KN), (W.transpose(1, 2).contiguous(), _abi.B_NK)):
        for out_dtype, out in ((torch.float32, _abi.F32), (dtype, t)):
            C = [torch.full((B, M, N), -1, dtype=out_dtype, device="cuda") for _ in range(2)]
            for c, v in zip(C, (variant, 1)):
                run(v, lambda lib: lib.tlq_gemm_f16_batched(P(A), P(Wd), P(c), B, M, N, K, t, out, code, st))
            assert torch.equal(C[0], C[1])
            if out_dtype == torch.float32:  # products are exact: what is left is the rounding of K sums in fp32, K 2^-24 of the sum of magnitudes at most
                want, size = A[-1].double() @ W[-1].double(), A[-1].double().abs() @ W[-1].double().abs()
                assert bool(((C[0][-1].double() - want).abs() <= K * 2.0 ** -24 * size).all())


@pytest.mark.parametrize("source,count", [("gemm_quad_f16", 20), ("gemm_quad_i8", 20)])
def test_no_spills(tmp_path, source, count):
    """The waits of the main loop count its loads: nothing may go through scratch memory there."""
    obj, llvm = os.path.join(build.OBJ_DIR, source + ".o"), "/opt/rocm/llvm/bin"
    if not (os.path.exists(obj) and os.path.exists(f"{llvm}/clang-offload-bundler")):
        pytest.skip("objects of a build and ROCm's LLVM tools wanted")
    bundle, code = tmp_path / "bundle", tmp_path / "code"
    subprocess.run([f"{llvm}/llvm-objcopy", "--dump-section", f".hip_fatbin={bundle}", obj, str(tmp_path / "copy.o")], check=True)
    subprocess.run([f"{llvm}/clang-offload-bundler", "--unbundle", "--type=o", f"--input={bundle}", f"--targets=hipv4-amdgcn-amd-amdhsa--{build.ARCH}",
                    f"--output={code}"], check=True)
    notes = subprocess.run([f"{llvm}/llvm-readelf", "--notes", str(code)], capture_output=True, text=True, check=True).stdout
    kernels = [(re.search(r"\.name:\s+(\S+)", k), k) for k in re.split(r"\n  - \.a(?:gpr_count|rgs)", notes)[1:]]
    quads = [(n[1], k) for n, k in kernels if n and "quad_gemm_mfma_kernel" in n[1]]
    assert len(quads) == count
    for name, k in quads:
        assert re.search(r"\.vgpr_spill_count: (\d+)", k)[1] == "0" and re.search(r"\.private_segment_fixed_size: (\d+)", k)[1] == "0", name
