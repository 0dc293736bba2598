"""The small-tile kernel of the int8, W4A8 and plain 16-bit products (csrc/gemm_small.h): every tile and weight layout, ragged rows and
columns, one wavefront to all, batches, every epilogue and sign convention -- integers bit for bit, 16-bit results against fp32."""
import ctypes
import re
import subprocess

import pytest
import torch

from helpers import assert_bit_equal, check_float_output, gen
from tilelang_ascend_amd import _abi, build

CODE = {torch.float16: _abi.F16, torch.bfloat16: _abi.BF16, torch.float32: _abi.F32}


@pytest.fixture
def lib():
    yield _abi.load()
    _abi.load().tlq_tune_small(0, 0)


def i8(seed, *shape):
    return torch.randint(-127, 128, shape, dtype=torch.int8, generator=gen(seed))


def called(lib, rc):
    log = lib.tlq_debug_launch_log_text().decode()
    lib.tlq_debug_launch_log(0)
    _abi.check(rc)
    torch.cuda.synchronize()
    assert "gemm_small_kernel" in log and log.count("[") == 1, log


TILES = [(1, 1), (2, 1), (4, 1), (1, 2), (2, 2), (4, 2), (1, 4), (2, 4), (4, 4)]  # activation tiles, weight tiles
SHAPES = [(1, 16, 128, 1), (17, 48, 256, 2), (33, 80, 640, 3), (64, 272, 1152, 4), (70, 1008, 2048, 8), (5, 144, 4224, 16)]


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", TILES)
@pytest.mark.parametrize("M,N,K,waves", SHAPES)
def test_int8_weights_by_rows_and_packed(lib, rows, cols, M, N, K, waves):
    P, st = _abi.ptr, torch.cuda.current_stream().cuda_stream
    print(f"small int8 {rows}x{cols} M={M} N={N} K={K} waves={waves}", flush=True)
    lib.tlq_tune_small(waves, 10 * rows + cols)
    A, W, sa, sb = i8(1, M, K), i8(2, N, K), torch.rand(M, generator=gen(3)), torch.rand(N, generator=gen(4))
    dA, dW, dsa, dsb = A.cuda(), W.cuda(), sa.cuda(), sb.cuda()
    acc = (A.double() @ W.double().T).to(torch.int32)  # exact
    C = torch.full((M, N), -1, dtype=torch.int32, device="cuda")
    lib.tlq_debug_launch_log(1)
    called(lib, lib.tlq_gemm_i8(P(dA), P(dW), P(C), 1, M, N, K, _abi.B_NK, st))
    assert torch.equal(C.cpu(), acc)
    for dt in (torch.float16, torch.bfloat16, torch.float32):
        out = torch.full((M, N), float("nan"), dtype=dt, device="cuda")
        lib.tlq_debug_launch_log(1)
        called(lib, lib.tlq_gemm_w8a8(P(dA), P(dW), P(dsa), P(dsb), P(out), 1, M, N, K, N, _abi.B_NK, CODE[dt], st))
        assert_bit_equal(out.cpu(), ((acc.float() * sa[:, None]) * sb).to(dt), f"rescaled {dt}")
    Wp = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, generator=gen(5))
    dWp = Wp.cuda()
    u = torch.stack([Wp & 15, Wp >> 4], -1).reshape(N, K).to(torch.int32)
    for mode, w in ((_abi.U4, u), (_abi.S4_TWOS, torch.where(u >= 8, u - 16, u)), (_abi.S4_OFFSET8, u - 8), (_abi.S4_OFFSET7, u - 7)):
        lib.tlq_debug_launch_log(1)
        called(lib, lib.tlq_gemm_w4a8(P(dA), P(dWp), P(C), M, N, K, mode, st))
        assert torch.equal(C.cpu(), (A.double() @ w.double().T).to(torch.int32)), mode


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 2, 4])
@pytest.mark.parametrize("M,N,K,waves", SHAPES)
@pytest.mark.parametrize("batch", [1, 3])
def test_weights_by_columns_in_batches(lib, rows, M, N, K, waves, batch):
    P, st = _abi.ptr, torch.cuda.current_stream().cuda_stream
    print(f"small [K, N] {rows} M={M} N={N} K={K} waves={waves} batch={batch}", flush=True)
    lib.tlq_tune_small(waves, 10 * rows + 4)
    A, W, sb = i8(11, batch, M, K), i8(12, batch, K, N), torch.rand(1, generator=gen(13))
    dA, dW, dsb = A.cuda(), W.cuda(), sb.cuda()
    acc = torch.bmm(A.double(), W.double()).to(torch.int32)
    C = torch.full((batch, M, N), -1, dtype=torch.int32, device="cuda")
    lib.tlq_debug_launch_log(1)
    called(lib, lib.tlq_gemm_i8(P(dA), P(dW), P(C), batch, M, N, K, _abi.B_KN, st))
    assert torch.equal(C.cpu(), acc)
    out = torch.full((batch, M, N), float("nan"), dtype=torch.float16, device="cuda")
    lib.tlq_debug_launch_log(1)
    called(lib, lib.tlq_gemm_w8a8_ws(P(dA), P(dW), None, P(dsb), P(out), None, 0, batch, M, N, K, 1, _abi.B_KN, _abi.F16, st))
    assert_bit_equal(out.cpu(), (acc.float() * sb).to(torch.float16), "one scale")
    for dt in (torch.float16, torch.bfloat16):
        X, B = torch.randn(batch, M, K, generator=gen(14)).to(dt), torch.randn(batch, K, N, generator=gen(15)).to(dt)
        D, dX, dB = torch.full((batch, M, N), float("nan"), dtype=dt, device="cuda"), X.cuda(), B.cuda()
        lib.tlq_debug_launch_log(1)
        called(lib, lib.tlq_gemm_f16_batched(P(dX), P(dB), P(D), batch, M, N, K, CODE[dt], CODE[dt], _abi.B_KN, st))
        check_float_output(D.cpu().reshape(batch * M, N), torch.bmm(X.float(), B.float()).reshape(batch * M, N), f"16-bit {dt}")


@pytest.mark.gpu
def test_estimates_take_it_where_it_is_ahead(lib):
    """The operators' own calls: small problems in one launch, large ones as before."""
    from tilelang_ascend_amd import ops

    def log_of(kernel, *args):
        lib.tlq_debug_launch_log(1)
        kernel(*args)
        text = lib.tlq_debug_launch_log_text().decode()
        lib.tlq_debug_launch_log(0)
        return text

    assert "gemm_small_kernel" in log_of(ops.int8_gemm_kernel_corrected(512, 3328), i8(1, 40, 3328).cuda(), i8(2, 512, 3328).cuda(), torch.rand(40).cuda(), torch.rand(512).cuda())
    assert "gemm_small_kernel" in log_of(ops.w4a8_gemm_cv(57, 1024, 3840), i8(1, 57, 3840).cuda(), torch.zeros(1024, 1920, dtype=torch.uint8).cuda(), i8(2, 1024, 3840).cuda())
    assert "gemm_small_kernel" in log_of(ops.batch_matmul(4, 34, 256, 5376, 1, 1, 1), torch.zeros(4, 34, 5376).half().cuda(), torch.zeros(4, 5376, 256).half().cuda())
    assert "gemm_small_kernel" not in log_of(ops.int8_gemm_kernel_corrected(4096, 4096), i8(1, 2048, 4096).cuda(), i8(2, 4096, 4096).cuda(), torch.rand(2048).cuda(), torch.rand(4096).cuda())


def test_plan_keeps_to_the_machine(lib):
    o = (ctypes.c_int64 * 4)()
    for kind in range(4):
        for M in (1, 17, 130, 3000):
            for N in (16, 1008, 14336):
                for row_bytes in (128, 11008, 28672):
                    assert lib.tlq_debug_small_tile(kind, 2, M, N, row_bytes, o) == 1
                    mt, rt, waves = o[0] // 16, o[1] // 16, o[2]
                    slot = mt * 2048 + (rt * 2048, 8192, 8192, rt * 1024)[kind]
                    assert mt in (1, 2, 4) and rt in ((1, 2, 4), (4,), (4,), (1, 2, 4))[kind] and 1 <= waves <= min(16, row_bytes // 128)
                    assert waves * slot * (4 if slot <= 4096 else 3 if slot <= 8192 else 2) <= 160 * 1024 and (rt * mt <= 4 or waves <= 8)
        assert lib.tlq_debug_small_tile(kind, 1, 1, 16, 192, o) == 0 and lib.tlq_debug_small_tile(kind, 1, 0, 16, 128, o) == 0


def test_no_register_spills(tmp_path):
    cmd = [build.hipcc_path(), *build.HIPCC_FLAGS, "-Rpass-analysis=kernel-resource-usage", "-c", f"{build.CSRC_DIR}/gemm_small.hip",
           "-o", str(tmp_path / "out.o")]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout[-2000:]
    blocks = [b for b in re.split(r"remark: Function Name: ", res.stdout)[1:] if "gemm_small_kernel" in b.split()[0]]
    assert len(blocks) == 39
    for b in blocks:
        assert re.search(r"ScratchSize \[bytes/lane\]: 0\b", b) and re.search(r"VGPRs Spill: 0\b", b), b[:300]


@pytest.mark.gpu
@pytest.mark.parametrize("what,B,M,N,K,small", [
    # where it measured ahead of what runs without it ...
    ("w4a8", 1, 57, 1024, 3840, True), ("w4a8", 1, 128, 4096, 11008, True), ("i8 NK", 1, 257, 1232, 8576, True), ("w8a8 NK", 1, 32, 4096, 14336, True),
    ("f16", 4, 34, 256, 5376, True),
    # ... and behind: K over groups of wavefronts, few rows in K slices, [K, N] weights of many columns
    ("i8 NK", 8, 1009, 160, 3456, False), ("w4a8", 1, 1374, 1184, 5376, False), ("f16", 3, 231, 1376, 8576, False), ("i8 KN", 1, 14, 704, 5760, False),
    ("w8a8 KN", 1, 89, 11440, 6528, False)])
def test_choice_against_the_larger_tiles(lib, what, B, M, N, K, small):
    """With the workspace that the entry points ask for, on a machine of 256 CUs."""
    P, st = _abi.ptr, torch.cuda.current_stream().cuda_stream
    print(f"choice {what} B={B} M={M} N={N} K={K}", flush=True)
    nk = what.endswith("NK")
    if what == "f16":
        A, W = torch.randn(B, M, K, generator=gen(1)).half().cuda(), torch.randn(B, K, N, generator=gen(2)).half().cuda()
    else:
        A, W = i8(1, B, M, K).cuda(), (torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, generator=gen(2)) if what == "w4a8" else i8(2, B, *((N, K) if nk else (K, N)))).cuda()
    C = torch.empty(B, M, N, dtype=torch.float16 if what == "f16" else torch.float32 if what.startswith("w8a8") else torch.int32, device="cuda")
    need = {"w8a8": lib.tlq_w8a8_workspace_bytes(B, M, N, K), "w4a8": N * K, "f16": lib.tlq_f16_workspace_bytes(B, M, N, K)}.get(what.split()[0], 0)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    layout = _abi.B_NK if nk else _abi.B_KN
    lib.tlq_debug_launch_log(1)
    if what == "w4a8":
        rc = lib.tlq_gemm_w4a8_ws(P(A), P(W), P(ws), need, P(C), M, N, K, _abi.U4, st)
    elif what == "f16":
        rc = lib.tlq_gemm_f16_ws(P(A), P(W), P(C), P(ws), need, B, M, N, K, _abi.F16, _abi.F16, layout, st)
    elif what.startswith("w8a8"):
        rc = lib.tlq_gemm_w8a8_ws(P(A), P(W), None, None, P(C), P(ws), need, B, M, N, K, 1, layout, _abi.F32, st)
    else:
        rc = lib.tlq_gemm_i8(P(A), P(W), P(C), B, M, N, K, layout, st)
    log = lib.tlq_debug_launch_log_text().decode()
    lib.tlq_debug_launch_log(0)
    _abi.check(rc)
    torch.cuda.synchronize()
    assert ("gemm_small_kernel" in log) == small or lib.tlq_device_cu_count() != 256, log
    if what == "w4a8":
        W = torch.stack([W & 15, W >> 4], -1).reshape(1, N, K)
    want = torch.bmm(A.double(), W.double().transpose(1, 2).contiguous() if nk or what == "w4a8" else W.double())
    if what == "f16":
        assert bool(((C.double() - want).abs() <= 2.0**-11 * want.abs() + K * 2.0**-24 * torch.bmm(A.double().abs(), W.double().abs()) * 1.001 + 2.0**-25).all())
    else:
        assert torch.equal(C.double(), want.float().double())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,unpacked", [(257, 512, 512, True), (300, 1040, 512, True), (600, 256, 1024, True), (256, 512, 512, False)])
def test_w4a8_above_256_rows_leaves_the_unpacked_weights_in_the_workspace(lib, M, N, K, unpacked):
    """What tlq.h says of a workspace that holds the int8 [N, K] matrix, also on problems that the small-tile kernel would win."""
    print(f"w4a8 workspace M={M} N={N} K={K}", flush=True)
    P, st = _abi.ptr, torch.cuda.current_stream().cuda_stream
    A, Wp = i8(1, M, K), torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, generator=gen(2))
    u = torch.stack([Wp & 15, Wp >> 4], -1).reshape(N, K).to(torch.int8)
    W = torch.where(u >= 8, u - 16, u)
    dA, dW, ws, C = A.cuda(), Wp.cuda(), torch.full((N, K), 99, dtype=torch.int8, device="cuda"), torch.full((M, N), -1, dtype=torch.int32, device="cuda")
    _abi.check(lib.tlq_gemm_w4a8_ws(P(dA), P(dW), P(ws), N * K, P(C), M, N, K, _abi.S4_TWOS, st))
    assert torch.equal(C.cpu(), (A.double() @ W.double().T).to(torch.int32))  # exact
    assert torch.equal(ws.cpu(), W) == unpacked
