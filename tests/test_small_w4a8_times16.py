"""The small-tile kernel multiplies two's complement and offset-8 int4 weights as 16 times their value while 16 x 8 x 128 K fits 31
bits: exact at the largest sums that allows, on either side of that length, with one wavefront and with several."""
import ctypes
import re
import subprocess

import pytest
import torch

from helpers import assert_bit_equal, gen
from tilelang_ascend_amd import _abi, build


@pytest.mark.gpu
@pytest.mark.parametrize("mode,low", [(_abi.S4_TWOS, 0x88), (_abi.S4_OFFSET8, 0x00)])
@pytest.mark.parametrize("M,N,K,waves,tiles", [(1, 16, 130944, 16, 11), (17, 36, 130944, 1, 22), (33, 64, 131072, 8, 44), (64, 80, 384, 2, 42)])
def test_largest_sums(mode, low, M, N, K, waves, tiles):
    g = gen(M + K)
    A = torch.randint(-128, 128, (M, K), dtype=torch.int8, generator=g)
    A[0] = -128
    Wp = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, generator=g)
    Wp[:2] = low  # every weight of the first rows is -8
    u = torch.stack([Wp & 15, Wp >> 4], dim=-1).reshape(N, K).to(torch.float64)
    w = u - 8 if mode == _abi.S4_OFFSET8 else torch.where(u >= 8, u - 16, u)
    want = (A.double() @ w.T.contiguous()).to(torch.int32)  # (sums of at most 2^27: exact)
    assert want[0, 0] == 1024 * K
    lib, st = _abi.load(), torch.cuda.current_stream().cuda_stream
    Ad, Wd, C = A.cuda(), Wp.cuda(), torch.full((M, N), 7, dtype=torch.int32, device="cuda")
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    lib.tlq_tune_small(waves, tiles)
    try:
        _abi.check(lib.tlq_gemm_w4a8(P(Ad), P(Wd), P(C), M, N, K, mode, st))
    finally:
        lib.tlq_tune_small(0, 0)
    torch.cuda.synchronize()
    assert_bit_equal(C.cpu(), want, f"W4A8 mode {mode} {M}x{N}x{K}")


def test_no_register_spills(tmp_path):
    cmd = [build.hipcc_path(), *build.HIPCC_FLAGS, "-Rpass-analysis=kernel-resource-usage", "-c", f"{build.CSRC_DIR}/gemm_small_w4a8.hip",
           "-o", str(tmp_path / "out.o")]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout[-2000:]
    blocks = [b for b in re.split(r"remark: Function Name: ", res.stdout)[1:] if "gemm_small_kernel" in b.split()[0]]
    assert len(blocks) == 9
    for b in blocks:
        assert re.search(r"ScratchSize \[bytes/lane\]: 0\b", b) and re.search(r"VGPRs Spill: 0\b", b), b[:300]
