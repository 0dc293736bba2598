"""The 256-row panel kernel fills the register file: its 256 accumulators have to be moved one by one where the output is written, or the compiler moves them
ahead and spills.  One register at most (an address, ahead of the main loop), read from the object that the build left."""
import os
import re
import subprocess

import pytest

from tilelang_ascend_amd import build

LLVM = "/opt/rocm/llvm/bin"


def test_the_panel_kernel_keeps_its_accumulators(tmp_path):
    obj = os.path.join(build.OBJ_DIR, "gemm_w4a16_panel256.o")
    if not (os.path.exists(obj) and os.path.exists(f"{LLVM}/clang-offload-bundler")):
        pytest.skip("objects of a build and ROCm's LLVM tools wanted")
    bundle, code = tmp_path / "bundle", tmp_path / "code"
    subprocess.run([f"{LLVM}/llvm-objcopy", "--dump-section", f".hip_fatbin={bundle}", obj, str(tmp_path / "copy.o")], check=True)
    subprocess.run([f"{LLVM}/clang-offload-bundler", "--unbundle", "--type=o", f"--input={bundle}", f"--targets=hipv4-amdgcn-amd-amdhsa--{build.ARCH}",
                    f"--output={code}"], check=True)
    notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", str(code)], capture_output=True, text=True, check=True).stdout
    kernels = [k for k in re.split(r"\n  - \.a(?:gpr_count|rgs)", notes)[1:] if "w4a16_panel256_kernel" in k]
    assert len(kernels) == 12
    assert [int(re.search(r"\.vgpr_spill_count: +(\d+)", k)[1]) <= 1 for k in kernels] == [True] * 12
