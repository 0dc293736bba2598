"""What a launch hands to the GPU: kernels take at most 112 bytes of arguments and none of the hidden ones that gridDim and blockDim bring
(256 bytes), because the host writes them on every call (csrc/tlq_common.h says what either costs).  Reads the metadata of the objects that
the library was linked from; no GPU needed."""
import os
import re
import subprocess

import pytest

from tilelang_ascend_amd import build

LLVM = "/opt/rocm/llvm/bin"
SOURCES = [s for s in build.SOURCES if not s.startswith(("gemm_addr_check", "abi"))]


@pytest.mark.parametrize("source", SOURCES)
def test_kernel_arguments(tmp_path, source):
    obj = os.path.join(build.OBJ_DIR, os.path.splitext(source)[0] + ".o")
    if not (os.path.exists(obj) and os.path.exists(f"{LLVM}/clang-offload-bundler")):
        pytest.skip("objects of a build and ROCm's LLVM tools wanted")
    bundle, code = tmp_path / "bundle", tmp_path / "code"
    if subprocess.run([f"{LLVM}/llvm-objcopy", "--dump-section", f".hip_fatbin={bundle}", obj, str(tmp_path / "copy.o")], capture_output=True).returncode:
        pytest.skip("no device code in this source")
    subprocess.run([f"{LLVM}/clang-offload-bundler", "--unbundle", "--type=o", f"--input={bundle}", f"--targets=hipv4-amdgcn-amd-amdhsa--{build.ARCH}",
                    f"--output={code}"], check=True)
    notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", str(code)], capture_output=True, text=True, check=True).stdout
    sizes = [int(s) for s in re.findall(r"\.kernarg_segment_size: (\d+)", notes)]
    assert not sizes or max(sizes) <= 112, f"{max(sizes)} bytes of arguments"
    assert "hidden_" not in notes, "a kernel uses gridDim or blockDim"


@pytest.mark.parametrize("source,kernel", [("gemv_w4a16", "gemv_w4a16_ring_kernel"), ("gemm_w4a16_decode", "w4a16_decode_kernel")])
def test_no_division_by_an_argument(tmp_path, source, kernel):
    """The decode kernels' work-groups take a few us in all and ask for their weights behind a handful of scalar instructions: what a division by one of
    their arguments gives -- thirty dependent instructions around a reciprocal -- comes from the host."""
    obj = os.path.join(build.OBJ_DIR, source + ".o")
    if not (os.path.exists(obj) and os.path.exists(f"{LLVM}/clang-offload-bundler")):
        pytest.skip("objects of a build and ROCm's LLVM tools wanted")
    bundle, code = tmp_path / "bundle", tmp_path / "code"
    subprocess.run([f"{LLVM}/llvm-objcopy", "--dump-section", f".hip_fatbin={bundle}", obj, str(tmp_path / "copy.o")], check=True)
    subprocess.run([f"{LLVM}/clang-offload-bundler", "--unbundle", "--type=o", f"--input={bundle}", f"--targets=hipv4-amdgcn-amd-amdhsa--{build.ARCH}",
                    f"--output={code}"], check=True)
    listing = subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn", str(code)], capture_output=True, text=True, check=True).stdout
    bodies = [k for k in re.split(r"\n[0-9a-f]{16} (?=<)", listing) if kernel in k.split("\n", 1)[0]]
    assert len(bodies) >= 4 and not [k.split("\n", 1)[0] for k in bodies if "v_rcp" in k]
