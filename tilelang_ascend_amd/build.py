"""Builds libtlq.so (HIP kernels + C ABI) for gfx950 with hipcc and tlq_host.so (the extension module that calls it), in-tree.

    python -m tilelang_ascend_amd.build [--force]

Mirrors the role of the reference's LibraryGenerator.compile_lib
(tilelang/jit/adapter/libgen.py:106-232: write source, shell out to the device compiler,
produce a .so that ctypes loads), except that the kernels are fixed sources rather than
generated ones, so there is one library for all operators (and one extension module in the place of the reference's Cython
wrapper, tilelang/jit/adapter/cython/cython_wrapper.pyx).
"""
from __future__ import annotations

import contextlib
import fcntl
import hashlib
import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
REPO_DIR = os.path.dirname(PKG_DIR)
CSRC_DIR = os.path.join(PKG_DIR, "csrc")
INCLUDE_DIR = os.path.join(REPO_DIR, "include")
LIB_DIR = os.path.join(PKG_DIR, "lib")
OBJ_DIR = os.path.join(LIB_DIR, "obj")
LIB_PATH = os.path.join(LIB_DIR, "libtlq.so")
HOST_PATH = os.path.join(LIB_DIR, "tlq_host.so")
STAMP_PATH = os.path.join(LIB_DIR, "libtlq.fingerprint")
HOST_STAMP_PATH = os.path.join(LIB_DIR, "tlq_host.fingerprint")

ARCH = "gfx950"
SOURCES = [
    "abi.hip",
    "unpack_dequant.hip",
    "decode_i4.hip",
    "decode_lowbit.hip",
    "act_quant.hip",
    "repack.hip",
    "gemv_plain.hip",
    "gemv_w4a16.hip",
    "gemm_w4a16.hip",
    "gemm_w4a16_small.hip",
    "gemm_w4a16_stream.hip",
    "gemm_w4a16_panel.hip",
    "gemm_w4a16_panel256.hip",
    "gemm_w4a16_panelm.hip",
    "w4a16_choice.hip",
    "gemm_w4a16_decode.hip",
    "gemm_int8.hip",
    "gemm_small.hip",
    "gemm_small_w4a8.hip",
    "gemm_f16.hip",
    "gemm_quad_f16.hip",
    "gemm_quad_i8.hip",
    "gemm_api.hip",
    "gemm_addr_check.hip",
    "gemm_w4a16_noalloc.hip",
]
# packed-fp32 VALU forms are disabled on purpose (some have produced silent wrong results on
# this hardware pool); hipcc's host pass warns that it does not know the feature.
HIPCC_FLAGS = [
    "-O3",
    "-std=c++17",
    "-fPIC",
    f"--offload-arch={ARCH}",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-ffp-contract=off",
    "-Wno-unused-command-line-argument",
    "-Wno-unknown-warning-option",
    f"-I{INCLUDE_DIR}",
    f"-I{CSRC_DIR}",
]


# the extension module through which Python makes the calls (csrc/host_calls.cpp): host code against torch's C++ headers
HOST_SOURCE = "host_calls.cpp"
HOST_FLAGS = ["-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f"-I{INCLUDE_DIR}"]


def hipcc_path() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found: cannot build libtlq.so")


def _fingerprint(flags, paths) -> str:
    """sha256 over flags and file contents.  Include folders are left out: they say where the checkout lies, not what is built
    (a checkout that is moved, or reached through another path, keeps its libraries)."""
    h = hashlib.sha256()
    h.update(" ".join(f for f in flags if not f.startswith("-I")).encode())
    for path in paths:
        if os.path.isfile(path):
            h.update(os.path.basename(path).encode())
            with open(path, "rb") as f:
                h.update(f.read())
    return h.hexdigest()


def source_fingerprint() -> str:
    """sha256 over kernel sources, headers and flags -- the analogue of the reference's kernel
    cache key (tilelang/cache/kernel_cache.py:71-117: hash of source + target + options)."""
    names = [n for n in sorted(os.listdir(CSRC_DIR)) if n != HOST_SOURCE]
    return _fingerprint(HIPCC_FLAGS, [os.path.join(CSRC_DIR, n) for n in names] + [os.path.join(INCLUDE_DIR, n) for n in ("tlq.h", "tlq_debug.h")])


def host_fingerprint() -> str:
    """The same for the extension module, which also belongs to one interpreter and one torch."""
    import sysconfig

    import torch

    flags = HOST_FLAGS + [str(sysconfig.get_config_var("SOABI")), torch.__version__]
    return _fingerprint(flags, [os.path.join(CSRC_DIR, HOST_SOURCE), os.path.join(INCLUDE_DIR, "tlq.h")])


def _compile_one(src: str, verbose: bool) -> str:
    obj = os.path.join(OBJ_DIR, os.path.splitext(src)[0] + ".o")
    cmd = [hipcc_path(), *HIPCC_FLAGS, "-c", os.path.join(CSRC_DIR, src), "-o", obj]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"Compilation Failed! {' '.join(cmd)}\n{res.stdout}")
    noise = ("packed-fp32-ops", "is not a recognized feature")
    out = "\n".join(l for l in res.stdout.splitlines() if not any(n in l for n in noise))
    if verbose and out.strip():
        print(out)
    return obj


def _compile_host() -> str:
    """tlq_host.so for the running interpreter and torch."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    tmp = HOST_PATH + ".tmp"
    rocm = os.path.dirname(os.path.dirname(hipcc_path()))
    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    includes = [*cpp_extension.include_paths(), os.path.join(rocm, "include"), sysconfig.get_paths()["include"]]
    compiler = shutil.which("g++") or os.path.join(rocm, "bin", "amdclang++")
    cmd = [compiler, *HOST_FLAGS, f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *(f"-isystem{p}" for p in includes), os.path.join(CSRC_DIR, HOST_SOURCE), "-o", tmp, f"-L{torch_lib}",
           "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch", "-ltorch_python"]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"Compilation Failed! {' '.join(cmd)}\n{res.stdout}")
    return tmp


def _record(path: str):
    try:
        with open(path) as f:
            return f.read().strip() or None
    except OSError:
        return None


def built_fingerprint():
    """Fingerprint the library on disk was built from (None when there is no record)."""
    return _record(STAMP_PATH)


def is_current() -> bool:
    return os.path.exists(LIB_PATH) and built_fingerprint() == source_fingerprint()


def is_stale() -> bool:
    """True when the library is absent, or carries a build record that names other sources than those on disk.
    A library without a record (copied on its own) cannot be judged and is taken as it is."""
    if not os.path.exists(LIB_PATH):
        return True
    fp = built_fingerprint()
    return fp is not None and fp != source_fingerprint()


def is_host_stale() -> bool:
    """The same for the extension module: absent, or built from other sources, for another interpreter or another torch."""
    if not os.path.exists(HOST_PATH):
        return True
    fp = _record(HOST_STAMP_PATH)
    return fp is not None and fp != host_fingerprint()


@contextlib.contextmanager
def build_lock():
    """Exclusive advisory lock on lib/.build.lock: two processes (pytest workers, a test run next to a benchmark)
    never compile into the same object directory or replace the library under each other.  The reference
    serialises its kernel cache the same way (tilelang/cache/kernel_cache.py:119-160, a lock around save / load)."""
    os.makedirs(LIB_DIR, exist_ok=True)
    with open(os.path.join(LIB_DIR, ".build.lock"), "w") as f:
        fcntl.flock(f, fcntl.LOCK_EX)
        try:
            yield
        finally:
            fcntl.flock(f, fcntl.LOCK_UN)


def build_library(force: bool = True, verbose: bool = False, jobs: int = 6, host: bool = True) -> str:
    """Compile every kernel source for gfx950 and link libtlq.so, then (host=True) the extension module that calls it.  With
    force=False what is up to date (matching record) is reused.  libtlq.so needs hipcc alone and is in place before the
    extension module, which needs torch's headers as well, is awaited.  Holds the build lock throughout; a process that waited
    for another one's build finds the library current and (force=False) returns at once."""
    with build_lock(), ThreadPoolExecutor(max_workers=1) as side:
        module = side.submit(_compile_host) if host and (force or is_host_stale()) else None
        if force or not is_current():
            _build_locked(verbose, jobs)
        if module is not None:
            _install(module.result(), HOST_PATH, HOST_STAMP_PATH, host_fingerprint())
    return LIB_PATH


def build_host() -> str:
    """The extension module alone, where it is absent or belongs to other sources, another interpreter or another torch."""
    with build_lock():
        if is_host_stale():
            _install(_compile_host(), HOST_PATH, HOST_STAMP_PATH, host_fingerprint())
    return HOST_PATH


def _install(tmp: str, path: str, stamp: str, fingerprint: str) -> None:
    os.replace(tmp, path)
    with open(stamp, "w") as f:
        f.write(fingerprint + "\n")


def _build_locked(verbose: bool, jobs: int) -> None:
    os.makedirs(OBJ_DIR, exist_ok=True)
    fp = source_fingerprint()
    srcs = [s for s in SOURCES if os.path.exists(os.path.join(CSRC_DIR, s))]
    missing = sorted(set(SOURCES) - set(srcs))
    if missing:
        raise RuntimeError(f"kernel sources missing: {missing}")
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        objs = list(pool.map(lambda s: _compile_one(s, verbose), srcs))
    tmp = LIB_PATH + ".tmp"
    cmd = [hipcc_path(), "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", tmp, *objs]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"Compilation Failed! {' '.join(cmd)}\n{res.stdout}")
    _install(tmp, LIB_PATH, STAMP_PATH, fp)


if __name__ == "__main__":
    path = build_library(force="--force" in sys.argv or True, verbose=True)
    print("built", path)
