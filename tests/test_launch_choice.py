"""What the library would launch, asked without a GPU: its calls of the HIP runtime go to tests/launch_recorder.c (256 compute units, every launch succeeds),
and its own launch log says which kernels ran.  In a process of its own, which never loads the runtime proper."""
import json
import os
import shutil
import subprocess
import sys

import pytest

from tilelang_ascend_amd import _abi

HERE = os.path.dirname(os.path.abspath(__file__))
PRELUDE = """
import ctypes, json, sys
rec = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
i64, i32, f32, p = ctypes.c_int64, ctypes.c_int, ctypes.c_float, ctypes.c_void_p
lib.tlq_debug_launch_log_text.restype = lib.tlq_last_error.restype = ctypes.c_char_p
lib.tlq_gemm_i8.argtypes = [p] * 3 + [i64] * 4 + [i32, p]
lib.tlq_gemm_w4a16_ws.argtypes = [p] * 5 + [i64] * 4 + [f32] + [i32] * 3 + [p, i64, p]
lib.tlq_w4a16_choice_set.argtypes = [i64] * 4 + [i32] * 2
A, W, C, S, WS = (i << 40 for i in range(1, 6))  # (addresses that nothing reads)
def log(call):
    lib.tlq_debug_launch_log(1)
    rc = call()
    text = lib.tlq_debug_launch_log_text().decode()
    lib.tlq_debug_launch_log(0)
    return [rc, text, lib.tlq_last_error().decode() if rc else ""]
def i8(B, M, N, K, layout):
    return log(lambda: lib.tlq_gemm_i8(A, W, C, B, M, N, K, layout, None))
"""


@pytest.fixture(scope="module")
def recorder(tmp_path_factory):
    if not shutil.which("gcc"):
        pytest.skip("a C compiler wanted")
    out = str(tmp_path_factory.mktemp("recorder") / "launch_recorder.so")
    subprocess.run(["gcc", "-O1", "-Wall", "-Wextra", "-shared", "-fPIC", os.path.join(HERE, "launch_recorder.c"), "-o", out], check=True)
    return out


def ask(recorder, code):
    """`code` behind the prelude in a process of its own; what it leaves in `result`."""
    done = subprocess.run([sys.executable, "-c", PRELUDE + code + "\nprint(json.dumps(result))", recorder, _abi.library_path()], capture_output=True, text=True, timeout=120)
    assert done.returncode == 0, done.stderr
    return json.loads(done.stdout)


# 128-row tiles are the two-stage or the ring kernel's, 256-row ones those of four wavefronts or of the two-stage kernel
@pytest.mark.parametrize("B,M,N,K", [(8, 2048, 4096, 4096), (8, 3072, 4096, 4096), (1, 513, 1040, 1024), (1, 100, 272, 400)])
@pytest.mark.parametrize("layout", [_abi.B_KN, _abi.B_NK])
def test_a_forced_int8_tile_holds_and_ends(recorder, B, M, N, K, layout):
    """Forced tiles and the automatic choice in turn on one shape, on one thread: each call by the tile that is set for it, and by none that was."""
    def each(tiles):
        return ask(recorder, f"""
result = []
for tile in {tiles}:
    lib.tlq_tune_i8_tile(tile)
    result.append(i8({B}, {M}, {N}, {K}, {layout}))
""")
    fresh = {tile: each([tile])[0] for tile in (0, 32, 128, 256)}
    assert all(rc == 0 for rc, _, _ in fresh.values()), fresh
    assert "256x256" in fresh[256][1] and "256" not in fresh[128][1] and "32x128" in fresh[32][1], fresh
    order = [0, 128, 256, 0, 256, 128, 0, 32, 0]
    assert each(order) == [fresh[tile] for tile in order]


@pytest.mark.parametrize("M,N,K", [(8202, 960, 3200), (1182, 6944, 6656), (6715, 1168, 3072)])
def test_forced_int8_slices_end_too(recorder, M, N, K):
    """Rows of full rounds and the rest: the rest is not asked of the small-tile kernel while K slices are forced, and is again afterwards."""
    one = f"i8(1, {M}, {N}, {K}, {_abi.B_NK})"
    auto, never = (ask(recorder, f"lib.tlq_tune_i8_split({split}); result = {one}") for split in (0, 1))
    assert auto != never  # (else the shape says nothing)
    assert ask(recorder, f"""
result = []
for split in (0, 1, 0, 1):
    lib.tlq_tune_i8_split(split)
    result.append({one})
""") == [auto, never, auto, never]


W4A16 = """
def w4a16(M, N, K, group, ws=0):
    return log(lambda: lib.tlq_gemm_w4a16_ws(A, W, S, None, C, M, N, K, group, 8.0, 1, 1, 0, WS if ws else None, ws, None))
"""


@pytest.mark.parametrize("M,N,K,group", [(1635, 272, 3584, 128), (1295, 560, 2816, 64), (2442, 224, 2944, 128), (1759, 496, 3072, 64)])
def test_last_rows_behind_a_tuned_kernel_that_gets_no_lds(recorder, M, N, K, group):
    """bfloat16 rows that would go along with the tuned 256-row kernel: where its launch fails, the rules decide for the head, and the last one to three rows are theirs too."""
    call = f"w4a16({M}, {N}, {K}, {group})"
    rules = ask(recorder, W4A16 + f"result = {call}")
    tuned = W4A16 + f"lib.tlq_w4a16_choice_set({M & ~3}, {N}, {K}, {group}, {_abi.BF16}, {_abi.ALGO_PANEL256})\n"
    assert rules[0] == 0 and " + " in rules[1], rules  # (the head and the rest, by different kernels)
    assert ask(recorder, tuned + f"result = {call}") == [0, "tlq_gemm_w4a16(panel256) [w4a16_panel256_kernel]", ""]
    assert ask(recorder, tuned + f"rec.recorder_refuse(b'panel256')\nresult = {call}") == rules


# The least workspaces with which the streaming kernel took these problems while every window of its scale area held 16 groups: the plans that the
# longer windows choose cut K into more slices, which do not fit.
@pytest.mark.parametrize("M,N,K,group,workspace", [(413, 664, 12672, 32, 10969280), (472, 3040, 4224, 64, 11479040), (499, 3488, 4224, 32, 13924096),
                                                   (464, 4912, 18944, 32, 27350016), (265, 4544, 4352, 32, 12087872)])
def test_streaming_kernel_in_the_workspaces_that_held_its_slices(recorder, M, N, K, group, workspace):
    def call(ws, layout, algo):
        return ask(recorder, f"""
lib.tlq_gemm_w4a16_layout_ws.argtypes = [p] * 5 + [i64] * 4 + [f32] + [i32] * 4 + [p, i64, p]
result = log(lambda: lib.tlq_gemm_w4a16_layout_ws(A, W, S, None, C, {M}, {N}, {K}, {group}, 8.0, 0, 0, {algo}, {layout}, WS, {ws}, None))
""")
    for layout in (_abi.W_PLAIN, _abi.W_INTERLEAVED_F16):
        for algo in (_abi.ALGO_AUTO, _abi.ALGO_STREAM):
            rc, text, error = call(workspace, layout, algo)
            assert rc == 0 and "w4a16_stream_kernel" in text, (layout, algo, text, error)
        rc, _, error = call(1 << 16, layout, _abi.ALGO_STREAM)  # (no plan's slices: refused, as ever)
        assert rc == 1 and "workspace" in error, error


# One group per row, written out per 128 values: the room for that is in the built-in scratch array where it holds the least workspace that the shape can use, and
# that size follows the plan with the fewer slices (51.8 MiB for the first, 69.0 by the other plan), and of two the one that cuts at all.
@pytest.mark.parametrize("M,N,K,most", [(376, 12032, 18816, 54288384), (458, 10192, 11648, 56015232), (407, 9376, 9344, 45792384)])
def test_least_workspace_counts_the_plan_with_the_fewer_slices(recorder, M, N, K, most):
    assert 0 < _abi.load().tlq_w4a16_workspace_bytes_min(M, N, K) <= most
    rc, text, error = ask(recorder, f"""
lib.tlq_gemm_w4a16_noalloc.argtypes = [p] * 5 + [i64] * 4 + [f32] + [i32] * 3 + [p]
result = log(lambda: lib.tlq_gemm_w4a16_noalloc(A, W, S, WS, C, {M}, {N}, {K}, {K}, 8.0, 1, 1, 0, None))
""")
    assert rc == 0 and "w4a16_stream_kernel" in text, (text, error)


# (bfloat16, groups of 64; a workspace too small for the dequantised weights, and none)
@pytest.mark.parametrize("M,N,K", [(2308, 1328, 4224), (2174, 1152, 3840), (2528, 2688, 4608), (4020, 576, 3584), (1059, 2416, 4736), (926, 1888, 3328), (565, 1040, 640)])
def test_calls_without_room_for_the_two_passes_are_not_decided_by_them(recorder, M, N, K):
    """What runs above 512 rows without the room that the two passes take does not follow the estimate of their plain GEMM, here made very low
    (tlq_tune_gemm_quad) and high (its oldest kernel alone)."""
    for ws in (0, N * K):
        auto, fast, slow = (ask(recorder, W4A16 + f"{tune}; result = w4a16({M}, {N}, {K}, 64, {ws})")
                            for tune in ("pass", "lib.tlq_tune_gemm_quad(11)", "lib.tlq_tune_gemm_groups(1); lib.tlq_tune_gemm_slots(0)"))
        assert auto[0] == 0 and "dequant" not in auto[1], auto
        assert auto == fast == slow


# 16-bit [N, K] products that have a cut, with a workspace for it: measured 47 / 73, 35 / 53, 39 / 58, 42 / 58 us in slices / in one launch; 13.8 / 10.0, 13.0 / 9.7, 14.0 / 10.4, 11.8 / 8.8
@pytest.mark.parametrize("M,N,K,slices", [(496, 2496, 11520, True), (1140, 768, 12224, True), (422, 2816, 8896, True), (368, 4096, 8896, True),
                                          (1111, 240, 2496, False), (2862, 64, 2368, False), (517, 528, 2624, False), (1526, 96, 2048, False)])
def test_one_launch_or_slices_of_k(recorder, M, N, K, slices):
    rc, text, error = ask(recorder, f"""
lib.tlq_gemm_f16_ws.argtypes = [p] * 4 + [i64] * 5 + [i32] * 3 + [p]
result = log(lambda: lib.tlq_gemm_f16_ws(A, W, C, WS, 1 << 32, 1, {M}, {N}, {K}, 0, 0, {_abi.B_NK}, None))
""")
    assert rc == 0 and ("K slices" in text) == slices, (text, error)


# The small-tile kernel against the tiles, measured: narrow results and long rows 15.6 / 24.3, 19.2 / 29.8, 22.5 / 34.7, 5.6 / 12.1, 6.0 / 8.7 us; two stages of K 8.3 / 5.8, 8.1 / 5.7
@pytest.mark.parametrize("kind,B,M,N,K,layout,small", [("w8a8", 9, 269, 64, 9344, _abi.B_KN, True), ("i8", 8, 464, 64, 11520, _abi.B_KN, True), ("f16", 4, 52, 512, 6080, _abi.B_KN, True),
                                                       ("w8a8", 5, 399, 16, 7424, _abi.B_NK, True), ("f16", 1, 3791, 64, 1856, _abi.B_KN, True),
                                                       ("w8a8", 1, 227, 3760, 256, _abi.B_KN, False), ("w8a8", 1, 99, 7264, 256, _abi.B_NK, False)])
def test_small_tiles_or_tiles(recorder, kind, B, M, N, K, layout, small):
    call = {"i8": f"lib.tlq_gemm_i8(A, W, C, {B}, {M}, {N}, {K}, {layout}, None)", "f16": f"lib.tlq_gemm_f16_batched(A, W, C, {B}, {M}, {N}, {K}, 0, 0, {layout}, None)",
            "w8a8": f"lib.tlq_gemm_w8a8(A, W, S, S, C, {B}, {M}, {N}, {K}, {N}, {layout}, 0, None)"}[kind]
    rc, text, error = ask(recorder, f"""
lib.tlq_gemm_f16_batched.argtypes = [p] * 3 + [i64] * 4 + [i32] * 3 + [p]
lib.tlq_gemm_w8a8.argtypes = [p] * 5 + [i64] * 5 + [i32] * 2 + [p]
result = log(lambda: {call})
""")
    assert rc == 0 and ("gemm_small_kernel" in text) == small, (text, error)


# an odd number of tile rows of 64, 128 x 64 against 64 x 128 tiles: 22.1 / 28.1, 26.8 / 33.5, 50.7 / 63.2, 28.6 / 34.8, 13.9 / 17.2 us
@pytest.mark.parametrize("kind,B,M,N,K", [("i8", 1, 416, 3456, 5040), ("i8", 1, 436, 2656, 9216), ("i8", 1, 694, 2624, 11440), ("w8a8", 1, 287, 4128, 7232), ("w8a8", 5, 140, 1536, 2704)])
def test_ring_tiles_that_leave_fewer_units_idle(recorder, kind, B, M, N, K):
    call = {"i8": f"lib.tlq_gemm_i8(A, W, C, {B}, {M}, {N}, {K}, {_abi.B_NK}, None)", "w8a8": f"lib.tlq_gemm_w8a8(A, W, S, S, C, {B}, {M}, {N}, {K}, {N}, {_abi.B_NK}, 0, None)"}[kind]
    rc, text, error = ask(recorder, f"""
lib.tlq_gemm_w8a8.argtypes = [p] * 5 + [i64] * 5 + [i32] * 2 + [p]
result = log(lambda: {call})
""")
    assert rc == 0 and "ring_gemm_mfma_kernel 128x64" in text, (text, error)


# 16-bit products of one and a half rounds of the ring kernel's tiles, two-stage kernel / ring kernel: 109 / 154, 146 / 189, 194 / 269 us
@pytest.mark.parametrize("B,M,N,K", [(1, 2797, 2192, 6896), (1, 2464, 1728, 9456), (8, 564, 1600, 8224)])
def test_two_stages_or_more_than_one_round_of_the_ring(recorder, B, M, N, K):
    rc, text, error = ask(recorder, f"""
lib.tlq_gemm_f16_batched.argtypes = [p] * 3 + [i64] * 4 + [i32] * 3 + [p]
result = log(lambda: lib.tlq_gemm_f16_batched(A, W, C, {B}, {M}, {N}, {K}, 0, 0, {_abi.B_NK}, None))
""")
    assert rc == 0 and "[gemm_mfma_kernel" in text, (text, error)


# A full workspace: the kernel named against the two passes, measured 12.9 / 19.9, 11.1 / 16.0, 9.1 / 12.9, 13.7 / 18.6, 12.6 / 17.2, 21.0 / 30.7, 101.7 / 104.3, 204 / 229 us
@pytest.mark.parametrize("M,N,K,group,kernel", [(564, 3328, 1280, 128, "w4a16_stream"), (872, 512, 2688, 128, "w4a16_small"), (875, 320, 2048, 256, "w4a16_small"),
                                                (864, 512, 3328, 64, "w4a16_small"), (1086, 5376, 384, 128, "w4a16_stream"), (2872, 384, 3328, 64, "w4a16_stream"),
                                                (4096, 4096, 4096, 128, "w4a16_panel256"), (2816, 10752, 4096, 128, "w4a16_panel256")])
def test_two_passes_or_one_kernel(recorder, M, N, K, group, kernel):
    rc, text, error = ask(recorder, W4A16 + f"result = w4a16({M}, {N}, {K}, {group}, 1 << 32)")
    assert rc == 0 and kernel in text and "dequant" not in text, (text, error)


# (bfloat16, groups, the workspace asked for; the sizes at which the GPU test of these rows compares results)
@pytest.mark.parametrize("M,N,K,group,kernels", [(1002, 8960, 1152, 64, ["w4a16_panel256"]), (1023, 8960, 1152, 64, ["w4a16_panel256"]), (2209, 14224, 1536, 128, ["w4a16_panel256"]),
                                                 (601, 11008, 4096, 128, ["w4a16_panelm"]), (639, 11008, 4096, 128, ["w4a16_panelm"]),
                                                 (641, 11008, 4096, 128, ["w4a16_panelm", "gemv"]), (839, 6144, 2048, 64, ["w4a16_stream"]), (641, 7936, 4224, 128, ["w4a16_stream"]),
                                                 (590, 1664, 5120, 128, ["w4a16_stream", "reduce"]), (1207, 1024, 6144, 64, ["w4a16_stream", "reduce"])])
def test_which_kernel_takes_the_last_rows(recorder, M, N, K, group, kernels):
    """The last one to three rows lie in a tile of the kernel that takes the others, each kernel without and with K slices, or have a launch of their own."""
    ws = _abi.load().tlq_w4a16_workspace_bytes(M, N, K)
    rc, text, error = ask(recorder, W4A16 + f"result = w4a16({M}, {N}, {K}, {group}, {ws})")
    launches = text.split(" + ")
    assert rc == 0 and len(launches) == len(kernels) and all(k in l for k, l in zip(kernels, launches)), (text, error)
