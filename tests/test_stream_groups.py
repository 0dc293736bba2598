"""The streaming W4A16 kernel with two and four groups of wavefronts over K, on every height of its activation tile, against the oracle: ragged
rows and columns, slices of one step and of several windows, each way its scales reach LDS (16-byte pieces, dwords from rows that start
on either half of one, 2-byte gathers), both word layouts; bit for bit on one-hot activations; and the automatic choice above 512 rows."""
import pytest
import torch

from helpers import DT, assert_bit_equal, check_float_output, gen, make_w4, w4a16_reference
from oracle import ref
from tilelang_ascend_amd import _abi

pytestmark = pytest.mark.gpu


def run(A, Wp, s, z, group, tiles, slice_steps, layout=0, out_dtype=None, shift=0, algo=None, exact=False):
    lib, P = _abi.load(), _abi.ptr
    M, K = A.shape
    N = Wp.shape[0]
    code = {torch.float16: _abi.F16, torch.bfloat16: _abi.BF16, torch.float32: _abi.F32}
    out_dtype = out_dtype or A.dtype
    zt = z if torch.is_tensor(z) else None

    def device(t):  # `shift` values into an allocation of its own
        if t is None:
            return None
        d = torch.empty(t.numel() + 8, dtype=t.dtype, device="cuda")
        d[shift : shift + t.numel()] = t.reshape(-1).cuda()
        return d[shift:]

    dA, dW, dS, dZ = A.cuda(), Wp.cuda(), device(s), device(zt)
    C = torch.full((M, N), float("nan"), dtype=out_dtype, device="cuda")
    print(f"stream groups M={M} N={N} K={K} g={group} {A.dtype} tiles={tiles} slice={slice_steps} layout={layout} shift={shift}", flush=True)
    lib.tlq_tune_w4a16_stream_tiles(tiles)
    lib.tlq_tune_w4a16_stream_slice(slice_steps)
    try:
        need = int(lib.tlq_w4a16_workspace_bytes(M, N, K))
        if not exact:  # (forced slices may be more than any plan's)
            need = max(need, 16 * M * N * 4)
        ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
        lib.tlq_debug_launch_log(1)
        rc = lib.tlq_gemm_w4a16_layout_ws(P(dA), P(dW), P(dS), P(dZ), P(C), M, N, K, group, 0.0 if zt is not None or z is None else float(z), code[A.dtype], code[out_dtype],
                                          _abi.ALGO_STREAM if algo is None else algo, layout, P(ws), need, torch.cuda.current_stream().cuda_stream)
        run.log = lib.tlq_debug_launch_log_text().decode()
        lib.tlq_debug_launch_log(0)
    finally:
        lib.tlq_tune_w4a16_stream_tiles(0)
        lib.tlq_tune_w4a16_stream_slice(0)
    _abi.check(rc)
    torch.cuda.synchronize()
    return C.cpu()


@pytest.mark.parametrize("in_dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("groups", [0, 16])
@pytest.mark.parametrize("tiles", [2, 4, 6, 8])
@pytest.mark.parametrize("M,N,K,group,slice_steps,zeros_kind,shift", [
    (33, 132, 128, 128, 1, "int", 0),             # one step
    (130, 260, 128 * 5, 64, 3, "frac", 0),        # 10 groups a row (dwords), slices that start on an odd group of pieces
    (97, 384, 128 * 7, 128, 4, "int", 0),         # odd groups: every other row starts on the second half of a dword
    (65, 516, 128 * 8, 64, 8, "int", 2),          # 16 groups, 4-byte aligned tensors
    (65, 260, 128 * 5, 64, 5, "int", 1),          # 2-byte aligned tensors: gathers
    (70, 256, 128 * 40, 64, 40, "mixed", 0),      # windows of 8 and 16 steps
    (129, 300, 128 * 35, 128, 35, "scalar8", 0),  # windows of rows of 35 groups
    (64, 128, 128 * 32, 4096, 8, "int", 0),       # slices inside one group
])
def test_against_the_oracle(in_dtype, groups, tiles, M, N, K, group, slice_steps, zeros_kind, shift):
    dt = DT[in_dtype]
    A = torch.randn(M, K, generator=gen(60)).to(dt)
    Wp, s, z = make_w4(N, K, group, dt, "int" if zeros_kind == "mixed" else zeros_kind, seed=61)
    if zeros_kind == "mixed":
        z = z.clone()
        z[:, 40:] = make_w4(N, K, group, dt, "frac", seed=62)[2][:, 40:]
    got = run(A, Wp, s, z, group, tiles + groups, slice_steps, shift=shift)
    assert "w4a16_stream_kernel" in run.log
    check_float_output(got, w4a16_reference(A, Wp, s, z, group), f"{in_dtype} tiles {tiles} groups {groups} {M}x{N}x{K} g{group} {zeros_kind}")


@pytest.mark.parametrize("in_dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("groups", [0, 16])
@pytest.mark.parametrize("zeros_kind", ["int", "frac", None])
@pytest.mark.parametrize("layout", [0, 1])
def test_one_hot_rows_return_the_dequantised_weights(in_dtype, groups, zeros_kind, layout):
    """A = rows of the identity: one non-zero product per output, in 16 bits and in 32, uncut and over K slices."""
    dt = DT[in_dtype]
    if layout and dt is torch.bfloat16:
        pytest.skip("repacked words are for float16")
    N, K, group, M = 272, 128 * 5, 128, 200
    A = torch.eye(K, dtype=dt)[torch.randperm(K, generator=gen(63))[:M]]
    Wp, s, z = make_w4(N, K, group, dt, zeros_kind, seed=64)
    want = ref.dequant_w4(Wp, s, z, group, dt)[:, A.float().argmax(dim=1)].T.contiguous()
    if layout:
        Wp = ref.interleave_weight(Wp.view(torch.int8), 4, "float16").view(torch.uint8).contiguous()
    for out_dtype, steps in ((dt, 5), (torch.float32, 5), (dt, 2)):
        assert_bit_equal(run(A, Wp, s, z, group, 8 + groups, steps, layout, out_dtype), want.to(out_dtype), f"{in_dtype} groups {groups} {zeros_kind} -> {out_dtype}, {steps} steps")


@pytest.mark.parametrize("M,N,K,group,in_dtype,by_xcd", [
    (403, 1280, 12544, 256, torch.float16, True),   # 33.9 us in the order of the grid, 25.7 by XCD
    (482, 1024, 16256, 128, torch.float16, True),   # 40.3, 29.1
    (450, 652, 15360, 64, torch.bfloat16, True),    # blocks of weight rows that are no multiple of eight, the last one cut
    (250, 14592, 2048, 128, torch.bfloat16, True),  # no K slices
    (257, 640, 10240, 128, torch.float16, False),   # 16.1, 18.5 by XCD
])
def test_order_of_the_work_groups(M, N, K, group, in_dtype, by_xcd):
    A = torch.randn(M, K, generator=gen(71)).to(in_dtype)
    Wp, s, z = make_w4(N, K, group, in_dtype, "int", seed=72)
    got = run(A, Wp, s, z, group, 0, 0)
    assert ("by XCD" in run.log) == by_xcd or _abi.load().tlq_device_cu_count() != 256, run.log
    check_float_output(got, w4a16_reference(A, Wp, s, z, group), f"{M}x{N}x{K}")


@pytest.mark.parametrize("M,N,K,group", [(663, 4096, 1792, 128), (1060, 4096, 640, 64), (556, 9216, 512, 256), (640, 896, 4352, 128)])
def test_automatic_choice_above_512_rows(M, N, K, group):
    A = torch.randn(M, K, generator=gen(65)).half()
    Wp, s, z = make_w4(N, K, group, torch.float16, "int", seed=66)
    got = run(A, Wp, s, z, group, 0, 0, algo=_abi.ALGO_AUTO, exact=True)
    assert "w4a16_stream_kernel" in run.log or _abi.load().tlq_device_cu_count() != 256, run.log
    check_float_output(got, w4a16_reference(A, Wp, s, z, group), f"{M}x{N}x{K}")


@pytest.mark.parametrize("s,z", [(float("inf"), 7.0), (float("nan"), 7.0), (-0.5, 300.0), (0.0, -3.0), (65504.0, 0.0), (6e-8, 8.0)])
def test_extreme_scales_and_zero_points(s, z):
    """Infinite, not-a-number, zero, largest and subnormal scales, zero points beyond what folds: the dequantised weights bit for bit."""
    N, K, group, M = 128, 256, 128, 64
    A = torch.zeros(M, K, dtype=torch.float16)
    Wp = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, generator=gen(67))
    S = torch.full((N, K // group), 0.01, dtype=torch.float16)
    Z = torch.full((N, K // group), 8.0, dtype=torch.float16)
    S[5, 0], Z[5, 0] = s, z
    A[torch.arange(M), torch.arange(M)] = 1.0  # (only products with the first group; 0 x inf and 0 x nan make every output of that row nan)
    W = ref.dequant_w4(Wp, S, Z, group, torch.float16)
    want = (A.double() @ W.double().T).half()
    for tiles in (4, 20):
        got = run(A, Wp, S, Z, group, tiles, 0)
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        assert_bit_equal(torch.nan_to_num(got + 0.0), torch.nan_to_num(want + 0.0), f"scale {s} zero point {z}")


@pytest.mark.parametrize("s,z", [(float("inf"), 7.0), (float("nan"), 7.0), (-0.5, 300.0), (0.0, -3.0), (3.0e38, 0.0), (1.2e-38, 8.0)])
def test_extreme_scales_and_zero_points_in_bfloat16(s, z):
    """The same in bfloat16: the largest finite scale overflows in the product of scale and weight, the smallest normal one does not vanish."""
    N, K, group, M = 128, 256, 128, 64
    A = torch.zeros(M, K, dtype=torch.bfloat16)
    Wp = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, generator=gen(67))
    S = torch.full((N, K // group), 0.01, dtype=torch.bfloat16)
    Z = torch.full((N, K // group), 8.0, dtype=torch.bfloat16)
    S[5, 0], Z[5, 0] = s, z
    A[torch.arange(M), torch.arange(M)] = 1.0
    W = ref.dequant_w4(Wp, S, Z, group, torch.bfloat16)
    want = (A.double() @ W.double().T).to(torch.bfloat16)
    for tiles in (4, 20):
        got = run(A, Wp, S, Z, group, tiles, 0)
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        assert_bit_equal(torch.nan_to_num(got + 0.0), torch.nan_to_num(want + 0.0), f"scale {s} zero point {z}")
