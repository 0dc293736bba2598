"""The kernel and tile of a plain product of one launch, asked on the host (tlq_debug_gemm_choice), and the loads of 192-row tiles by four wavefronts."""
import ctypes

import pytest

from tilelang_ascend_amd import _abi

PLAIN_128, RING, PLAIN_256, QUAD, QUAD_256 = 1, {2, 3, 4, 5}, 6, {7, 8, 9, 10, 11}, 12
F16_KN, F16_NK, I8_KN, I8_NK = range(4)
SHAPES = [(b, m, n, k) for b in (1, 3) for m in (1, 32, 33, 128, 129, 512, 2050, 8192) for n in (16, 272, 4096, 14336) for k in (64, 128, 264, 512, 1024, 4096)]


@pytest.fixture
def lib():
    lib = _abi.load()
    yield lib
    lib.tlq_tune_gemm_groups(0), lib.tlq_tune_gemm_quad(0), lib.tlq_tune_gemm_slots(1)


def k_bytes(kind, k):
    return k if kind >= I8_KN else 2 * k


@pytest.mark.parametrize("kind", range(4))
def test_every_choice_can_run(lib, kind):
    """No ring kernel on up to 32 rows or fewer than four stages of K, no four wavefronts on a partial stage, 256-row tiles above 128 rows only; an estimate with each."""
    us = ctypes.c_double()
    for b, m, n, k in SHAPES:
        v = lib.tlq_debug_gemm_choice(kind, b, m, n, k, ctypes.addressof(us))
        kb = k_bytes(kind, k)
        assert 1 <= v <= 12 and us.value > 0, (b, m, n, k, v)
        assert not (v in RING and (m <= 32 or kb <= 384)), (b, m, n, k, v)
        assert not (v in QUAD | {QUAD_256} and (kb % 128 or kb < 256)), (b, m, n, k, v)
        assert not (v in QUAD and (m <= 32 or b * m * n < 64 * 128 * 128)), (b, m, n, k, v)
        assert not (v in {PLAIN_256, QUAD_256} and m <= 128), (b, m, n, k, v)
        assert v == lib.tlq_debug_gemm_choice(kind, b, m, n, k, None)


@pytest.mark.parametrize("kind", range(4))
def test_the_tuning_hooks_hold(lib, kind):
    for b, m, n, k in SHAPES:
        stages, whole = -(-k_bytes(kind, k) // 128), k_bytes(kind, k) % 128 == 0
        auto = lib.tlq_debug_gemm_choice(kind, b, m, n, k, None)
        lib.tlq_tune_gemm_groups(1)
        assert lib.tlq_debug_gemm_choice(kind, b, m, n, k, None) not in RING
        lib.tlq_tune_gemm_groups(3)
        assert (lib.tlq_debug_gemm_choice(kind, b, m, n, k, None) == 3) == (stages >= 4)
        lib.tlq_tune_gemm_groups(0)
        lib.tlq_tune_gemm_quad(1)
        assert lib.tlq_debug_gemm_choice(kind, b, m, n, k, None) not in QUAD
        lib.tlq_tune_gemm_quad(8)
        assert (lib.tlq_debug_gemm_choice(kind, b, m, n, k, None) == 8) == (whole and stages >= 2) or auto == 8
        lib.tlq_tune_gemm_quad(0)
        lib.tlq_tune_gemm_slots(0)
        assert lib.tlq_debug_gemm_choice(kind, b, m, n, k, None) not in QUAD | {QUAD_256}
        lib.tlq_tune_gemm_slots(1)
        assert lib.tlq_debug_gemm_choice(kind, b, m, n, k, None) == auto


def test_bad_arguments_have_no_choice(lib):
    for bad in ((-1, 1, 64, 64, 64), (4, 1, 64, 64, 64), (0, 0, 64, 64, 64), (0, 1, 0, 64, 64), (0, 1, 64, 0, 64), (0, 1, 64, 64, 0)):
        assert lib.tlq_debug_gemm_choice(*bad, None) == 0


def test_activation_loads_of_192_row_tiles(lib):
    for rows, k in [(256, 64), (300, 192), (1000, 4160), (4096, 4096), (193, 128), (191, 128), (1, 64), (2305, 320)]:
        for row_bytes in (k, 2 * k):
            if row_bytes % 128 == 0:  # (whole stages of K alone)
                assert lib.tlq_debug_check_gemm_addressing(0, rows, row_bytes, 192, 256) == 0, _abi.last_error()
