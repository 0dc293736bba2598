"""The streaming W4A16 kernel on slices of several windows of scales: blocks of 256 weight rows under 33 .. 96 activation rows hold 32 groups at a time there
(16 in slices of one window).  Group counts around one and two windows, each way the scales reach LDS, a zero point that leaves the folded dequantiser in a later window."""
import pytest
import torch

from helpers import check_float_output, gen, make_w4, w4a16_reference
from test_stream_groups import run


@pytest.mark.gpu
@pytest.mark.parametrize("M,tiles", [(60, 4), (90, 6), (97, 6)])
@pytest.mark.parametrize("group,groups,slice_steps,shift", [
    (128, 17, 17, 0), (128, 31, 31, 0), (128, 32, 32, 0), (128, 33, 33, 0), (128, 65, 65, 0),  # odd counts: dwords, gathers from the second window on
    (64, 34, 17, 0), (64, 64, 32, 0), (64, 96, 48, 2), (32, 68, 17, 0), (32, 96, 24, 1), (64, 80, 20, 0)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("zeros", ["int", "late", "scalar8"])
def test_windows(M, tiles, group, groups, slice_steps, shift, dtype, zeros):
    N, K = 276, group * groups
    A = torch.randn(M, K, generator=gen(groups)).to(dtype)
    Wp, s, z = make_w4(N, K, group, dtype, "int" if zeros == "late" else zeros, seed=groups + M)
    if zeros == "late":
        z[:, groups - 1] += 0.5
    check_float_output(run(A, Wp, s, z, group, tiles, slice_steps, shift=shift), w4a16_reference(A, Wp, s, z, group), f"{groups} groups of {group}")
