"""The activation quantiser where several work-groups share a row (up to two rows per CU, rows of 4096 to 16384 values): bit for bit the oracle's, at
the edges of the parts, the chunks per lane and the row counts, for each type; and where amax sits in the last chunk, in no part's own or nowhere."""
import pytest
import torch

from oracle import ref
from tilelang_ascend_amd import ops

pytestmark = pytest.mark.gpu
_T = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float32": torch.float32}


@pytest.mark.parametrize("in_dtype", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("round_scale", [False, True])
@pytest.mark.parametrize("M,N", [(1, 4096), (1, 4104), (3, 8192), (31, 16384), (32, 14336), (33, 14336), (64, 8200), (65, 12288), (128, 16384), (129, 4096), (200, 5504),
                                 (256, 16376), (511, 4096), (512, 8192), (513, 4096), (32, 4088), (7, 16392)])
def test_parts_of_a_row(in_dtype, round_scale, M, N):
    print(f"act quant parts M={M} N={N} {in_dtype} round={round_scale}", flush=True)
    x = torch.randn(M, N, generator=torch.Generator().manual_seed(M + N)).to(_T[in_dtype])
    x[0] = 0
    x[M - 1, N - 1] = 97.0  # the row's maximum in its last value
    x[M // 2, 5] = float("nan")  # left out of the maximum
    x[:, 7] = -0.0
    want_y, want_s = ref.act_quant_torch(torch.nan_to_num(x, nan=0.0), round_scale, exact_log2=True)
    y, s = ops.act_quant_kernel_int8_optimized(N, round_scale=round_scale, in_dtype=in_dtype)(x.cuda())
    y, s = y.cpu(), s.cpu()
    seen = ~torch.isnan(x)
    assert torch.equal(s, want_s.reshape(-1)) and torch.equal(y[seen], want_y[seen])


@pytest.mark.parametrize("M,N", [(8200, 4096), (4099, 2056), (4100, 4104)])
def test_many_rows(M, N):
    """More rows than work-groups, and row lengths on either side of one wavefront per row."""
    x = torch.randn(M, N, generator=torch.Generator().manual_seed(M + N)).to(torch.bfloat16)
    y, s = ops.act_quant_kernel_int8_optimized(N)(x.cuda())
    want_y, want_s = ref.act_quant_torch(x)
    assert torch.equal(s.cpu(), want_s.reshape(-1)) and torch.equal(y.cpu(), want_y)
