// The small-tile kernel (gemm_small.h) on packed int4 weights multiplied as 16 times their value: a file of its own beside
// gemm_small.hip, whose kernels take as long to compile.
#include "gemm_small.h"

namespace tlq {

int small_w4a8_times16_launch(const SmallTile& t, const SmallParams& p, const EpiInt32::Params& pe, int64_t M, int64_t N, hipStream_t st) {
  return launch_tile<MmaI8, kSmallW4, EpiInt32, true>(t, p, pe, 1, M, N, "tlq_gemm_w4a8", st);
}

}  // namespace tlq
