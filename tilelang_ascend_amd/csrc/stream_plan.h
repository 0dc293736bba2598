// Launch geometry of the streaming W4A16 kernel (gemm_w4a16_stream.hip), and its launch.
#pragma once

#include "tlq_common.h"

namespace tlq {

constexpr int64_t kStreamMaxRows = 8192;  // activation rows that a plan is made for (512 where the kernel is asked for by name)
struct StreamPlan {
  bool ok;                // the kernel applies
  int tm;                 // 16-row activation tiles per work-group: 2, 4, 6, 8
  int m_blocks, n_blocks;
  int split, slice_steps; // K slices, steps of 128 values in each
  int kg;                 // groups of wavefronts over K: 2 (256 weight rows per work-group) or 4 (128)
  double us;              // estimate
};
StreamPlan w4a16_stream_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus);
int gemm_w4a16_stream(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t M, int64_t N,
                      int64_t K, int64_t group, float zero_scalar, int in_dtype, int out_dtype, int w_layout, const StreamPlan& p,
                      float* partial, hipStream_t st);

}  // namespace tlq
