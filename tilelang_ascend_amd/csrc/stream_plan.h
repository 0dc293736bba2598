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
  bool by_xcd;            // the order of the work-groups (stream_item)
};
// Which block of weight rows, K slice and block of activation rows work-group `id` of n_blocks x slices x m_blocks takes.  Work-groups go to the
// eight XCDs round-robin.  Weight rows fastest: with eight blocks of weight rows and more every XCD meets all slices of all activations, and fetches them
// into its L2.  By XCD: each takes an eighth of the work in a row -- slice after slice, in a slice a run of weight rows with all their activation rows.
struct StreamItem {
  int n, slice, m;
};
__host__ __device__ inline StreamItem stream_item(uint32_t id, uint32_t n_blocks, uint32_t slices, uint32_t m_blocks, bool by_xcd) {
  if (!by_xcd) return StreamItem{(int)(id % n_blocks), (int)(id / n_blocks % slices), (int)(id / n_blocks / slices)};
  const uint32_t total = n_blocks * slices * m_blocks, xcd = id & 7u, rest = total & 7u;
  const uint32_t at = xcd * (total >> 3) + (xcd < rest ? xcd : rest) + (id >> 3), t = at / m_blocks;
  return StreamItem{(int)(t % n_blocks), (int)(t / n_blocks), (int)(at % m_blocks)};
}
// short_windows: the plan as it is if no window of the scale area holds more groups than those of a slice of one window (fewer K slices on some problems).
StreamPlan w4a16_stream_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus, bool short_windows = false);
int gemm_w4a16_stream(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t M, int64_t N,
                      int64_t K, int64_t group, float zero_scalar, int in_dtype, int out_dtype, int w_layout, const StreamPlan& p,
                      float* partial, hipStream_t st);

}  // namespace tlq
