// The small-tile kernels (gemm_w4a16_small.hip; gemm_small.{h,hip}): what a plan is and what the entry points call.
#pragma once
#include "tlq_common.h"

namespace tlq {

// Tile (16 mt activation rows x 16 rt weight rows), wavefronts per work-group (the cut of K), estimated time of a call; ok = false
// where the kernel does not apply.
struct SmallTile {
  bool ok;
  int mt, rt, waves;
  double us;
};

// W4A16.  force_*: a forced variant, 0 = by estimate.  `what`: the entry point and family on whose behalf the kernel runs, for the
// launch log and error texts.
SmallTile w4a16_small_plan(int64_t M, int64_t N, int64_t K, int64_t group, const void* scales, const void* zeros, int force_waves, int force_rt, int force_mt);
int gemm_w4a16_small(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t M, int64_t N, int64_t K, int64_t group,
                     float zero_scalar, int in_dtype, int out_dtype, int w_layout, const SmallTile& p, const char* what, hipStream_t st);

// The int8, W4A8 and plain 16-bit products, by how their weights are stored
enum SmallW { kSmallNK = 0 /* int8 [N, K] */, kSmallKN8 = 1 /* int8 [K, N] */, kSmallKN16 = 2 /* 16-bit [K, N] */, kSmallW4 = 3 /* packed int4 [N, K / 2] */ };
// how the packed weights are multiplied (gemm_small.h); a kind of its own for small_tile_plan, which prices it
enum { kSmallW4Times16 = 4 };
inline bool small_w4a8_times16(int sign_mode, int64_t K) { return (sign_mode == TLQ_S4_TWOS || sign_mode == TLQ_S4_OFFSET8) && K <= 131071; }
SmallTile small_tile_plan(int kind, int64_t batch, int64_t M, int64_t N, int64_t row_bytes);  // row_bytes: bytes of K in an activation row
bool small_tile_forced();
int small_i8(const SmallTile& t, const void* A, const void* B, void* C, int64_t batch, int64_t M, int64_t N, int64_t K, int b_layout, hipStream_t st);
int small_w8a8(const SmallTile& t, const void* A, const void* B, const void* scale_a, const void* scale_b, void* C, int64_t batch, int64_t M, int64_t N, int64_t K,
               int64_t n_scale_b, int b_layout, int out_dtype, hipStream_t st);
int small_w4a8(const SmallTile& t, const void* A, const void* Wp, void* C, int64_t M, int64_t N, int64_t K, int sign_mode, hipStream_t st);
int small_f16(const SmallTile& t, const void* A, const void* B, void* C, int64_t batch, int64_t M, int64_t N, int64_t K, int in_dtype, int out_dtype, hipStream_t st);  // [K, N] weights

}  // namespace tlq
