// Launches of the small-tile kernel (gemm_small.h): int8 products (exact int32, or rescaled), W4A8, plain 16-bit products with
// [K, N] weights; the choice of tile and wavefronts, and an estimate of the call's time that the callers hold against their own.
#include "gemm_small.h"

namespace tlq {

static thread_local int g_small_waves = 0, g_small_tiles = 0;  // tuning and tests: forced variant; tiles < 0: never

// The estimate, in microseconds: a launch, rounds of the work-groups the machine holds at once (LDS and registers) x the longest chain
// of steps in a wavefront, what a CU does per step of its share of the tiles (operand reads, multiplications), what it stores, and
// the weights' trip from memory -- once, and again for every further tile of activation rows.  Fitted per kind to 970 problems (M 1 .. 1500,
// N 256 .. 14400, K 256 .. 14336, one to eight batches) x up to 45 forced variants each: 14 - 22 % rms over all variants; the
// variant it picks is 4 - 5 % behind the fastest on average.
// Packed int4 weights multiplied as 16 times their value (kSmallW4Times16) have a row of their own: the one before it is 1.37 x what they
// take.  700 problems (M 1 .. 1500, N 256 .. 14336, K 256 .. 14336) x up to 36 variants, the adding of the wavefronts' tiles as a further term:
// 11 % rms; 6.5 % for the variant it picks, which is 3.4 % behind the fastest on average (3.9 with the other row).
struct SmallCost {
  double launch, round, step, rt, rt_mt, store, again, weights, sums;
};
static constexpr SmallCost kSmallCost[5] = {{3.4, 1.33, 0.049, 0.0028, 0.0092, 0.047, 0.19, 0.29, 0.0},   // int8 [N, K] (rt: stands for mt here)
                                            {2.4, 1.57, 0.112, 0.0, 0.0112, 0.080, 0.29, 1.35, 0.0},      // int8 [K, N]
                                            {1.75, 1.43, 0.085, 0.0045, 0.0106, 0.020, 0.22, 0.58, 0.0},  // 16-bit [K, N]
                                            {3.0, 0.71, 0.391, 0.0444, 0.0118, 0.046, 0.0, 0.0, 0.0},    // packed int4
                                            {2.01, 0.815, 0.1635, 0.0058, 0.0086, 0.0339, 0.147, 0.344, 0.0159}};  // the same, times 16

static SmallTile small_tile_now(int kind, int64_t batch, int64_t M, int64_t N, int64_t steps) {
  SmallTile best{false, 0, 0, 0, 0.0};
  int cus = tlq_device_cu_count();
  if (cus <= 0) cus = 256;
  const SmallW w = kind == kSmallW4Times16 ? kSmallW4 : (SmallW)kind;
  for (int mt = 1; mt <= 4; mt *= 2) {
    if (g_small_tiles > 0 ? mt != g_small_tiles / 10 : mt > 1 && mt * 8 >= M) continue;  // (half of the tile would be padding)
    for (int rt = 1; rt <= 4; rt *= 2) {
      if ((w == kSmallKN8 || w == kSmallKN16) && rt != 4) continue;
      if (g_small_tiles > 0 && rt != g_small_tiles % 10) continue;
      const int lds = small_lds(w, rt, mt), cap = rt * mt <= 4 ? 16 : 8, most = 160 * 1024 / lds < cap ? 160 * 1024 / lds : cap;
      const int64_t tiles_m = ceil_div(M, (int64_t)16 * mt), tiles_n = ceil_div(N, (int64_t)16 * rt), blocks = batch * tiles_m * tiles_n;
      if (blocks > 1 << 20 || tiles_m > 65535 || batch > 65535) continue;
      for (int want = g_small_waves ? g_small_waves : 1; want <= (g_small_waves ? g_small_waves : 16); want *= 2) {
        int64_t wv = want < most ? want : most;
        if (wv > steps) wv = steps;
        int64_t held = 160 * 1024 / (wv * lds);
        const int64_t by_registers = (rt * mt <= 4 ? 32 : 12) / wv;
        if (held > by_registers) held = by_registers;
        if (held < 1) held = 1;
        const double rounds = (double)ceil_div(blocks, cus * held), per_cu = (double)ceil_div(blocks, (int64_t)cus) * (double)steps;
        const SmallCost& c = kSmallCost[kind];
        const double w_mb5 = (double)batch * (double)N * (double)steps * (w == kSmallW4 ? 64.0 : 128.0) / 5e6;  // us at 5 TB/s
        const double us = c.launch + rounds * (c.round + c.step * (double)ceil_div(steps, wv)) + per_cu * (c.rt * (w == kSmallNK ? mt : rt) + c.rt_mt * rt * mt) +
                          (c.store + (wv > 1 ? c.sums * (double)wv : 0.0)) * (double)ceil_div(blocks, (int64_t)cus) * rt * mt + w_mb5 * (c.weights + c.again * (double)(tiles_m - 1));
        if (!best.ok || us < best.us * 0.995) best = SmallTile{true, mt, rt, (int)wv, us};
      }
    }
  }
  if (best.us < 5.0) best.us = 5.0;  // (the launch)
  return best;
}

SmallTile small_tile_plan(int kind, int64_t batch, int64_t M, int64_t N, int64_t row_bytes) {
  if (g_small_tiles < 0 || batch < 1 || M < 1 || N < 16 || row_bytes < 128 || row_bytes % 128 != 0) return SmallTile{false, 0, 0, 0, 0.0};
  return small_tile_now(kind, batch, M, N, row_bytes / 128);
}
bool small_tile_forced() { return g_small_tiles > 0; }

int small_i8(const SmallTile& t, const void* A, const void* B, void* C, int64_t batch, int64_t M, int64_t N, int64_t K, int b_layout, hipStream_t st) {
  EpiInt32::Params pe{(int32_t*)C, N, M * N};
  const SmallParams p = small_params(A, B, M, N, K, b_layout == TLQ_B_NK ? K : N, N * K);
  return b_layout == TLQ_B_NK ? launch_tile<MmaI8, kSmallNK, EpiInt32>(t, p, pe, batch, M, N, "tlq_gemm_i8", st)
                              : launch_tile<MmaI8, kSmallKN8, EpiInt32>(t, p, pe, batch, M, N, "tlq_gemm_i8", st);
}

int small_w8a8(const SmallTile& t, const void* A, const void* B, const void* scale_a, const void* scale_b, void* C, int64_t batch, int64_t M, int64_t N, int64_t K,
               int64_t n_scale_b, int b_layout, int out_dtype, hipStream_t st) {
  EpiRescale::Params pe{C, N, M, (const float*)scale_a, (const float*)scale_b, n_scale_b, out_dtype};
  const SmallParams p = small_params(A, B, M, N, K, b_layout == TLQ_B_NK ? K : N, N * K);
  return b_layout == TLQ_B_NK ? launch_tile<MmaI8, kSmallNK, EpiRescale>(t, p, pe, batch, M, N, "tlq_gemm_w8a8", st)
                              : launch_tile<MmaI8, kSmallKN8, EpiRescale>(t, p, pe, batch, M, N, "tlq_gemm_w8a8", st);
}

int small_w4a8(const SmallTile& t, const void* A, const void* Wp, void* C, int64_t M, int64_t N, int64_t K, int sign_mode, hipStream_t st) {
  EpiInt32::Params pe{(int32_t*)C, N, M * N};
  SmallParams p = small_params(A, Wp, M, N, K, K / 2, 0);
  p.sign_mode = (uint16_t)sign_mode;
  if (small_w4a8_times16(sign_mode, K)) return small_w4a8_times16_launch(t, p, pe, M, N, st);
  return launch_tile<MmaI8, kSmallW4, EpiInt32>(t, p, pe, 1, M, N, "tlq_gemm_w4a8", st);
}

int small_f16(const SmallTile& t, const void* A, const void* B, void* C, int64_t batch, int64_t M, int64_t N, int64_t K, int in_dtype, int out_dtype, hipStream_t st) {
  EpiFloat::Params pe{C, N, M * N, out_dtype};
  const SmallParams p = small_params(A, B, M, N, K * 2, N * 2, N * K * 2);
  return in_dtype == TLQ_F16 ? launch_tile<MmaF16, kSmallKN16, EpiFloat>(t, p, pe, batch, M, N, "tlq_gemm_f16", st)
                             : launch_tile<MmaBF16, kSmallKN16, EpiFloat>(t, p, pe, batch, M, N, "tlq_gemm_f16", st);
}

}  // namespace tlq

extern "C" {
// Forces the small-tile kernel of the int8, W4A8 and plain 16-bit products: tiles = 10 x activation tiles + weight tiles (1 | 2 | 4 each),
// waves wavefronts per work-group; 0, 0: by estimate; tiles < 0: never.
void tlq_tune_small(int waves, int tiles) { tlq::tuning_changed(), tlq::g_small_waves = waves < 0 || waves > 16 ? 0 : waves, tlq::g_small_tiles = tiles; }
int tlq_debug_small_tile(int kind, int64_t batch, int64_t M, int64_t N, int64_t row_bytes, void* plan_out) {
  const tlq::SmallTile t = tlq::small_tile_plan(kind, batch, M, N, row_bytes);
  if (plan_out) {
    int64_t* o = (int64_t*)plan_out;
    o[0] = 16 * t.mt, o[1] = 16 * t.rt, o[2] = t.waves, o[3] = (int64_t)(t.us * 1000.0);
  }
  return t.ok ? 1 : 0;
}
}
