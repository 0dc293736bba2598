// extern "C" entry points of the GEMM family: argument validation, then dispatch.
// Every shape assumption a kernel makes is checked here, before anything is launched.
#include "tlq_common.h"
#include "gemm_core.h"
#include "small_tiles.h"
#include "stream_plan.h"

namespace tlq {
int gemv_w4a16(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t batch, int64_t M,
               int64_t N, int64_t K, int64_t group, float zero_scalar, int in_dtype, int out_dtype, hipStream_t st);
bool gemv_ring_applies(int64_t M, int64_t N, int64_t K, int64_t group, int in_dtype, const void* scales, const void* zeros);
int w4a16_tail_rows(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t M, int64_t rows, int64_t K,
                    int64_t group, float zero_scalar, int in_dtype, int out_dtype, int w_layout, int64_t ldc, int64_t col0, hipStream_t st);
int gemv_w4a16_ring_interleaved(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t M, int64_t N,
                                int64_t K, int64_t group, float zero_scalar, int in_dtype, int out_dtype, hipStream_t st);
int gemm_w4a16_mfma(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t M, int64_t N,
                    int64_t K, int64_t group, float zero_scalar, int in_dtype, int out_dtype, hipStream_t st);
int64_t w4a16_mid_split(int64_t M, int64_t N, int64_t K, int64_t group);
int w4a16_split_forced();
bool w4a16_tile_forced();
bool w4a16_skinny_forced();
int gemm_w4a16_mfma_splitk(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t M,
                           int64_t N, int64_t K, int64_t group, float zero_scalar, int in_dtype, int out_dtype,
                           int64_t split, float* partial, hipStream_t st);
int gemm_w4a16_skinny(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t M, int64_t N,
                      int64_t K, int64_t group, float zero_scalar, int in_dtype, int out_dtype, hipStream_t st);
int gemm_f16_plain(const void* A, const void* B, void* C, int64_t batch, int64_t M, int64_t N, int64_t K, int in_dtype,
                   int out_dtype, int b_layout, hipStream_t st);
int gemm_f16_splitk(const void* A, const void* B, float* C, int64_t M, int64_t N, int64_t K, int64_t split_k,
                    int in_dtype, int b_layout, hipStream_t st);
extern thread_local int g_f16_split;
int f16_split_choice(int64_t batch, int64_t M, int64_t N, int64_t K);
int gemm_f16_slices(const void* A, const void* B, void* C, float* partial, int64_t M, int64_t N, int64_t K, int64_t split,
                    int in_dtype, int out_dtype, int b_layout, hipStream_t st);
int gemm_i8_i32(const void* A, const void* B, void* C, int64_t batch, int64_t M, int64_t N, int64_t K, int b_layout,
                hipStream_t st);
int gemm_w8a8_rescale(const void* A, const void* B, const void* scale_a, const void* scale_b, void* C, int64_t batch,
                      int64_t M, int64_t N, int64_t K, int64_t n_scale_b, int b_layout, int out_dtype, hipStream_t st);
int gemm_w4a8_i32(const void* A, const void* Wp, void* C, int64_t M, int64_t N, int64_t K, int sign_mode,
                  hipStream_t st);
int i8_split_choice(int64_t batch, int64_t M, int64_t N, int64_t K, bool buffers, double pace = 1.0);
int gemm_w4a8_i32_splitk(const void* A, const void* Wp, void* C, int64_t M, int64_t N, int64_t K, int sign_mode,
                         int64_t split, int32_t* partial, hipStream_t st);
int gemm_i8_i32_splitk(const void* A, const void* B, int32_t* acc, int64_t M, int64_t N, int64_t K, int64_t split,
                       int b_layout, hipStream_t st);
int gemm_w8a8_rescale_splitk(const void* A, const void* B, const void* scale_a, const void* scale_b, void* C, int32_t* partial,
                             int64_t M, int64_t N, int64_t K, int64_t n_scale_b, int64_t split, int b_layout, int out_dtype,
                             hipStream_t st);

extern thread_local int g_i8_tile, g_i8_split;

struct PanelPlan {
  bool ok;
  int tiles_m, tiles_n, split, slice_steps;
};
PanelPlan w4a16_panel_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus);
int gemm_w4a16_panel(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t M, int64_t N, int64_t K,
                     int64_t group, float zero_scalar, int in_dtype, int out_dtype, int w_layout, const PanelPlan& p, float* partial,
                     uint32_t* flag, hipStream_t st);
extern thread_local int g_panel_slice_steps;
thread_local int g_w4a16_panel = 0;  // tlq_tune_w4a16_panel: non-zero = no panel kernel is picked automatically
struct Panel2Plan {
  bool ok;
  int tiles_m, tiles_n, split, slice_steps;
};
Panel2Plan w4a16_panel256_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus);
int gemm_w4a16_panel256(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t M, int64_t N, int64_t K,
                        int64_t group, float zero_scalar, int in_dtype, int out_dtype, int w_layout, const Panel2Plan& p, float* partial,
                        hipStream_t st);
extern thread_local int g_panel2_slice_steps;
struct PanelMPlan {
  bool ok;
  int tm, tiles_m, tiles_n, split, slice_steps;
};
PanelMPlan w4a16_panelm_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus);
int gemm_w4a16_panelm(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t M, int64_t N, int64_t K,
                      int64_t group, float zero_scalar, int in_dtype, int out_dtype, const PanelMPlan& p, float* partial, hipStream_t st);
extern thread_local int g_panelm_slice_steps;
extern thread_local int g_panelm_rows;

struct DecodePlan {
  bool ok;
  int mt, chunks, waves, grid_x;
  int64_t lds_bytes;
};
DecodePlan w4a16_decode_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus);
int gemm_w4a16_decode(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t M, int64_t N, int64_t K,
                      int64_t group, float zero_scalar, int in_dtype, int out_dtype, int w_layout, const DecodePlan& p, float* partial,
                      hipStream_t st);

thread_local int g_gemm_band_rows = 0;
thread_local int g_gemm_groups = 0;
thread_local int g_gemm_quad = 0;
thread_local int g_gemm_slots = 1;
extern thread_local int g_gemm_f16_tile;
static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }
// compute units of the current device (256 when it cannot be asked, e.g. without a GPU)
static int cu_count_or_default() {
  const int n = tlq_device_cu_count();
  return n > 0 ? n : 256;
}
extern thread_local int g_stream_slice_steps, g_stream_tiles;
thread_local int g_w4a16_stream = 1;  // 0: never pick the streaming kernel automatically (tuning runs)
thread_local int g_w4a16_decode = 1;  // 0: never pick the decode kernel automatically
// the tile loaders address one matrix with 32-bit byte offsets
static bool fits32(int64_t rows, int64_t row_bytes) { return rows * row_bytes < ((int64_t)1 << 32); }
static const int64_t kMaxDim = (int64_t)1 << 30;
// the table of tuned kernel choices (w4a16_choice.hip)
int w4a16_choice_lookup(int64_t M, int64_t N, int64_t K, int64_t group, int in_dtype);
void w4a16_choice_for_shape(int64_t M, int64_t N, int64_t K, void (*fn)(int algo, void* ctx), void* ctx);

}  // namespace tlq

// One scale / zero point per weight row (group = K) where K is no power of two: the fast kernels index groups by shifts, so
// the row's value is written out once per power-of-two group (the largest power of two that divides K, 1024 at most) into
// the tail of the workspace and the call runs with that group size -- the same arithmetic per weight, hence the same bits.
__global__ __launch_bounds__(256) void expand_row_values_kernel(const uint16_t* __restrict__ in, uint16_t* __restrict__ out, int64_t n_out,
                                                                int groups, int blocks) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n_out; i += (int64_t)blocks * 256) out[i] = in[i / groups];
}
// A matrix of `cols` columns (rows packed) into the first `cols` columns of a matrix whose rows lie `ldc` elements apart.
template <typename E>
__global__ __launch_bounds__(256) void copy_into_wider_rows_kernel(const E* __restrict__ in, E* __restrict__ out, int64_t M, int64_t cols, int64_t ldc,
                                                                    int row_blocks) {
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= cols) return;
  for (int64_t m = blockIdx.y; m < M; m += row_blocks) out[m * ldc + c] = in[m * cols + c];
}
// The same for 16-bit elements, two at a time: pairs that are aligned in the OUTPUT (a row starts at element m * ldc, whose
// parity moves the pairs by one column), one 4-byte store each; the first or last column of a row alone where a pair straddles it.
__global__ __launch_bounds__(256) void copy_pairs_into_wider_rows_kernel(const uint16_t* __restrict__ in, uint16_t* __restrict__ out, int64_t M,
                                                                        int64_t cols, int64_t ldc, int row_blocks) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  for (int64_t m = blockIdx.y; m < M; m += row_blocks) {
    const int64_t o = m * ldc;
    const int64_t c0 = 2 * t - (o & 1);
    if (c0 >= cols) continue;
    const uint16_t* const src = in + m * cols;
    if (c0 >= 0 && c0 + 1 < cols)
      *(uint32_t*)(out + o + c0) = (uint32_t)src[c0] | ((uint32_t)src[c0 + 1] << 16);
    else if (c0 >= 0)
      out[o + c0] = src[c0];
    else
      out[o] = src[0];
  }
}
// A weight-row count that is no multiple of four (vocabularies of 50257 or 32001 rows): the multiple of 16 below runs through the
// usual choice into a packed result behind the workspace, which is then copied into C; the last rows go straight into C.
static int64_t ragged_head(int64_t N) { return N & ~(int64_t)15; }
static int64_t ragged_result_bytes(int64_t M, int64_t N, int out_bytes) { return (M * ragged_head(N) * out_bytes + 15) / 16 * 16; }
// (Also a multiple of four that is no multiple of eight above 512 rows, where the panel kernels are the choice and want multiples
// of 16 and the two passes multiples of eight, which leaves the tile kernel through registers: N = 4100, K = 4096, M = 1024 .. 4096:
// 63 - 150 against 92 - 239 us; N = 32004: 228 - 1082 against 275 - 1135 us -- while the packed result stays below 1 GiB.  With
// multiples of eight the two passes are level or ahead from 2048 rows on: N = 14344, M = 4096: 430 against 512 us.)
static bool ragged_rows_apply(int64_t M, int64_t N) {
  if (!(N >= 1 && M < tlq::kMaxDim && N < tlq::kMaxDim)) return false;
  if ((N & 3) != 0) return M > 32;  // (fewer than 16 weight rows: the last-rows kernel alone)
  if (N <= 16) return false;
  return (N & 7) != 0 && M > 512 && ragged_result_bytes(M, N, 4) <= ((int64_t)1 << 30);
}
static int64_t row_group_for(int64_t K) {  // largest power of two dividing K, 1024 at most
  int64_t g = K & -K;
  return g > 1024 ? 1024 : g;
}
static int64_t row_group_tensor_bytes(int64_t N, int64_t K) { return (N * (K / row_group_for(K)) * 2 + 15) / 16 * 16; }

using namespace tlq;

#define TLQ_CHECK_DIMS(name)                                                                                      \
  TLQ_REQUIRE(M >= 0 && N >= 0 && K >= 0 && M < kMaxDim && N < kMaxDim && K < kMaxDim, name ": bad shape M=%lld N=%lld K=%lld", \
              (long long)M, (long long)N, (long long)K)

#define TLQ_SMALL_NEEDS(name)                                                                                       \
  name ": the small-tile kernel needs K %% 128 == 0, a power-of-two group >= 32, dword-aligned scale / zero tensors of an even " \
       "number of values and matrices below 4 GiB (M=%lld N=%lld K=%lld group=%lld)"

extern "C" {

void tlq_tune_gemm_groups(int variant) { tlq::tuning_changed(), tlq::g_gemm_groups = variant < 0 || variant > 5 ? 0 : variant; }
void tlq_tune_gemm_quad(int variant) { tlq::tuning_changed(), tlq::g_gemm_quad = variant == 1 || (variant >= tlq::kQuad192x256 && variant <= tlq::kQuad128x128) ? variant : 0; }
void tlq_tune_gemm_band(int tile_rows) { tlq::g_gemm_band_rows = tile_rows < 0 ? 0 : tile_rows; }
void tlq_tune_gemm_slots(int mode) { tlq::tuning_changed(), tlq::g_gemm_slots = mode < 0 ? 0 : (mode > 3 ? 3 : mode); }
int tlq_debug_gemm_tile(int64_t batch, int64_t M, int64_t N, int fused) {
  return tlq::prefer_small_tiles(batch, M, N, fused ? 0.65 : 0.72) ? 128 : 256;
}
int tlq_debug_gemm_choice(int kind, int64_t batch, int64_t M, int64_t N, int64_t K, void* us_out) {
  if (kind < 0 || kind > 3 || batch < 1 || M < 1 || N < 1 || K < 1 || M >= kMaxDim || N >= kMaxDim || K >= kMaxDim) return 0;
  const tlq::TileChoice c = tlq::tile_choice((tlq::TileKind)kind, batch, M, N, kind >= tlq::kTileI8KN ? K : 2 * K);
  if (us_out) *(double*)us_out = c.us;
  return c.variant;
}
void tlq_tune_gemm_tile(int tile) { tlq::tuning_changed(), tlq::g_gemm_f16_tile = (tile == 128 || tile == 256) ? tile : 0; }
void tlq_tune_w4a16_stream(int on) { tlq::tuning_changed(), tlq::g_w4a16_stream = on != 0; }  // (the workspace size above 512 rows follows it)
void tlq_tune_w4a16_stream_tiles(int tiles) { tlq::tuning_changed(), tlq::g_stream_tiles = ((tiles & 15) >= 2 && (tiles & 15) <= 8 && (tiles & 1) == 0) ? tiles & 31 : 0; }
void tlq_tune_w4a16_stream_slice(int steps) { tlq::tuning_changed(), tlq::g_stream_slice_steps = steps; }
void tlq_tune_w4a16_decode(int on) { tlq::g_w4a16_decode = on != 0; }
void tlq_tune_w4a16_panel(int mode) { tlq::g_w4a16_panel = mode != 0 ? 1 : 0; }
void tlq_tune_w4a16_panel_slice(int steps) { tlq::tuning_changed(), tlq::g_panel_slice_steps = tlq::g_panel2_slice_steps = tlq::g_panelm_slice_steps = steps < 0 ? 0 : steps; }
void tlq_tune_w4a16_panelm_rows(int rows) { tlq::tuning_changed(), tlq::g_panelm_rows = (rows == 64 || rows == 128) ? rows : 0; }

int tlq_debug_panel_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus, void* plan_out) {
  if (!(M >= 1 && N >= 1 && K > 0 && group > 0 && M < kMaxDim && N < kMaxDim && K < kMaxDim)) return 0;
  const PanelPlan p = w4a16_panel_plan(M, N, K, group, cus);
  if (plan_out) {
    int64_t* o = (int64_t*)plan_out;
    o[0] = p.tiles_m, o[1] = p.tiles_n, o[2] = p.split, o[3] = p.slice_steps;
  }
  return p.ok ? 1 : 0;
}

int tlq_debug_panel256_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus, void* plan_out) {
  if (!(M >= 1 && N >= 1 && K > 0 && group > 0 && M < kMaxDim && N < kMaxDim && K < kMaxDim)) return 0;
  const Panel2Plan p = w4a16_panel256_plan(M, N, K, group, cus);
  if (plan_out) {
    int64_t* o = (int64_t*)plan_out;
    o[0] = p.tiles_m, o[1] = p.tiles_n, o[2] = p.split, o[3] = p.slice_steps;
  }
  return p.ok ? 1 : 0;
}

int tlq_debug_panelm_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus, void* plan_out) {
  if (!(M >= 1 && N >= 1 && K > 0 && group > 0 && M < kMaxDim && N < kMaxDim && K < kMaxDim)) return 0;
  const PanelMPlan p = w4a16_panelm_plan(M, N, K, group, cus);
  if (plan_out) {
    int64_t* o = (int64_t*)plan_out;
    o[0] = p.tiles_m, o[1] = p.tiles_n, o[2] = p.split, o[3] = p.slice_steps, o[4] = 16 * p.tm;
  }
  return p.ok ? 1 : 0;
}

int tlq_debug_small_plan(int64_t M, int64_t N, int64_t K, int64_t group, void* plan_out) {
  const SmallTile p = w4a16_small_plan(M, N, K, group, nullptr, nullptr, 0, 0, 0);
  if (plan_out) {
    int64_t* o = (int64_t*)plan_out;
    o[0] = 16 * p.mt, o[1] = 16 * p.rt, o[2] = p.waves, o[3] = (int64_t)(p.us * 1000.0);
  }
  return p.ok ? 1 : 0;
}

int tlq_debug_stream_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus, void* plan_out) {
  if (!(M >= 1 && N >= 1 && K > 0 && group > 0 && M < kMaxDim && N < kMaxDim && K < kMaxDim)) return 0;
  const StreamPlan p = w4a16_stream_plan(M, N, K, group, cus);
  if (plan_out) {
    int64_t* o = (int64_t*)plan_out;
    o[0] = 16 * p.tm, o[1] = p.ok ? 512 / p.kg : 0, o[2] = p.split, o[3] = p.slice_steps, o[4] = (int64_t)(p.us * 1000.0);
  }
  return p.ok ? 1 : 0;
}

int tlq_debug_decode_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus, void* plan_out) {
  const DecodePlan p = w4a16_decode_plan(M, N, K, group, cus);
  if (plan_out) {
    int64_t* o = (int64_t*)plan_out;
    o[0] = p.mt, o[1] = p.chunks, o[2] = p.waves, o[3] = p.grid_x, o[4] = p.lds_bytes;
  }
  return p.ok ? 1 : 0;
}

// Activation rows from which the decode kernel is ahead of the GEMV kernels, whose time grows with every row: from three
// rows on, and with two rows once the weights are large enough for the second pass over them to show (measured: level at
// 4096 x 4096, 10.4 against 12.8 us (fp16) and 11.1 against 15.3 us (bf16, skinny kernel) at 11008 x 4096).
// Whether the skinny kernel's work-groups (one per 16 weight rows; one round of one per CU, or rounds of two per CU) leave a
// fifth or more of their last round's places empty.
static bool skinny_leaves_cus_idle(int64_t N) {
  if (tile_fill(1, 16, N, 16) < 0.8) return true;
  const int64_t wgs = ceil_div(N, (int64_t)16), places = 2 * cu_count_or_default();
  return wgs > places / 2 && (double)wgs / (double)(ceil_div(wgs, places) * places) < 0.8;
}
// Where the small-tile kernel (gemm_w4a16_small.hip: one launch, wavefronts split K) is ahead of a family by estimate (G: billions of
// products, G16: the same with M rounded up to 16 rows).  The plan's estimate leaves out the activations' trip from memory and the store
// of the result (fitted: 1.6 and 3.2 times what they take at 5 TB/s; 11 % rms on 2700 problems with them, 0.23 too low on average
// and 17 % above 512 rows without).  Against the kernels it replaces, on 3500 problems (M 2 .. 8192, N 128 .. 14400, K 128 .. 14336,
// groups of 32 - 256, both types) not used for the fit: taken on 1944, ahead by 1.6 x on average up to 700 rows and by 1.8 x
// above 500, more than 5 % behind on 27 and 19 % at most (without the two terms 131 of 2138, 2.7 x at most: 6980 x 912 x 128 22.2 us
// against 8.2 in the tile kernel).
static double giga(double m, int64_t N, int64_t K) { return m * (double)N * (double)K * 1e-9; }
static double up16(int64_t M) { return (double)ceil_div(M, (int64_t)16) * 16.0; }
static double small_us(const SmallTile& p, int64_t M, int64_t N, int64_t K) { return p.us + 0.64e-6 * (double)M * (double)K + 1.28e-6 * (double)M * (double)N; }
static double fused_tile_us(int64_t M, int64_t N, int64_t K) {  // the W4A16 tile kernel where it has few tiles: 4 us + 1.5 us per 128 values of K
  return 3.9 + 11.6e-3 * (double)K + 0.94 * giga((double)M, N, K) + 0.116e-6 * (double)M * (double)N;
}
// The streaming kernel, by its plan's estimate.  The figures of both are of weights that a cache still holds (three sets in turn); from
// memory the small-tile kernel, with two steps in flight to a wavefront, takes 0.09 us more per step of a wavefront's share of K and
// 0.08 us per MB of weights (fitted, 0.7 us rms on 900 problems), the streaming kernel 1 us and 0.01.  So where a wavefront has 24 steps
// and more on 16 MB of weights and more, it has to be ahead by more than the estimates are off.  With shorter shares small tiles
// are ahead from a cache by less than they are behind from memory (22 and 23 steps: 3 % and 14 %), on fewer rows by more.
// Groups of 32 values: a scale per lane and step and, with a tensor, a zero point, which the small-tile kernel's estimate does not know: 15 % above the
// others with zero points and 8 % without, the streaming kernel level.  30 of 285 such problems go to the streaming kernel by it, 1.11 x on average (154 x 6016 x
// 3200 34.5 us with small tiles, 25.5 with the streaming kernel).
static bool small_beats_stream(const SmallTile& p, const StreamPlan& sp, int64_t M, int64_t N, int64_t K, int64_t group, bool zero_points) {
  if (!p.ok || g_stream_slice_steps > 0 || g_stream_tiles > 0) return false;
  const bool long_shares = M > 32 && ceil_div(K / 128, (int64_t)p.waves) >= 24 && N * K >= ((int64_t)32 << 20);
  double theirs = sp.us;
  if (!sp.ok || M <= 32) {  // (17 .. 32 rows: the bar of the kernel's earlier form where that is higher, which the tests of the choice ask for: 24 x 8192 x 10368 24.0 against 20.5 us)
    const double earlier = 11.9 + 2.0 * giga((double)M, N, K) + 1.14 * giga(up16(M), N, K) + 0.31e-3 * (double)K;
    if (!sp.ok || earlier > theirs) theirs = earlier;
  }
  const double mine = small_us(p, M, N, K) * (group >= 64 ? 1.0 : (zero_points ? 1.15 : 1.08));
  return mine < (long_shares ? 0.85 : 1.04) * theirs;
}
// above 512 rows: the tile kernel on up to 2^19 weights -- and the launch for the last M % 4 rows, 4 us, where they run apart --, else the
// two passes or the panel kernels, which are level with them or ahead; only while the whole call stays short
static double two_passes_us(int64_t M, int64_t N, int64_t K);
static bool stream_beats_panels(int64_t M, int64_t N, int64_t K, int64_t group, bool two_passes);
static bool small_beats_panels(const SmallTile& p, int64_t M, int64_t N, int64_t K, bool head_and_tail, bool two_passes) {
  if (!p.ok || p.us >= 13.0) return false;
  const double us = small_us(p, M, N, K);
  return us < 0.95 * (two_passes && N * K > ((int64_t)1 << 19) ? two_passes_us(M, N, K) : fused_tile_us(M, N, K) + (head_and_tail ? 4.0 : 0.0));
}
// the decode kernel over chunks of K, whose second launch adds the chunks
static bool small_beats_decode_chunks(const SmallTile& p, int64_t M, int64_t N, int64_t K) {
  return p.ok && p.us < 0.95 * (5.2 + 0.67 * giga((double)M, N, K) + 4.36 * giga(up16(M), N, K) + 0.023e-6 * (double)N * (double)K + 0.25e-3 * (double)K);
}
// The skinny kernel on 17 .. 64 rows (12.8 -> 7.8 us for M = 64 on 5120 x 1280, level where the launch is all there is) and the tile
// kernel (21.5 -> 5.9 us for 116 rows on 368 x 1280, 256 x 256 x 256 6.8 -> 5.4 us): the family the automatic choice runs in their place.
static int small_or(int algo, int64_t M, int64_t N, int64_t K, int64_t group, const void* scales, const void* zeros) {
  if (algo == TLQ_ALGO_SKINNY ? M <= 16 || w4a16_skinny_forced() : algo != TLQ_ALGO_MFMA || N % 4 != 0 || w4a16_tile_forced()) return algo;
  const SmallTile p = w4a16_small_plan(M, N, K, group, scales, zeros, 0, 0, 0);
  const double theirs = algo == TLQ_ALGO_SKINNY ? 0.95 * (5.2 + 7.0 * giga((double)M, N, K) + 4.1 * giga(up16(M), N, K) + 0.3e-3 * (double)K)
                                                : 0.95 * fused_tile_us(M, N, K);
  return p.ok && (algo == TLQ_ALGO_SKINNY ? p.us : small_us(p, M, N, K)) < theirs ? TLQ_ALGO_SMALL : algo;
}
static bool decode_preferred(int64_t M, int64_t N, int64_t K) { return M > 2 || (M == 2 && N * K >= ((int64_t)1 << 24)); }

// The kernel of tlq_gemm_w4a16 by its rules (up to 64 rows; more rows come here only where every kernel above wants a workspace).
static bool w4a16_decode_in_one_chunk(const DecodePlan& dp, const void* scales, const void* zeros) {
  return dp.ok && dp.chunks == 1 && (((uintptr_t)scales | (uintptr_t)zeros) & 3) == 0;
}
static int w4a16_few_rows_choice(int64_t M, int64_t N, int64_t K, int64_t group, int in_dtype, const void* scales, const void* zeros, bool decode_ok) {
  // The skinny kernel takes the same time for every M up to 16 (the weights bound it); the GEMV kernels grow with
  // M.  Measured crossovers: fp16 GEMV wins at M = 1, and at M = 2 while K <= 4096; the bf16 GEMV dequantises
  // element by element and wins only at M = 1 in its register-resident form (rows of up to 16384 values: level with the
  // skinny kernel on 4096 weight rows, 15 against 25 us on 5120 rows of 13824 values).
  const bool skinny_ok = M <= 64 && K % 128 == 0 && fits32(M, K * 2) && fits32(N, K / 2);
  // two fp16 activation rows on many weight rows: the ring GEMV (8.9 against 10.3 us for the decode kernel at
  // 11008 x 4096, 5.2 against 6.2 us at 8192 x 2048; with 4096 rows, one per wavefront, the decode kernel is 5 % ahead)
  if (M == 2 && N >= 8192 && gemv_ring_applies(M, N, K, group, in_dtype, scales, zeros)) return TLQ_ALGO_GEMV;
  if (decode_preferred(M, N, K) && decode_ok && g_w4a16_decode) return TLQ_ALGO_DECODE;
  if (M > 4) return skinny_ok ? TLQ_ALGO_SKINNY : TLQ_ALGO_MFMA;
  if (!skinny_ok) return TLQ_ALGO_GEMV;
  if (in_dtype == TLQ_BF16) return (M == 1 && K <= 16384 && (group & (group - 1)) == 0) ? TLQ_ALGO_GEMV : TLQ_ALGO_SKINNY;
  return ((M == 1 && K <= 16384) || (M == 2 && K <= 4096)) ? TLQ_ALGO_GEMV : TLQ_ALGO_SKINNY;  // (longer rows: no register-resident GEMV)
}
// Do the last M % 4 of many rows, run by themselves, go to the fp16 GEMV kernels?  Those apply scale and zero point to fp32 sums of
// exact products, where every other kernel multiplies weights rounded to 16 bits: rows that have had that precision keep it.
static bool last_rows_take_f16_gemv(int64_t M, int64_t N, int64_t K, int64_t group, int in_dtype, const void* scales, const void* zeros) {
  const int64_t rows = M & 3;
  if (rows == 0 || in_dtype != TLQ_F16) return false;
  if (w4a16_choice_lookup(rows, N, K, group, in_dtype) == TLQ_ALGO_GEMV) return true;
  const DecodePlan dp = w4a16_decode_plan(rows, N, K, group, cu_count_or_default());
  return w4a16_few_rows_choice(rows, N, K, group, in_dtype, scales, zeros, w4a16_decode_in_one_chunk(dp, scales, zeros)) == TLQ_ALGO_GEMV;
}

int tlq_gemm_w4a16(const void* A, const void* w_packed, const void* scales, const void* zeros, void* C, int64_t M,
                   int64_t N, int64_t K, int64_t group, float zero_scalar, int in_dtype, int out_dtype, int algo,
                   void* stream) {
  TLQ_CHECK_DIMS("tlq_gemm_w4a16");
  TLQ_REQUIRE(in_dtype == TLQ_F16 || in_dtype == TLQ_BF16, "tlq_gemm_w4a16: in_dtype must be float16 or bfloat16 (got %d)",
              in_dtype);
  TLQ_REQUIRE(out_dtype == TLQ_F16 || out_dtype == TLQ_BF16 || out_dtype == TLQ_F32,
              "tlq_gemm_w4a16: out_dtype must be float16, bfloat16 or float32 (got %d)", out_dtype);
  TLQ_REQUIRE((algo >= TLQ_ALGO_AUTO && algo <= TLQ_ALGO_SKINNY) || algo == TLQ_ALGO_DECODE || algo == TLQ_ALGO_SMALL, "tlq_gemm_w4a16: bad algo %d", algo);
  if (M == 0 || N == 0) return 0;
  if (algo == TLQ_ALGO_AUTO) {
    // a tuned choice for this call signature (tlq_w4a16_choice_set) goes first; where that kernel refuses the call (its
    // shape or alignment rules: nothing launched), the rules below decide as if there were none
    const int chosen = w4a16_choice_lookup(M, N, K, group, in_dtype);
    if ((chosen >= TLQ_ALGO_GEMV && chosen <= TLQ_ALGO_SKINNY) || chosen == TLQ_ALGO_DECODE || chosen == TLQ_ALGO_SMALL) {
      const uint64_t before = launch_count();
      const int rc = tlq_gemm_w4a16(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, chosen, stream);
      if (rc == 0 || launch_count() != before) return rc;
      set_error("%s", "");
    }
  }
  // More than 64 rows: the choice of the entry point with a workspace, called without one -- the streaming and panel kernels
  // need none where they do not cut K (4096 x 4096 x 4096 bf16: 105 us in the 256-row panel kernel against 146 us in the
  // tile kernel below, which is where that call comes back to whenever a kernel would need the workspace).
  static thread_local bool choosing_without_workspace = false;
  if (algo == TLQ_ALGO_AUTO && M > 64 && !choosing_without_workspace) {
    choosing_without_workspace = true;
    const int rc = tlq_gemm_w4a16_ws(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_ALGO_AUTO, nullptr, 0, stream);
    choosing_without_workspace = false;
    return rc;
  }
  TLQ_REQUIRE(K > 0 && K % 64 == 0, "tlq_gemm_w4a16: K=%lld must be a positive multiple of 64", (long long)K);
  TLQ_REQUIRE(group > 0 && K % group == 0 && group % 32 == 0,
              "tlq_gemm_w4a16: group=%lld must divide K=%lld and be a multiple of 32", (long long)group, (long long)K);
  TLQ_REQUIRE(A && w_packed && C, "tlq_gemm_w4a16: null pointer");
  TLQ_REQUIRE(aligned16(A) && aligned16(w_packed) && aligned16(C), "tlq_gemm_w4a16: A, w_packed and C must be 16-byte aligned");
  TLQ_REQUIRE(((uintptr_t)scales & 1) == 0 && ((uintptr_t)zeros & 1) == 0, "tlq_gemm_w4a16: scales / zeros misaligned");
  hipStream_t st = (hipStream_t)stream;
  // The decode kernel (M <= 32): without a workspace only rows of up to 4096 values (one chunk of K).  Its scale / zero
  // gathers read aligned dwords: the tensors must start on a dword boundary (their length is checked by the plan).
  const DecodePlan dp = M <= 32 ? w4a16_decode_plan(M, N, K, group, cu_count_or_default()) : DecodePlan{false, 0, 0, 0, 0, 0};
  const bool decode_ok = w4a16_decode_in_one_chunk(dp, scales, zeros);
  if (algo == TLQ_ALGO_AUTO) algo = small_or(w4a16_few_rows_choice(M, N, K, group, in_dtype, scales, zeros, decode_ok), M, N, K, group, scales, zeros);
  if (algo == TLQ_ALGO_SMALL) {
    const SmallTile p = w4a16_small_plan(M, N, K, group, scales, zeros, 0, 0, 0);
    TLQ_REQUIRE(p.ok, TLQ_SMALL_NEEDS("tlq_gemm_w4a16"), (long long)M, (long long)N, (long long)K, (long long)group);
    return gemm_w4a16_small(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_W_PLAIN, p, "tlq_gemm_w4a16(small)", st);
  }
  if (algo == TLQ_ALGO_DECODE) {
    TLQ_REQUIRE(decode_ok, "tlq_gemm_w4a16: the decode kernel needs 1 <= M <= 32, K %% 256 == 0, K <= 4096 without a workspace, a power-of-two "
                "group and dword-aligned scale / zero tensors (M=%lld N=%lld K=%lld group=%lld)", (long long)M, (long long)N, (long long)K,
                (long long)group);
    return gemm_w4a16_decode(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_W_PLAIN, dp, nullptr, st);
  }
  if (algo == TLQ_ALGO_SKINNY) {
    TLQ_REQUIRE(M <= 64, "tlq_gemm_w4a16: the skinny kernel handles M <= 64 (got %lld)", (long long)M);
    TLQ_REQUIRE(K % 128 == 0, "tlq_gemm_w4a16: the skinny kernel needs K %% 128 == 0 (got %lld)", (long long)K);
    TLQ_REQUIRE(fits32(M, K * 2) && fits32(N, K / 2), "tlq_gemm_w4a16: a matrix spans 4 GiB or more");
    return gemm_w4a16_skinny(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, st);
  }
  if (algo == TLQ_ALGO_GEMV) {
    TLQ_REQUIRE(M <= 16, "tlq_gemm_w4a16: the GEMV kernel handles M <= 16 (got %lld)", (long long)M);
    return gemv_w4a16(A, w_packed, scales, zeros, C, 1, M, N, K, group, zero_scalar, in_dtype, out_dtype, st);
  }
  TLQ_REQUIRE(N % 4 == 0, "tlq_gemm_w4a16: the MFMA kernel needs N %% 4 == 0 (got %lld)", (long long)N);
  TLQ_REQUIRE(fits32(M, K * 2) && fits32(N, K / 2), "tlq_gemm_w4a16: a matrix spans 4 GiB or more");
  return gemm_w4a16_mfma(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, st);
}

// M from which dequantising the whole matrix once and running the plain GEMM on it beats converting the
// weights again in every row block of the fused kernel (measured on the MLP shapes: level at M = 256 for
// N = 14336, K = 4096 and 20-40 % ahead from there on and for N = 4096, K = 14336)
static const int64_t kTwoPassMinM = 256;

// most K slices the streaming kernel cuts for any group size (the smallest group allows the shortest slices).  least: those of the plan of short windows where it cuts
// fewer, since a call whose workspace does not hold the best plan's runs by it (stream_plan_for), or where the best one does not cut at all: a size that no kernel
// asks for would be that of the two passes then, and keep callers with less from the scratch that the rows' own scales want
static int64_t stream_max_split(int64_t M, int64_t N, int64_t K, bool least = false) {
  int64_t most = 0;
  for (int64_t group = 32; group <= K; group *= 2) {
    if (K % group) continue;
    const StreamPlan p = w4a16_stream_plan(M, N, K, group, cu_count_or_default());  // (the count the launch plans with)
    int64_t split = p.ok ? p.split : 0;
    if (least && p.ok)
      if (const StreamPlan other = w4a16_stream_plan(M, N, K, group, cu_count_or_default(), true); other.ok && (other.split < split || split == 1)) split = other.split;
    if (split > most) most = split;
  }
  return most;
}
// What tlq_w4a16_workspace_bytes counts in its place up to 512 rows: no fewer slices than fill the CUs with blocks of 256 weight rows.  No plan
// launches those (64 x 4096 x 14336: 16, its plans cut 8 at most); the size of such a call is part of what callers are promised,
// so it stays.  The least size and the size by name count the plans' own.
static int64_t stream_promised_split(int64_t M, int64_t N, int64_t K) {
  const int64_t most = stream_max_split(M, N, K);
  if (most == 0 || K < 1024) return most;
  const int64_t blocks = ceil_div(N, (int64_t)256) * ceil_div(M, (int64_t)(M > 64 ? 128 : (M > 32 ? 64 : 32)));
  int64_t fill = cu_count_or_default() / blocks;
  if (fill > 16) fill = 16;
  if (fill > K / 128 / 4) fill = K / 128 / 4;
  return fill > most ? fill : most;
}

// Second of the two passes: the plain GEMM on the dequantised matrix at the head of the workspace.  What the workspace
// holds beyond that matrix is room for fp32 matrices of K slices (few output tiles: tlq_gemm_f16_ws).
static int plain_gemm_on_workspace(const void* A, void* workspace, int64_t workspace_bytes, void* C, int64_t M, int64_t N,
                                   int64_t K, int in_dtype, int out_dtype, void* stream) {
  const int64_t head = (N * K * 2 + 15) / 16 * 16;
  return tlq_gemm_f16_ws(A, workspace, C, (uint8_t*)workspace + head, workspace_bytes - head, 1, M, N, K, in_dtype, out_dtype,
                         TLQ_B_NK, stream);
}

// fp32 partial sums of the K slices of the kernels for small and middle M (sized for the smallest group, which allows the
// most slices); 0 when none of them cuts K
static int64_t w4a16_partial_sum_bytes(int64_t M, int64_t N, int64_t K, bool least = false) {
  int64_t split = w4a16_mid_split(M, N, K, 32);
  const int64_t ssplit = M > 512 ? 0 : (least ? stream_max_split(M, N, K, true) : stream_promised_split(M, N, K));
  if (ssplit > split) split = ssplit;
  if (M <= 32) {  // the decode kernel cuts rows longer than 4096 values into chunks
    const DecodePlan dp = w4a16_decode_plan(M, N, K, 32, cu_count_or_default());
    if (dp.ok && dp.chunks > split) split = dp.chunks;
  }
  return split > 1 ? split * M * N * 4 : 0;
}

// The four-wavefront panel kernels take any row count: rows past the matrix repeat its last.  Asked for by name they take multiples of four, as they
// always did, and above 512 rows the automatic choice calls them for those (with_rows_behind); up to 512 rows it plans for the next one.
static int64_t whole_fours(int64_t M) { return (M + 3) & ~(int64_t)3; }

// what the panel kernel may ask of the workspace for any group size: the partial tiles of its K slices and the flag word
static int64_t panel_workspace_bytes(int64_t M, int64_t N, int64_t K, bool any_rows = false) {
  if (!(M >= 1 && N >= 1 && K > 0 && M < kMaxDim && N < kMaxDim && K < kMaxDim)) return 0;
  int64_t need = 0;
  for (int64_t group = 32; group <= 1024; group *= 2) {
    if (K % group != 0) continue;
    const PanelPlan pp = w4a16_panel_plan(M, N, K, group, cu_count_or_default());
    if (pp.ok) {
      const int64_t b = (pp.split > 1 ? (int64_t)pp.split * M * N * 4 : 0) + 16;
      if (b > need) need = b;
    }
    const Panel2Plan p2 = w4a16_panel256_plan(any_rows ? whole_fours(M) : M, N, K, group, cu_count_or_default());
    if (p2.ok) {
      const int64_t b = (p2.split > 1 ? (int64_t)p2.split * M * N * 4 : 0) + (M % 4 == 0 ? 16 : 0);  // (the word is the 128-row kernel's)
      if (b > need) need = b;
    }
  }
  return need;
}

// the same for the middle-M panel kernel
static int64_t panelm_workspace_bytes(int64_t M, int64_t N, int64_t K, bool any_rows = false) {
  if (!(M >= 1 && N >= 1 && K > 0 && M < kMaxDim && N < kMaxDim && K < kMaxDim)) return 0;
  int64_t need = 0;
  for (int64_t group = 32; group <= 1024; group *= 2) {
    if (K % group != 0) continue;
    const PanelMPlan pm = w4a16_panelm_plan(any_rows ? whole_fours(M) : M, N, K, group, cu_count_or_default());
    if (pm.ok && pm.split > 1 && (int64_t)pm.split * M * N * 4 > need) need = (int64_t)pm.split * M * N * 4;
  }
  return need;
}

// The automatic choice takes the middle-M panel kernel from 257 to 512 activation rows on matrices of 2^25 weights or more
// (measured against the streaming kernel on five (N, K) pairs, groups of 128 and 64, fp16 with a zero-point tensor:
// 14336 x 4096 and 4096 x 14336: 43.5 - 43.9 against 45.8 - 47.0 us at 256 rows, 56 - 59 against 65 - 71 us at 384, 62 - 76 against
// 70 - 80 us at 512; 8192 x 8192: 47 / 66 / 77 against 49 / 74 / 82 us; below 256 rows and on 4096 x 4096 or 5120 x 5120 the
// streaming kernel is level or ahead by up to 15 %).  From 196 to 256 rows (two tiles of 128 rows, the second more than half
// full) the matrix has to be larger: 44 million weights with 10240 outputs or more, 56 million with fewer (10240 x 4096 at
// 196 - 252 rows: 36 - 41 us for the streaming kernel against 40 - 43 us; at 256 rows the streaming kernel takes
// 36 - 41 against 41 - 45 us on 6144 x 6144, 5120 x 8192 and 8192 x 5120 and 44 - 48 against 46 - 51 us on 7168 x 7168; at
// 200 - 248 rows the middle-M kernel takes 112 - 125 against 130 - 145 us on 28672 x 8192, 59 - 67 against 67 - 79 us on
// 28672 x 4096 and is 2 - 7 % ahead on 11008 x 4096, 12288 x 4096, 14336 x 4096, 4096 x 14336 and 8192 x 8192).
static bool panelm_preferred(int64_t M, int64_t N, int64_t K) {
  if (M < 196 || M > 512 || N * K < ((int64_t)1 << 25)) return false;
  return M > 256 || N * K >= (N >= 10240 ? 44000000 : 56000000);
}

// One tile of 128 rows (97 .. 128 activation rows) on matrices of 2^27 weights or more: the middle-M kernel is 9 - 18 % ahead of
// the streaming kernel (N = 50304, K = 4096, M = 128: 64.5 against 76.1 us; N = 65536, K = 8192: 144 against 154 us;
// N = 28672, K = 8192, M = 112: 74 against 82 us; N = 8192, K = 28672: 76 against 81 us; level at 64 and 96 rows).
static bool panelm_one_tile(int64_t M, int64_t N, int64_t K) { return M > 96 && M <= 128 && N * K >= ((int64_t)1 << 27); }

// 65 .. 128 rows on output-layer widths: the 128-row panel kernel, whose work-groups own 512 weight rows, where they fill more
// than five eighths of the machine in ONE round -- the streaming kernel's work-groups (256 weight rows) then need two, the second
// one partly empty (N = 102400, K = 4096, M = 96: 106 against 124 us; K = 5120: 133 against 159 us; N = 128256, K = 4096: 123
// against 136 us; N = 81920: 100 against 111 us).  Not with longer rows (N = 81920, K = 8192: 208 against 204 us).
static bool panel_one_round(int64_t M, int64_t N, int64_t K) {
  const int64_t cus_now = cu_count_or_default();
  const int64_t tiles = ceil_div(N, (int64_t)512);
  return M > 64 && M <= 128 && K <= 5120 && tiles <= cus_now && tiles * 8 >= cus_now * 5;
}

// What an explicitly named kernel family may ask of the workspace for any group size.
int64_t tlq_w4a16_workspace_bytes_for(int64_t M, int64_t N, int64_t K, int algo) {
  if (M <= 0 || N <= 0 || K <= 0 || M >= kMaxDim || N >= kMaxDim || K >= kMaxDim) return 0;
  switch (algo) {
    case TLQ_ALGO_AUTO: return tlq_w4a16_workspace_bytes(M, N, K);
    case TLQ_ALGO_TWO_PASS: return (N * K * 2 + 15) / 16 * 16 + tlq_f16_workspace_bytes(1, M, N, K);
    case TLQ_ALGO_STREAM: {
      const int64_t split = M <= 512 ? stream_max_split(M, N, K) : 0;
      return split > 1 ? split * M * N * 4 : 0;
    }
    case TLQ_ALGO_DECODE: {
      if (M > 32) return 0;
      const DecodePlan dp = w4a16_decode_plan(M, N, K, 32, cu_count_or_default());
      return dp.ok && dp.chunks > 1 ? (int64_t)dp.chunks * M * N * 4 : 0;
    }
    case TLQ_ALGO_MFMA: {  // with a workspace the tile kernel runs over K slices where it has few output tiles
      const int64_t split = w4a16_mid_split(M, N, K, 32);
      return split > 1 ? split * M * N * 4 : 0;
    }
    case TLQ_ALGO_PANEL:
    case TLQ_ALGO_PANEL256: return panel_workspace_bytes(M, N, K);
    case TLQ_ALGO_PANELM: return panelm_workspace_bytes(M, N, K);
    default: return 0;  // GEMV, skinny, small tiles: no workspace
  }
}

static int64_t w4a16_kernel_workspace_bytes(int64_t M, int64_t N, int64_t K);
static int64_t w4a16_workspace_bytes_now(int64_t M, int64_t N, int64_t K);
int64_t tlq_w4a16_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (N <= 0 || K <= 0) return 0;
  static thread_local PlanTable<int64_t> known;
  return known.get(M, N, K, 0, [&] { return w4a16_workspace_bytes_now(M, N, K); });
}
static int64_t w4a16_workspace_bytes_now(int64_t M, int64_t N, int64_t K) {
  int64_t need = w4a16_kernel_workspace_bytes(M, N, K);
  // (a weight-row count that is no multiple of four: what the multiple of 16 below asks for, then its packed result, sized for fp32)
  if (ragged_rows_apply(M, N)) need = ragged_head(N) == 0 ? 0 : (w4a16_kernel_workspace_bytes(M, ragged_head(N), K) + 15) / 16 * 16 + ragged_result_bytes(M, N, 4);
  // (rows whose length is no power of two with one group per row: room behind everything else for the scales and zero points
  // written out per power-of-two group)
  if ((K & (K - 1)) != 0 && K % 64 == 0) return (need + 15) / 16 * 16 + 2 * row_group_tensor_bytes(N, K) + 16;
  return need;
}
// what the kernels themselves may ask for
static int64_t w4a16_kernel_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  int64_t need = w4a16_partial_sum_bytes(M, N, K);
  // (above 512 rows a row count that is no multiple of four runs as the multiple below plus a tail: room for that call)
  if (M > 512 && (M & 3) != 0) {
    const int64_t head = w4a16_kernel_workspace_bytes(M & ~(int64_t)3, N, K);
    if (head > need) need = head;
  }
  // tuned choices for this shape (any group, any type): room for the chosen family as well
  int64_t tuned[4] = {0, M, N, K};
  w4a16_choice_for_shape(M, N, K, [](int algo, void* ctx) {
    int64_t* const n = (int64_t*)ctx;
    if (algo == TLQ_ALGO_AUTO) return;
    const int64_t b = tlq_w4a16_workspace_bytes_for(n[1], n[2], n[3], algo);
    if (b > n[0]) n[0] = b;
  }, tuned);
  if (tuned[0] > need) need = tuned[0];
  if (M > 512 && M <= kStreamMaxRows) {  // partial sums of the streaming kernel, where it is the choice for some group size
    for (int64_t group = 32; group <= K && K % group == 0; group *= 2) {
      if (!stream_beats_panels(M, N, K, group, true)) continue;
      const StreamPlan sp = w4a16_stream_plan(M, N, K, group, cu_count_or_default());
      if (sp.split > 1 && (int64_t)sp.split * M * N * 4 > need) need = (int64_t)sp.split * M * N * 4;
    }
  }
  if (panelm_preferred(M, N, K) || panelm_one_tile(M, N, K) || M > 512 || (M >= 196 && N * K >= ((int64_t)1 << 25))) {  // (above 512 rows: where its estimate beats the 256-row kernel's)
    const int64_t pm = panelm_workspace_bytes(M, N, K, M <= 512);
    if (pm > need) need = pm;
  }
  if (M > 128 || panelm_preferred(M, N, K) || panel_one_round(M, N, K)) {  // (129 .. 512 rows: where the 256-row kernel's estimate beats the middle-M or the streaming kernel's)
    const int64_t pn = panel_workspace_bytes(M, N, K, M <= 512);
    if (pn > need) need = pn;
  }
  // two passes (which of the two is taken depends on the group size, so the size covers both): the dequantised matrix,
  // then room for the K slices of the plain GEMM where it has few output tiles
  if (M >= kTwoPassMinM) {
    const int64_t two = (N * K * 2 + 15) / 16 * 16 + tlq_f16_workspace_bytes(1, M, N, K);
    if (two > need) need = two;
  }
  return need;
}

int64_t tlq_w4a16_workspace_bytes_min(int64_t M, int64_t N, int64_t K) {
  if (N <= 0 || K <= 0) return 0;
  const int64_t partial = w4a16_partial_sum_bytes(M, N, K, true);
  if (partial > 0) return partial;
  return M >= kTwoPassMinM ? N * K * 2 : 0;
}

// Estimated time of a panel kernel's launch (us): rounds of work-groups x (steps per K slice x step time + fixed part), plus
// the pass that adds the slices' partial tiles (a launch, their write and their read) where K is cut.
static double panel_estimate_us(int tiles_m, int tiles_n, int split, int slice_steps, double step_us, double fixed_us, int64_t M,
                                int64_t N, int64_t cus) {
  const int64_t wgs = (int64_t)tiles_m * tiles_n * split;
  const double rounds = (double)ceil_div(wgs, cus);
  return rounds * ((double)slice_steps * step_us + fixed_us) + (split > 1 ? 3.0 + (double)(split + 1) * (double)M * (double)N * 4.0 / 4e6 : 0.0);
}
// Above 512 rows: does the middle-M kernel (128-row tiles) beat the 256-row kernel by estimate?
static bool panelm_estimate_wins(int64_t M, int64_t N, int64_t K, int64_t group) {
  const int64_t cus_now = cu_count_or_default();
  const PanelMPlan pm = w4a16_panelm_plan(M, N, K, group, (int)cus_now);
  const Panel2Plan p2 = w4a16_panel256_plan(M, N, K, group, (int)cus_now);
  if (!pm.ok || !p2.ok || pm.tm != 8) return false;
  const double est_m = panel_estimate_us(pm.tiles_m, pm.tiles_n, pm.split, pm.slice_steps, 2.2, 6.0, M, N, cus_now);
  const double est_2 = panel_estimate_us(p2.tiles_m, p2.tiles_n, p2.split, p2.slice_steps, 3.3, 8.0, M, N, cus_now);
  return est_m < 0.94 * est_2;
}
// 256 .. 512 rows: does the 256-row kernel beat the middle-M kernel by the same estimate?
static bool panel256_estimate_wins(int64_t M, int64_t N, int64_t K, int64_t group) {
  const int64_t cus_now = cu_count_or_default();
  const PanelMPlan pm = w4a16_panelm_plan(whole_fours(M), N, K, group, (int)cus_now);
  const Panel2Plan p2 = w4a16_panel256_plan(whole_fours(M), N, K, group, (int)cus_now);
  if (!pm.ok || !p2.ok) return false;
  const double est_m = panel_estimate_us(pm.tiles_m, pm.tiles_n, pm.split, pm.slice_steps, pm.tm == 8 ? 2.2 : 1.8, 6.0, M, N, cus_now);
  const double est_2 = panel_estimate_us(p2.tiles_m, p2.tiles_n, p2.split, p2.slice_steps, 3.3, 8.0, M, N, cus_now);
  return est_2 < 0.9 * est_m;
}

// 256 rows on 2^25 weights and more that panelm_preferred leaves to the streaming kernel: the middle-M kernel in binary16 where full
// tiles make whole rounds of its work-groups and its estimate (14 % high there, hence 0.87) is no more than 2 % above the streaming kernel's.
// About level with what the streaming kernel took before its groups of wavefronts (256 x 8192 x 4096 31.7 against 30.9 us, 256 x 8192 x
// 6144 39.3 against 40.8), which is why the test of this choice names it; the streaming kernel's estimate is 10 - 15 % high there and it would
// take 26.0 and 36.9.  With partly filled tiles, longer slices or bfloat16 the same rounds are further behind (232 x 8192 x 6656 45.3
// against 43.5, 256 x 8192 x 4096 bf16 31.6 against 30.0): there the streaming kernel runs (38.8 and 27.2).
static bool panelm_whole_rounds(int64_t M, int64_t N, int64_t K, int64_t group, int in_dtype) {
  if (M != 256 || N % 256 != 0 || N * K < ((int64_t)1 << 25) || group <= 0 || in_dtype != TLQ_F16) return false;
  const int64_t cus_now = cu_count_or_default();
  const PanelMPlan pm = w4a16_panelm_plan(M, N, K, group, (int)cus_now);
  if (!pm.ok || pm.tm != 8 || ((int64_t)pm.tiles_m * pm.tiles_n * pm.split) % cus_now != 0) return false;
  const StreamPlan sp = w4a16_stream_plan(M, N, K, group, (int)cus_now);
  return !sp.ok || 0.87 * panel_estimate_us(pm.tiles_m, pm.tiles_n, pm.split, pm.slice_steps, 2.2, 6.0, M, N, cus_now) < 1.02 * sp.us;
}

// 129 .. 512 rows: does the 256-row kernel beat the streaming kernel?  By the estimates of both, the panel kernel's at 0.94 (it is 15 % high, the streaming kernel's 2 %):
// 0.2 % behind the faster of the two on average on 370 problems (matrices of 2^25 - 3e8 weights, groups of 64 and 128, both types).  Between 0.97 and 1.06, and
// on matrices beyond those, row counts that are no multiple of four stay with the streaming kernel, the others go by its older price, rounds x (2.2 us a step of
// 128 rows, 1.75 of 96, + 8) for blocks of 256 weight rows (by that price alone 0.6 % behind: 468 x 16768 x 12288 291 -> 241 us, 288 x 26448 x 9216 227 -> 198).
// 423 x 27904 x 6528 in groups of 32 238 -> 176, 459 x 27136 x 4736 151 -> 127.
static bool panel256_beats_stream(int64_t M, int64_t N, int64_t K, int64_t group, const StreamPlan& sp) {
  if (M <= 128 || !sp.ok || (sp.tm != 8 && sp.tm != 6)) return false;
  static thread_local PlanTable<bool> known;
  return known.get(M, N, K, group, [&] {
    const int64_t cus_now = cu_count_or_default();
    const Panel2Plan p2 = w4a16_panel256_plan(whole_fours(M), N, K, group, (int)cus_now);
    if (!p2.ok) return false;
    const double est_2 = panel_estimate_us(p2.tiles_m, p2.tiles_n, p2.split, p2.slice_steps, 3.3, 8.0, M, N, cus_now);
    if (0.94 * est_2 < 0.97 * sp.us) return true;
    if (M % 4 != 0 || (0.94 * est_2 > 1.06 * sp.us && N * K <= 300000000 && N <= 32768)) return false;
    if (sp.kg == 4) return 0.9 * est_2 < sp.us;
    return est_2 < 0.95 * panel_estimate_us(sp.m_blocks, sp.n_blocks, sp.split, sp.slice_steps, sp.tm == 8 ? 2.2 : 1.75, 8.0, M, N, cus_now);
  });
}

// Where panelm_preferred speaks for the middle-M and the 256-row kernel: does the streaming kernel beat both?  By the estimates, the middle-M kernel's at 0.86 (it is
// 26 % high) and with the same distances: of 30 such problems 14 were 3 % and more behind without this question (288 x 5376 x 13312 71.2 against 54.1 us, 308 x 14720 x
// 4096 56.7 against 50.8).  Up to 256 binary16 rows, a multiple of four, the middle-M kernel stays (the test of the choice names it: 256 x 14336 x 4096 43.7 against
// 36.4 us).
static bool stream_beats_middle(int64_t M, int64_t N, int64_t K, int64_t group, int in_dtype, const StreamPlan& sp) {
  if (!sp.ok || !g_w4a16_stream || (M <= 256 && M % 4 == 0 && in_dtype == TLQ_F16)) return false;
  static thread_local PlanTable<bool> known;
  return known.get(M, N, K, group, [&] {
    const int64_t cus_now = cu_count_or_default();
    const double bar = (M % 4 == 0 ? 1.06 : 0.97) * sp.us;
    const PanelMPlan pm = w4a16_panelm_plan(whole_fours(M), N, K, group, (int)cus_now);
    const Panel2Plan p2 = w4a16_panel256_plan(whole_fours(M), N, K, group, (int)cus_now);
    if (pm.ok && 0.86 * panel_estimate_us(pm.tiles_m, pm.tiles_n, pm.split, pm.slice_steps, pm.tm == 8 ? 2.2 : 1.8, 6.0, M, N, cus_now) < bar) return false;
    return !(p2.ok && 0.94 * panel_estimate_us(p2.tiles_m, p2.tiles_n, p2.split, p2.slice_steps, 3.3, 8.0, M, N, cus_now) < bar);
  });
}

// The automatic choice takes the 256-row panel kernel where the last round of its work-groups fills more than half of the CUs
// (measured: 2 - 21 % behind the two passes at 0.375 -- 96 work-groups --, 3 % behind at exactly one half, ahead from there on:
// N = 11008, K = 4096, M = 768, 129 work-groups: 92 against 107 us).
static const double kPanel256Fill = 0.502;
static bool panel256_fills(int64_t M, int64_t N, int64_t K, int64_t group) {
  const int64_t cus_now = cu_count_or_default();
  const Panel2Plan pp = w4a16_panel256_plan(M, N, K, group, (int)cus_now);
  if (!pp.ok) return false;
  const int64_t wgs = (int64_t)pp.tiles_m * pp.tiles_n * pp.split;
  return (double)wgs / (double)(ceil_div(wgs, cus_now) * cus_now) >= kPanel256Fill;
}

// Above 512 rows: do the two passes beat what the panel kernels would run?  The dequantisation pass costs 3 us and the weights' bytes, the
// plain GEMM behind it runs large products at 1.4 - 1.5 PFLOP/s where the 256-row panel kernel reaches 1.2 - 1.3 (8192 x 14336 x 4096 fp16 in groups of
// 64 774 -> 684 us), has smaller tiles, and takes any row count, while the panel kernels have 8 us per round of
// work-groups (many rounds of short rows: 4868 x 3152 x 384 bf16 36.9 -> 25.5 us, 6631 x 4608 x 256 38.7 -> 29.8) and leave
// one to three rows to a launch of their own (639 x 5680 x 896 29.2 -> 22.6 us, 7671 x 512 x 3200 49.0 -> 35.9).  With the plain GEMM's tiles between
// 128 x 128 and 256 x 256 the two passes are ahead of the 256-row kernel on all but 17 of 163 random problems that either takes (M 513 .. 8192, N 256 ..
// 14336, K 256 .. 14336, groups of 64 and 128, both types): those of fewer than 1024 rows and more than 2000 values, and a few of one partial round.
// The 256-row kernel's time against its estimate / 1.21, or 1.38 PFLOP/s: 1.05 (8 % rms) on 420 random problems and 1.07 on 264 of round sizes (M 768 .. 8192, N 1024 .. 14336), 7 % less
// of it without a tensor of zero points where K is long; that of the two passes 1.0 (7 %).  With the bars below the choice is 0.5 % behind the faster of the two on either set
// (4096^3 bf16, scalar zero point, 101.7 - 104.9 us here, 104.3 - 107.9 in the two passes; with a tensor 111.6 and 103.2).  (The middle-M kernel's bars are those that the tests of the choice ask for, 1003 x 2048 x 4096 in groups of 64
// 35 us in a launch for 1000 rows and one for three, 29 in the two passes.)  Where neither panel kernel would run, all rows go through the two passes and none is left over.
static double plain_nk_us(int64_t M, int64_t N, int64_t K);
static bool tiles_beat_slices(TileKind tile, int kind, int64_t M, int64_t N, int64_t K, int64_t k_bytes);
// (fitted to 1900 calls of 6 - 100 us, 7 % rms: right behind the dequantisation the ring kernel takes 19 % more than on its own, the kernels of larger tiles do not.
// Without that the passes looked 12 % too fast and took calls from the streaming and the small-tile kernel: 564 x 3328 x 1280 19.9 for 12.9 us, 801 x 384 x 2176
// 13.9 for 9.6)
static double two_passes_us(int64_t M, int64_t N, int64_t K) {
  if (f16_split_choice(1, M, N, K) > 1 && !tiles_beat_slices(kTileF16NK, 2, M, N, K, K * 2)) return 2.6 + (double)N * (double)K * 2.5 / 4.8e6 + plain_nk_us(M, N, K);
  const TileChoice c = tile_choice(kTileF16NK, 1, M, N, K * 2);
  const bool ring = c.variant >= kGroup128x128 && c.variant <= kGroup64x64;
  return ring ? 2.7 + 0.31e-6 * (double)N * (double)K + 1.19 * c.us : 4.6 + 0.645e-6 * (double)N * (double)K + 0.93 * c.us;
}
static bool two_passes_beat_panels(int64_t M, int64_t N, int64_t K, int64_t group, bool rest_goes_along, bool zero_points) {
  static thread_local PlanTable<bool> known;
  return known.get(M, N, K, group * 4 + rest_goes_along * 2 + zero_points, [&] {
    const int64_t cus_now = cu_count_or_default(), head = M & ~(int64_t)3;
    const PanelMPlan pm = w4a16_panelm_plan(head, N, K, group, (int)cus_now);
    const Panel2Plan p2 = w4a16_panel256_plan(head, N, K, group, (int)cus_now);
    if (!p2.ok || N % 8 != 0) return false;
    double panels;
    const bool middle = pm.ok && panelm_estimate_wins(head, N, K, group);
    if (middle)
      panels = panel_estimate_us(pm.tiles_m, pm.tiles_n, pm.split, pm.slice_steps, 2.2, 6.0, head, N, cus_now);
    else if (panel256_fills(head, N, K, group))
      panels = panel_estimate_us(p2.tiles_m, p2.tiles_n, p2.split, p2.slice_steps, 3.3, 8.0, head, N, cus_now);
    else
      return true;
    const double best = 2.0 * (double)M * (double)N * (double)K / 1.38e9;  // at 1.38 PFLOP/s
    panels = panels / 1.21 > best ? panels / 1.21 : best;
    // (rows that go along cost no launch.  Above 2048 rows they are counted as one all the same: the panels' estimate is low there, 6 problems of 10 that not counting
    // it moves are 1 - 13 % slower; up to 2048 rows 10 of 11 are faster, 1.01 - 1.18 x, 518 x 7440 x 1024 24.5 -> 16.4 us)
    const bool rest = head != M && !(rest_goes_along && M <= 2048 && ceil_div(head, (int64_t)(middle ? 128 : 256)) == ceil_div(M, (int64_t)(middle ? 128 : 256)));
    const double two = two_passes_us(M, N, K), with_rest = panels + (rest ? 4.5 : 0.0);
    return middle ? two < (rest ? 0.9 : 1.0) * with_rest : two < (M <= 1024 ? 1.05 : zero_points || K <= 512 ? 1.13 : 1.08) * with_rest;
  });
}
static bool room_for_two_passes(int64_t N, int64_t K, const void* workspace, int64_t workspace_bytes) {
  return N > 0 && K > 0 && N < kMaxDim && K < kMaxDim && workspace != nullptr && workspace_bytes >= N * K * 2 && aligned16(workspace);
}
// Many rows on up to 2^19 weights: the two passes or the tile kernel in one launch (4907 x 256 x 2048 16.8 against 38.9 us).  By the estimate before this one, at 0.9, 13 of 27
// problems above 512 rows went to the two passes, 1.28 x on average, one of them 3 % behind; 112 calls between a bar of 0.9 and this one are 1.17 x faster in them.
static bool two_passes_beat_tiles(int64_t M, int64_t N, int64_t K) {
  static thread_local PlanTable<bool> known;
  return M > 512 && N % 8 == 0 && known.get(M, N, K, 0, [&] { return two_passes_us(M, N, K) < fused_tile_us(M, N, K); });
}

// Above 512 rows: does the streaming kernel beat the panel kernels (their estimates are 13 - 19 % high, see above; a row count that is no
// multiple of four costs them a launch) and the two passes?  On 300 random problems (M 513 .. 4096, up to 2e11 operations) where the rule
// alone decided, 1.13 x on average over what ran before (1.9 x at most: 663 x 4096 x 1792 34.1 -> 17.5 us), more than 5 % behind on 7;
// with the regions that the entry point leaves to the others 1.06 x.
static bool stream_beats_panels(int64_t M, int64_t N, int64_t K, int64_t group, bool two_passes) {
  static thread_local PlanTable<bool> known;
  return g_w4a16_stream && known.get(M, N, K, group * 2 + two_passes, [&] {
    const StreamPlan sp = w4a16_stream_plan(M, N, K, group, cu_count_or_default());
    if (!sp.ok) return false;
    const int64_t cus_now = cu_count_or_default(), head = M & ~(int64_t)3;
    const int64_t tiles = ceil_div(M, (int64_t)128) * ceil_div(N, (int64_t)128);
    // (without room for the two passes it is the tile kernel that would run: 1.05 x its estimate in one round of tiles, 1.2 - 1.3 x in two, 1.4 x beyond; by an
    // estimate of passes that cannot run 2308 x 1328 x 4224 took 80 us in the tile kernel for 44 here; 1138 random calls that either moves 1.22 x on average)
    double other = fused_tile_us(M, N, K) * (two_passes || (tiles <= cus_now && K <= 512) ? 1.0 : tiles <= cus_now ? 1.05 : tiles <= 2 * cus_now ? 1.25 : 1.4);
    if (two_passes && N % 8 == 0) other = 1.04 * two_passes_us(M, N, K);
    // (short rows in one round of 128 x 128 tiles: the tile kernel, 3388 x 384 x 384 8.5 against 9.9 us, 2816 x 1792 x 128 7.1 against 9.2, which its estimate is
    // some 10 % above)
    if (K <= 512 && tiles <= cus_now && 0.9 * fused_tile_us(M, N, K) < other) other = 0.9 * fused_tile_us(M, N, K);
    const PanelMPlan pm = w4a16_panelm_plan(head, N, K, group, (int)cus_now);
    const Panel2Plan p2 = w4a16_panel256_plan(head, N, K, group, (int)cus_now);
    double panels = 1e30;
    if (pm.ok && pm.tm == 8) panels = panel_estimate_us(pm.tiles_m, pm.tiles_n, pm.split, pm.slice_steps, 2.2, 6.0, head, N, cus_now);
    if (p2.ok) {
      const double us = panel_estimate_us(p2.tiles_m, p2.tiles_n, p2.split, p2.slice_steps, 3.3, 8.0, head, N, cus_now);
      if (us < panels) panels = us;
    }
    panels = 0.87 * panels + (head != M ? 5.5 : 0.0);
    return sp.us < (two_passes || K > 512 ? 0.98 : 0.95) * other && sp.us < 0.95 * panels;
  });
}
static bool stream_workspace_ok(const StreamPlan& sp, int64_t M, int64_t N, const void* workspace, int64_t workspace_bytes) {
  return sp.ok && (sp.split == 1 || (workspace && aligned16(workspace) && workspace_bytes >= (int64_t)sp.split * M * N * 4));
}
// By name: 512 rows at most.  Where the workspace does not hold the K slices of the best plan, the plan by short windows, which cuts fewer on some problems: its
// slices are what such calls were sized for before windows were longer (472 x 3040 x 4224 in groups of 64: two slices for three).
static StreamPlan stream_plan_for(int64_t M, int64_t N, int64_t K, int64_t group, int algo, const void* workspace, int64_t workspace_bytes) {
  if (!(M >= 1 && N >= 1 && K > 0 && group > 0 && M < kMaxDim && N < kMaxDim && K < kMaxDim)) return StreamPlan{};
  if (M > 512 && !(g_stream_tiles > 0 || (algo == TLQ_ALGO_AUTO && stream_beats_panels(M, N, K, group, room_for_two_passes(N, K, workspace, workspace_bytes))))) return StreamPlan{};
  const StreamPlan best = w4a16_stream_plan(M, N, K, group, cu_count_or_default());
  if (!best.ok || stream_workspace_ok(best, M, N, workspace, workspace_bytes)) return best;
  const StreamPlan other = w4a16_stream_plan(M, N, K, group, cu_count_or_default(), true);
  return stream_workspace_ok(other, M, N, workspace, workspace_bytes) ? other : best;
}
static bool stream_args_ok(const void* A, const void* w_packed, const void* scales, const void* zeros, const void* C, int64_t M, int64_t N, int64_t K, int in_dtype,
                           int out_dtype) {
  return A && w_packed && C && aligned16(A) && aligned16(w_packed) && aligned16(C) && (in_dtype == TLQ_F16 || in_dtype == TLQ_BF16) &&
         (out_dtype == TLQ_F16 || out_dtype == TLQ_BF16 || out_dtype == TLQ_F32) && (M * N) % 4 == 0 && ((uintptr_t)scales & 1) == 0 &&
         ((uintptr_t)zeros & 1) == 0 && K > 0 && fits32(M, K * 2) && fits32(N, K / 2);
}

// The one to three rows of the same matrices behind the M (a multiple of four) that the automatic choice is called for: the four-wavefront panel kernels and the streaming kernel take them along
// where they lie in the last of the tiles that M rows take anyway, and set this to zero once they are launched (not ahead of it: a tuned kernel that fails leaves them to the rules).  (One tile row more would cost a round where the head's tiles fill
// the machine: 4097 x 4096 x 4096 runs 4096 rows in one round and the last row by itself.)
static thread_local int64_t g_rows_behind = 0;
static int64_t with_rows_behind(int64_t M, int64_t tile) { return ceil_div(M, tile) == ceil_div(M + g_rows_behind, tile) ? M + g_rows_behind : M; }
static int rows_behind_done(int rc, bool along) {
  if (rc == 0 && along) g_rows_behind = 0;
  return rc;
}

// The panel kernel (large M, one launch, weights dequantised on the operand read).  Returns -1 when it does not take the
// problem (nothing launched, no error set), else the launch's return code.
static int try_panel(const void* A, const void* w_packed, const void* scales, const void* zeros, void* C, int64_t M, int64_t N,
                     int64_t K, int64_t group, float zero_scalar, int in_dtype, int out_dtype, int w_layout, void* workspace,
                     int64_t workspace_bytes, void* stream) {
  if (!(M >= 1 && N >= 1 && K > 0 && group > 0 && M < kMaxDim && N < kMaxDim && K < kMaxDim)) return -1;
  const PanelPlan pp = w4a16_panel_plan(M, N, K, group, cu_count_or_default());
  if (!pp.ok) return -1;
  const bool args_ok = A && w_packed && C && aligned16(A) && aligned16(w_packed) && aligned16(C) && aligned16(scales) &&
                       aligned16(zeros) && (in_dtype == TLQ_F16 || in_dtype == TLQ_BF16) &&
                       (out_dtype == TLQ_F16 || out_dtype == TLQ_BF16 || out_dtype == TLQ_F32) && (M * N) % 4 == 0 &&
                       fits32(M, K * 2) && fits32(N, K / 2) && fits32(N, (K / group) * 2);
  if (!args_ok) return -1;
  // workspace: the partial tiles of the K slices, then (with a zero-point tensor) one word for the kernel's flag
  const int64_t part_bytes = pp.split > 1 ? (int64_t)pp.split * M * N * 4 : 0;
  const int64_t need = part_bytes + (zeros ? 16 : 0);
  if (need > 0 && !(workspace && aligned16(workspace) && workspace_bytes >= need)) return -1;
  return gemm_w4a16_panel(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, w_layout, pp,
                          (float*)workspace, zeros ? (uint32_t*)((uint8_t*)workspace + part_bytes) : nullptr, (hipStream_t)stream);
}

// The 256-row panel kernel: the same contract.
static int try_panel256(const void* A, const void* w_packed, const void* scales, const void* zeros, void* C, int64_t M, int64_t N,
                        int64_t K, int64_t group, float zero_scalar, int in_dtype, int out_dtype, int w_layout, void* workspace,
                        int64_t workspace_bytes, void* stream, bool any_rows = false) {
  if (!(M >= 1 && N >= 1 && K > 0 && group > 0 && M < kMaxDim && N < kMaxDim && K < kMaxDim)) return -1;
  const Panel2Plan pp = w4a16_panel256_plan(any_rows ? whole_fours(M) : M, N, K, group, cu_count_or_default());
  if (!pp.ok) return -1;
  int64_t rows = with_rows_behind(M, 256);
  auto need = [&] { return pp.split > 1 ? (int64_t)pp.split * rows * N * 4 : (int64_t)0; };
  if (need() > workspace_bytes || !fits32(rows, K * 2)) rows = M;
  const bool args_ok = A && w_packed && C && aligned16(A) && aligned16(w_packed) && aligned16(C) && ((uintptr_t)scales & 1) == 0 &&
                       ((uintptr_t)zeros & 1) == 0 && (in_dtype == TLQ_F16 || in_dtype == TLQ_BF16) &&
                       (out_dtype == TLQ_F16 || out_dtype == TLQ_BF16 || out_dtype == TLQ_F32) && (M * N) % 4 == 0 &&
                       fits32(M, K * 2) && fits32(N, K / 2) && fits32(N, (K / group) * 2);
  if (!args_ok) return -1;
  if (need() > 0 && !(workspace && aligned16(workspace) && workspace_bytes >= need())) return -1;
  const int rc = gemm_w4a16_panel256(A, w_packed, scales, zeros, C, rows, N, K, group, zero_scalar, in_dtype, out_dtype,
                                     w_layout, pp, (float*)workspace, (hipStream_t)stream);
  return rows_behind_done(rc, rows != M);
}

// The middle-M panel kernel.  Returns -1 when it does not take the problem (nothing launched, no error set).
static int try_panelm(const void* A, const void* w_packed, const void* scales, const void* zeros, void* C, int64_t M, int64_t N,
                      int64_t K, int64_t group, float zero_scalar, int in_dtype, int out_dtype, void* workspace,
                      int64_t workspace_bytes, void* stream, bool any_rows = false) {
  if (!(M >= 1 && N >= 1 && K > 0 && group > 0 && M < kMaxDim && N < kMaxDim && K < kMaxDim)) return -1;
  const PanelMPlan pp = w4a16_panelm_plan(any_rows ? whole_fours(M) : M, N, K, group, cu_count_or_default());
  if (!pp.ok) return -1;
  int64_t rows = with_rows_behind(M, 16 * pp.tm);
  auto need = [&] { return pp.split > 1 ? (int64_t)pp.split * rows * N * 4 : (int64_t)0; };
  if (need() > workspace_bytes || !fits32(rows, K * 2)) rows = M;
  const bool args_ok = A && w_packed && C && aligned16(A) && aligned16(w_packed) && aligned16(C) && aligned16(scales) &&
                       aligned16(zeros) && (in_dtype == TLQ_F16 || in_dtype == TLQ_BF16) &&
                       (out_dtype == TLQ_F16 || out_dtype == TLQ_BF16 || out_dtype == TLQ_F32) && (M * N) % 4 == 0 &&
                       fits32(M, K * 2) && fits32(N, K / 2) && fits32(N, (K / group) * 2);
  if (!args_ok) return -1;
  if (need() > 0 && !(workspace && aligned16(workspace) && workspace_bytes >= need())) return -1;
  const int rc = gemm_w4a16_panelm(A, w_packed, scales, zeros, C, rows, N, K, group, zero_scalar, in_dtype, out_dtype,
                                   pp, (float*)workspace, (hipStream_t)stream);
  return rows_behind_done(rc, rows != M);
}

// One group per weight row on rows whose length is no power of two (K = 11008, 5120, 3584 ...): only the oldest kernels take
// such a group (M = 64, N = 4096, K = 11008: 59 us against 23 us with groups of 128).  The row's scale / zero point is
// written out per power-of-two group into the tail of the workspace (one small launch per tensor) and the call goes on with
// that group and the workspace in front of the tail.  Returns 0 where that does not apply (no such group, no room: the call
// goes on as it is), 1 with `out` filled in, -1 after a failed launch.
struct RowValues {
  const void* scales;
  const void* zeros;
  int64_t group, workspace_bytes;
};
static int write_out_row_values(const void* scales, const void* zeros, int64_t M, int64_t N, int64_t K, int64_t group, int in_dtype,
                                void* workspace, int64_t workspace_bytes, void* stream, RowValues& out) {
  if (!(M >= 1 && N >= 1 && N < kMaxDim && K >= 64 && K < kMaxDim && group == K && (K & (K - 1)) != 0 && K % 64 == 0 &&
        (in_dtype == TLQ_F16 || in_dtype == TLQ_BF16)))
    return 0;
  const int64_t g_eff = row_group_for(K), groups = K / g_eff, tensor_bytes = row_group_tensor_bytes(N, K);
  out = RowValues{scales, zeros, g_eff, workspace_bytes};
  if (!scales && !zeros) return 1;  // no tensors: any group size says the same
  const int64_t tail = ((scales ? 1 : 0) + (zeros ? 1 : 0)) * tensor_bytes;
  const int64_t head_bytes = (workspace_bytes - tail) & ~(int64_t)15;
  if (!(workspace && aligned16(workspace) && workspace_bytes >= tail + 16 && ((uintptr_t)scales & 1) == 0 && ((uintptr_t)zeros & 1) == 0)) return 0;
  uint8_t* const base = (uint8_t*)workspace + head_bytes;
  const int64_t n_out = N * groups;
  const int grid = (int)((n_out + 255) / 256 > 4096 ? 4096 : (n_out + 255) / 256);
  if (scales) {
    expand_row_values_kernel<<<grid, 256, 0, (hipStream_t)stream>>>((const uint16_t*)scales, (uint16_t*)base, n_out, (int)groups, grid);
    if (!check_launch("tlq_gemm_w4a16 (one scale per row, written out per group)", "expand_row_values_kernel")) return -1;
    out.scales = base;
  }
  if (zeros) {
    uint8_t* const zb = base + (scales ? tensor_bytes : 0);
    expand_row_values_kernel<<<grid, 256, 0, (hipStream_t)stream>>>((const uint16_t*)zeros, (uint16_t*)zb, n_out, (int)groups, grid);
    if (!check_launch("tlq_gemm_w4a16 (one zero point per row, written out per group)", "expand_row_values_kernel")) return -1;
    out.zeros = zb;
  }
  out.workspace_bytes = head_bytes;
  return 1;
}

// A weight-row count that is no multiple of four, more than 32 activation rows: only the skinny kernel (up to 64 rows) takes it as
// it is (N = 32001, K = 4096, M = 64: 88 us against 42 us for N = 32000; more rows were refused).  With room behind the workspace
// for the packed result of the first N - N % 16 rows: those through the usual choice, a copy into C, the last rows straight into C.
// `taken` says whether the call was answered here (the return value is then its result).
static int run_ragged_rows(const void* A, const void* w_packed, const void* scales, const void* zeros, void* C, int64_t M, int64_t N, int64_t K,
                           int64_t group, float zero_scalar, int in_dtype, int out_dtype, int w_layout, void* workspace, int64_t workspace_bytes,
                           void* stream, bool& taken) {
  taken = false;
  if (!(ragged_rows_apply(M, N) && K > 0 && K % 64 == 0 && group > 0 && K % group == 0 && group % 32 == 0 && A && w_packed && C &&
        (in_dtype == TLQ_F16 || in_dtype == TLQ_BF16) && (out_dtype == TLQ_F16 || out_dtype == TLQ_BF16 || out_dtype == TLQ_F32) &&
        ((uintptr_t)scales & 1) == 0 && ((uintptr_t)zeros & 1) == 0 && aligned16(A) && aligned16(w_packed) && aligned16(C)))
    return 0;
  const int out_bytes = out_dtype == TLQ_F32 ? 4 : 2;
  const int64_t head = ragged_head(N), result_bytes = ragged_result_bytes(M, N, out_bytes);
  if (!(head == 0 || (workspace && aligned16(workspace) && workspace_bytes >= result_bytes))) return 0;
  taken = true;
  const int64_t front = head == 0 ? 0 : (workspace_bytes - result_bytes) & ~(int64_t)15;
  uint8_t* const packed = (uint8_t*)workspace + front;
  const int64_t groups = K / group;
  if (head > 0) {
    if (int rc = tlq_gemm_w4a16_layout_ws(A, w_packed, scales, zeros, packed, M, head, K, group, zero_scalar, in_dtype, out_dtype, TLQ_ALGO_AUTO, w_layout,
                                          workspace, front, stream))
      return rc;
    const dim3 grid((unsigned)ceil_div(head, (int64_t)256), (unsigned)(M > 4096 ? 4096 : M));
    if (out_bytes == 4)
      copy_into_wider_rows_kernel<uint32_t><<<grid, 256, 0, (hipStream_t)stream>>>((const uint32_t*)packed, (uint32_t*)C, M, head, N, (int)grid.y);
    else
      copy_pairs_into_wider_rows_kernel<<<dim3((unsigned)ceil_div(head / 2 + 1, (int64_t)256), grid.y), 256, 0, (hipStream_t)stream>>>(
          (const uint16_t*)packed, (uint16_t*)C, M, head, N, (int)grid.y);
    if (!check_launch("tlq_gemm_w4a16 (packed result into C)", out_bytes == 4 ? "copy_into_wider_rows_kernel" : "copy_pairs_into_wider_rows_kernel")) return 1;
  }
  const int eb = 2;  // scales and zero points: 16-bit values
  return w4a16_tail_rows(A, (const uint8_t*)w_packed + head * (K / 2), scales ? (const uint8_t*)scales + head * groups * eb : nullptr,
                         zeros ? (const uint8_t*)zeros + head * groups * eb : nullptr, C, M, N - head, K, group, zero_scalar, in_dtype, out_dtype, w_layout, N,
                         head, (hipStream_t)stream);
}

int tlq_gemm_w4a16_ws(const void* A, const void* w_packed, const void* scales, const void* zeros, void* C, int64_t M,
                      int64_t N, int64_t K, int64_t group, float zero_scalar, int in_dtype, int out_dtype, int algo,
                      void* workspace, int64_t workspace_bytes, void* stream) {
  TLQ_REQUIRE((algo >= TLQ_ALGO_AUTO && algo <= TLQ_ALGO_PANELM) || algo == TLQ_ALGO_SMALL, "tlq_gemm_w4a16_ws: bad algo %d", algo);
  if (algo != TLQ_ALGO_TWO_PASS) {  // (not for the two passes by name: their dequantisation pass takes any group as it is)
    RowValues rv;
    const int wrote = write_out_row_values(scales, zeros, M, N, K, group, in_dtype, workspace, workspace_bytes, stream, rv);
    if (wrote < 0) return 1;
    if (wrote > 0)
      return tlq_gemm_w4a16_ws(A, w_packed, rv.scales, rv.zeros, C, M, N, K, rv.group, zero_scalar, in_dtype, out_dtype, algo, workspace, rv.workspace_bytes, stream);
  }
  if (algo == TLQ_ALGO_AUTO) {
    bool taken = false;
    const int rc = run_ragged_rows(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_W_PLAIN, workspace, workspace_bytes, stream, taken);
    if (taken) return rc;
  }
  if (algo == TLQ_ALGO_AUTO && M >= 1 && N >= 1) {
    // a tuned choice for this call signature goes first (as in tlq_gemm_w4a16); a kernel that refuses the call -- its shape
    // rules, the alignment of an operand, a workspace smaller than it needs -- has launched nothing, and the rules decide
    const int chosen = w4a16_choice_lookup(M, N, K, group, in_dtype);
    if (chosen != TLQ_ALGO_AUTO) {
      const uint64_t before = launch_count();
      const int rc = tlq_gemm_w4a16_ws(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, chosen, workspace,
                                       workspace_bytes, stream);
      if (rc == 0 || launch_count() != before) return rc;
      set_error("%s", "");
    }
  }
  const bool two_passes_fit = room_for_two_passes(N, K, workspace, workspace_bytes);
  // Above 512 rows the panel kernels are the fast path, and they were written for row counts that are multiples of four (their direct
  // loads move four activation rows).  Any other count -- prompt lengths are what they are -- runs as its multiple of four
  // below through the same choice plus the last one to three rows through the small-M kernels, which is one short launch
  // more instead of the two passes for everything (measured: M = 1001, N = 14336, K = 4096: 147 us in one piece, 128 us for
  // 1000 rows; M = 2049, N = K = 8192: 392 against 249 us; M = 601, N = K = 8192: 164 against 120 us; the tail takes 6 - 15 us).
  // One launch or two passes for all rows instead, where their estimates say so -- but not where the last rows belong to the fp16
  // GEMV kernels, whose results are closer to exact arithmetic.  bfloat16 rows, which every kernel multiplies by the same rounded weights, go along
  // with the head where they lie in its last tile (with_rows_behind): 33 of 105 random problems, 1.10 x on average (1002 x 8960 x 1152 37.7 -> 32.8 us, 3999 x 4096 x
  // 4096 117.3 -> 111.9, 1207 x 1024 x 6144 36.2 -> 29.2), one of them slower (1366 x 4224 x 512 14.5 -> 14.9).
  const bool head_and_tail = algo == TLQ_ALGO_AUTO && !g_w4a16_panel && M > 512 && (M & 3) != 0 && M < kMaxDim && N >= 16 && N % 16 == 0 &&
                             N < kMaxDim && K > 0 && K < kMaxDim && group > 0 && A && C && (in_dtype == TLQ_F16 || in_dtype == TLQ_BF16) &&
                             (out_dtype == TLQ_F16 || out_dtype == TLQ_BF16 || out_dtype == TLQ_F32) &&
                             w4a16_panel256_plan(M & ~(int64_t)3, N, K, group, cu_count_or_default()).ok;
  const bool keep_tail = head_and_tail && last_rows_take_f16_gemv(M, N, K, group, in_dtype, scales, zeros);
  // Many rows on so few and short weight rows that the whole call is a matter of latency: the small-tile kernel
  // (weight-row counts that are no multiple of four need the room of run_ragged_rows above, whatever the number of rows)
  if (algo == TLQ_ALGO_AUTO && !keep_tail && M > 512 && M < kMaxDim && N >= 1 && N % 4 == 0 && N < kMaxDim && K > 0 && K < kMaxDim && group > 0 && A && w_packed && C && aligned16(A) &&
      aligned16(w_packed) && aligned16(C) && (in_dtype == TLQ_F16 || in_dtype == TLQ_BF16) &&
      (out_dtype == TLQ_F16 || out_dtype == TLQ_BF16 || out_dtype == TLQ_F32)) {
    const SmallTile small = w4a16_small_plan(M, N, K, group, scales, zeros, 0, 0, 0);
    if (small_beats_panels(small, M, N, K, head_and_tail, two_passes_fit))
      return gemm_w4a16_small(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_W_PLAIN, small, "tlq_gemm_w4a16(small)",
                              (hipStream_t)stream);
  }
  // 33 rows and more: the small-tile kernel or the streaming kernel, whichever estimate is lower, up to 512 rows (the best of eight
  // families on 398 of 400 random problems), above 512 rows where the streaming kernel's estimate beats the panel kernels' and the two
  // passes' (stream_beats_panels).  The rules further down decide on 2^26 weights and more (2^25 from 196 rows on): the middle-M kernel where
  // panelm_preferred or panelm_whole_rounds say so, though the streaming kernel is ahead on some of it (256 x 14336 x 4096 43.7 against 36.4
  // us, which the test of that choice names), then the 128-row, the 256-row or the streaming kernel.  Above 512 rows two regions keep what
  // ran before the streaming kernel took such calls, though it is level or ahead: the two passes, where they ran, on weight-row counts
  // that are no multiple of 128 or no more than 256 (639 x 5680 x 896 22.2 against 15.5 us), and, where the panel kernels ran, a launch for
  // the last three fp16 rows.  The automatic choice's tests name those kernels too.
  bool stream_region = algo == TLQ_ALGO_AUTO && g_w4a16_stream && !keep_tail && M > 32 && M <= kStreamMaxRows && N > 0 && K > 0 && group > 0 && N < kMaxDim && K < kMaxDim &&
                       N * K < ((int64_t)1 << (M > 195 ? 25 : 26));
  // (the estimate first: it is kept per shape, the choice among the others is not and takes 1.8 us of host time)
  if (M > 512 && stream_region && (stream_region = g_stream_tiles > 0 || stream_beats_panels(M, N, K, group, two_passes_fit))) {
    const int64_t head = M & ~(int64_t)3;
    const bool two = two_passes_fit && N % 8 == 0 && (two_passes_beat_panels(M, N, K, group, in_dtype == TLQ_BF16, zeros != nullptr) || !(panelm_estimate_wins(head, N, K, group) || panel256_fills(head, N, K, group)));
    stream_region = two ? N % 128 == 0 && N > 256 : !head_and_tail;
  }
  if (stream_region) {
    const StreamPlan sp = stream_plan_for(M, N, K, group, algo, workspace, workspace_bytes);
    // (129 .. 512 rows where the 256-row kernel's estimate is ahead: on short rows of wide matrices, 472 x 20352 x 1152 in groups of 32 32.0 against
    // 39.7 us, 316 x 24960 x 256 16.8 against 20.2; it runs further down)
    const bool panel = M <= 512 && !g_w4a16_panel && panel256_beats_stream(M, N, K, group, sp);
    int64_t rows = sp.ok ? with_rows_behind(M, 16 * sp.tm) : M;
    if (!stream_workspace_ok(sp, rows, N, workspace, workspace_bytes) || !fits32(rows, K * 2)) rows = M;
    if (!panel && stream_workspace_ok(sp, rows, N, workspace, workspace_bytes) && stream_args_ok(A, w_packed, scales, zeros, C, M, N, K, in_dtype, out_dtype)) {
      const SmallTile small = w4a16_small_plan(M, N, K, group, scales, zeros, 0, 0, 0);
      // (96 rows and more on short rows, one round of 128 x 128 tiles: the tile kernel, 4.5 us + 1.45 us per 128 values of K -- 264 x 7168 x 256
      // 6.8 against 9.2 us; and, which the tests of the choice ask for, a round that is nearly full, up to 1024 values: 512 x 8192 x 1024
      // 18.0 against 16.1 us)
      const int64_t tiles128 = ceil_div(M, (int64_t)128) * ceil_div(N, (int64_t)128), cus_now = cu_count_or_default();
      const bool tiles = M >= 96 && M <= 512 && tiles128 <= cus_now && ((K <= 1024 && tiles128 * 8 >= cus_now * 7) || fused_tile_us(M, N, K) < 1.02 * sp.us);
      if (tiles)
        return tlq_gemm_w4a16(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype,
                              small_or(TLQ_ALGO_MFMA, M, N, K, group, scales, zeros), stream);
      if (M <= 512 && small_beats_stream(small, sp, M, N, K, group, zeros != nullptr))
        return gemm_w4a16_small(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_W_PLAIN, small, "tlq_gemm_w4a16(small)",
                                (hipStream_t)stream);
      const int rc = gemm_w4a16_stream(A, w_packed, scales, zeros, C, rows, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_W_PLAIN, sp, (float*)workspace,
                                       (hipStream_t)stream);
      return rows_behind_done(rc, rows != M);
    }
  }
  if (head_and_tail && (keep_tail || !(two_passes_fit && two_passes_beat_panels(M, N, K, group, in_dtype == TLQ_BF16, zeros != nullptr)))) {
    const int64_t head = M & ~(int64_t)3;
    const bool may_go_along = in_dtype == TLQ_BF16;
    g_rows_behind = may_go_along ? M - head : 0;
    const int rc = tlq_gemm_w4a16_ws(A, w_packed, scales, zeros, C, head, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_ALGO_AUTO, workspace,
                                     workspace_bytes, stream);
    const bool went_along = may_go_along && g_rows_behind == 0;
    g_rows_behind = 0;
    if (rc != 0 || went_along) return rc;
    const int64_t out_bytes = out_dtype == TLQ_F32 ? 4 : 2;
    return tlq_gemm_w4a16((const uint8_t*)A + head * K * 2, w_packed, scales, zeros, (uint8_t*)C + head * N * out_bytes, M - head, N, K, group,
                          zero_scalar, in_dtype, out_dtype, TLQ_ALGO_AUTO, stream);
  }
  if (algo == TLQ_ALGO_PANELM) {
    const int rc = try_panelm(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, workspace, workspace_bytes, stream);
    TLQ_REQUIRE(rc >= 0, "tlq_gemm_w4a16_ws: the middle-M panel kernel needs K %% 128 == 0, M %% 4 == 0, N %% 16 == 0, a power-of-two group "
                ">= 64 with (K / group) %% 8 == 0, 16-byte aligned operands, scale and zero tensors, and a workspace for its K slices (M=%lld "
                "N=%lld K=%lld group=%lld, workspace %lld)", (long long)M, (long long)N, (long long)K, (long long)group, (long long)workspace_bytes);
    return rc;
  }
  if (algo == TLQ_ALGO_PANEL256) {
    const int rc = try_panel256(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_W_PLAIN, workspace,
                                workspace_bytes, stream);
    TLQ_REQUIRE(rc >= 0, "tlq_gemm_w4a16_ws: the 256-row panel kernel needs K %% 128 == 0, M %% 4 == 0, N %% 16 == 0, a power-of-two group "
                ">= 32, 16-byte aligned operands and a workspace for its K slices (M=%lld "
                "N=%lld K=%lld group=%lld, workspace %lld)", (long long)M, (long long)N, (long long)K, (long long)group, (long long)workspace_bytes);
    return rc;
  }
  if (algo == TLQ_ALGO_PANEL) {
    const int rc = try_panel(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_W_PLAIN, workspace,
                             workspace_bytes, stream);
    TLQ_REQUIRE(rc >= 0, "tlq_gemm_w4a16_ws: the panel kernel needs K %% 128 == 0, M %% 4 == 0, N %% 16 == 0, a power-of-two group >= 32 "
                "with (K / group) %% 8 == 0, 16-byte aligned operands, scale and zero tensors, and a workspace for its K slices and (with a "
                "zero-point tensor) 16 bytes more (M=%lld N=%lld K=%lld group=%lld, workspace %lld)", (long long)M, (long long)N, (long long)K, (long long)group, (long long)workspace_bytes);
    return rc;
  }
  // decode batches: rows longer than 4096 values run as chunks of K whose fp32 partial sums live in the workspace
  if (((algo == TLQ_ALGO_AUTO && g_w4a16_decode && (decode_preferred(M, N, K) || K > 16384)) || algo == TLQ_ALGO_DECODE) && M <= 32 && M >= 1 && N >= 1 && K > 0 && group > 0 &&
      N < kMaxDim && K < kMaxDim) {
    const DecodePlan dp = w4a16_decode_plan(M, N, K, group, cu_count_or_default());
    const bool args_ok = A && w_packed && C && aligned16(A) && aligned16(w_packed) && aligned16(C) &&
                         (in_dtype == TLQ_F16 || in_dtype == TLQ_BF16) &&
                         (out_dtype == TLQ_F16 || out_dtype == TLQ_BF16 || out_dtype == TLQ_F32) &&
                         (((uintptr_t)scales | (uintptr_t)zeros) & 3) == 0;
    // measured on rows of 14336 values: with up to 16 activation rows the skinny kernel is level or ahead (no second
    // launch for the partial sums), from 17 rows on the decode kernel is 10 - 15 % ahead of the streaming kernel
    // (also for rows of more than 16384 values, which the register-resident GEMV does not take: M = 1, N = 8192,
    // K = 28672: 32 against 49 us for the generic GEMV;
    // from 64 MB of weights on -- N = 28672, K = 8192, M = 16: 31.6 against 45.6 us -- and where the skinny kernel's
    // work-groups, one per 16 weight rows, would leave a fifth of the machine or more idle in their last round:
    // N = 5120, K = 13824: 15.8 against 23.6 us; with 8192 or 13824 weight rows the skinny kernel is level or ahead.
    // Two of its work-groups share a CU, so that holds for rounds of twice the CU count as well: N = 10240, K = 8192
    // (640 work-groups on 512 places): 15 against 20 - 26 us; N = 12288, K = 6144 (768): 14 - 15 against 17 - 21 us;
    // N = 17408, K = 5120 (1088): 17 - 19 against 20 - 24 us; with 512 or 960 work-groups the skinny kernel is ahead)
    if (algo == TLQ_ALGO_AUTO && dp.ok && dp.chunks > 1 && args_ok) {
      const SmallTile small = w4a16_small_plan(M, N, K, group, scales, zeros, 0, 0, 0);
      if (small_beats_decode_chunks(small, M, N, K))
        return gemm_w4a16_small(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_W_PLAIN, small, "tlq_gemm_w4a16(small)",
                                (hipStream_t)stream);
    }
    if (dp.ok && dp.chunks > 1 && (algo == TLQ_ALGO_DECODE || M > 16 || K > 16384 || N * (K / 2) >= ((int64_t)64 << 20) || skinny_leaves_cus_idle(N)) && args_ok && (M * N) % 4 == 0 && workspace && aligned16(workspace) &&
        workspace_bytes >= (int64_t)dp.chunks * M * N * 4)
      return gemm_w4a16_decode(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_W_PLAIN, dp,
                               (float*)workspace, (hipStream_t)stream);
    if (algo == TLQ_ALGO_DECODE && !(dp.ok && dp.chunks == 1)) {
      set_error("tlq_gemm_w4a16_ws: the decode kernel needs 1 <= M <= 32, K %% 256 == 0, a power-of-two group, dword-aligned scale / zero "
                "tensors, M * N %% 4 == 0 and a workspace of %lld bytes (M=%lld N=%lld K=%lld group=%lld, workspace %lld)",
                (long long)(dp.ok ? (int64_t)dp.chunks * M * N * 4 : 0), (long long)M, (long long)N, (long long)K, (long long)group,
                (long long)workspace_bytes);
      return 1;
    }
  }
  if (algo == TLQ_ALGO_AUTO && M >= 1 && N >= 1 && K > 0 && N < kMaxDim && K < kMaxDim) {
    // Small problems are launch-bound: a second launch (for the partial sums of K slices, or for the dequantisation
    // pass) costs more than it saves.  Measured: 256^3 6.5 against 9.5 us, M = 128 on 1024 x 512 9.7 against 12.4 us,
    // M = 64 on 1024^2 6.7 against 11.4 us and on 2048^2 11.0 against 13.0 us; the streaming kernel with its K slices is
    // ahead from M = 256 on 1024^2 (15.5 against 20.8 us) and for M = 40 on 1024 rows of 4096 values (13.0 against 16.5 us).
    // Short rows (K <= 2048) on up to 2^24 weights, 33 .. 64 activation rows: the skinny kernel's single launch is ahead of the
    // streaming kernel, whose launch has 8 us that do not depend on K (N = 8192, K = 1024: 7.9 / 8.4 against 12.5 / 13.4 us at
    // 40 / 64 rows; N = 16384, K = 1024: 10.7 / 12.4 against 13.8 / 15.6 us; N = 8192, K = 2048: 12.0 / 14.9 against 14.7 / 16.4 us;
    // behind from 2^25 weights on and with rows of 3072 values).
    const int64_t nk = N * K;
    // (rows of more than 1280 values only where the skinny kernel's work-groups, one per 16 weight rows, run in one round or
    // fill their last round: N = 6144, K = 2048, 384 work-groups: 16 - 22 against 14 - 15 us)
    const bool skinny_fills = ceil_div(N, (int64_t)16) <= cu_count_or_default() || tile_fill(1, 16, N, 16) >= 0.8;
    if ((M <= 64 && (nk <= ((int64_t)1 << 21) || (nk <= ((int64_t)1 << 24) && (K <= 1280 || (K <= 2048 && skinny_fills))))) || (nk <= ((int64_t)1 << 19) && !(two_passes_fit && two_passes_beat_tiles(M, N, K))))
      return tlq_gemm_w4a16(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_ALGO_AUTO, stream);
    // Short rows, 96 .. 512 activation rows, one round of 128 x 128 tiles: the tile kernel in one launch takes 4.5 us + 1.45 us
    // per 128 values of K whatever M and N, the streaming kernel 11 - 15 us at K = 512 and 19 - 30 us at K = 1024 .. 1536.
    // Measured on five values of N from 2048 to 32768 x six of M: ahead by 1.1 - 1.4 x on all 23 cases at K = 512, by
    // 1.07 - 1.4 x at K = 1024 from 96 tiles on (level or behind with 64 tiles and fewer), by 1.1 - 1.27 x at K = 1536 from 128
    // tiles and 128 rows on; behind at K = 2048.  (Groups of 32 values at K = 1024: from 192 tiles on; fp16 with a zero-point
    // tensor is 3 - 16 % behind on 96 - 128 tiles.)  Out of sample (eight values of K from 384 to 2560 x seven of N x seven of M, both
    // types, against the build before): 1.1 - 1.5 x on the cases that change, none more than 3 % slower.
    const int64_t tiles128 = ceil_div(M, (int64_t)128) * ceil_div(N, (int64_t)128);
    if (M >= 96 && M <= 512 && N % 4 == 0 && tiles128 <= cu_count_or_default() &&
        (K <= 512 || (K <= 768 && tiles128 >= 96) || (K <= 1024 && tiles128 >= (group < 64 ? 192 : 96)) || (K <= 1536 && tiles128 >= 128 && (M == 128 || M > 192))))  // (129 .. 192 rows: the streaming kernel's blocks of 96 rows are level there)
      return tlq_gemm_w4a16(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype,
                            small_or(TLQ_ALGO_MFMA, M, N, K, group, scales, zeros), stream);
    // 17 .. 32 activation rows whose K is one chunk of the decode kernel: that kernel, which needs no workspace
    // (M = 32, N = 14336, K = 4096: 16.8 against 20 us for the streaming kernel)
    if (M > 16 && M <= 32 && g_w4a16_decode && group > 0) {
      const DecodePlan dp = w4a16_decode_plan(M, N, K, group, cu_count_or_default());
      if (dp.ok && dp.chunks == 1 && (((uintptr_t)scales | (uintptr_t)zeros) & 3) == 0)
        return tlq_gemm_w4a16(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_ALGO_AUTO, stream);
    }
  }
  const int64_t need = (N > 0 && K > 0) ? N * K * 2 : 0;
  const bool have = workspace != nullptr && workspace_bytes >= need && aligned16(workspace);
  if (algo == TLQ_ALGO_TWO_PASS)
    TLQ_REQUIRE(have, "tlq_gemm_w4a16_ws: the two-pass path needs a 16-byte aligned workspace of %lld bytes (got %lld)",
                (long long)need, (long long)workspace_bytes);
  // 256 .. 512 activation rows on large matrices: the middle-M panel kernel
  // (not up to 256 rows with groups of 512 values or more: the panel kernels cut K into windows of eight groups -- 32 steps and
  // more -- and run uncut or nearly so, the streaming kernel cuts inside a group: N = 14336, K = 4096, M = 256: 50 against 59 us;
  // N = 11008: 47 against 58 us; N = K = 8192: 52 against 61 us; from 384 rows on the panel kernels are ahead again)
  auto stream_instead = [&] {
    const StreamPlan sp = stream_plan_for(M, N, K, group, algo, workspace, workspace_bytes);
    return stream_beats_middle(M, N, K, group, in_dtype, sp) && stream_workspace_ok(sp, M, N, workspace, workspace_bytes) &&
           stream_args_ok(A, w_packed, scales, zeros, C, M, N, K, in_dtype, out_dtype);
  };
  if (algo == TLQ_ALGO_AUTO && !g_w4a16_panel && group > 0 && (panelm_preferred(M, N, K) || panelm_whole_rounds(M, N, K, group, in_dtype)) && !(M <= 256 && group >= 512) &&
      !stream_instead()) {
    // (very wide matrices: where the 128-row tiles need a second round of work-groups and the 256-row tiles do not, the
    // 256-row kernel by the same estimate -- N = 28672, K = 4096, M = 512: 104 against 129 us)
    if (panel256_estimate_wins(M, N, K, group)) {
      const int rc = try_panel256(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_W_PLAIN, workspace,
                                  workspace_bytes, stream, true);
      if (rc >= 0) return rc;
    }
    const int rc = try_panelm(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, workspace, workspace_bytes, stream, true);
    if (rc >= 0) return rc;
  }
  if (algo == TLQ_ALGO_AUTO && !g_w4a16_panel && panel_one_round(M, N, K) && group > 0) {
    const int rc = try_panel(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_W_PLAIN, workspace, workspace_bytes, stream);
    if (rc >= 0) return rc;
  }
  if (algo == TLQ_ALGO_AUTO && !g_w4a16_panel && panelm_one_tile(M, N, K) && group > 0) {
    const int rc = try_panelm(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, workspace, workspace_bytes, stream, true);
    if (rc >= 0) return rc;
  }
  // 17 .. 512 activation rows: the streaming kernel (weights once per 128 rows, deep ring of direct loads)
  if ((algo == TLQ_ALGO_AUTO && g_w4a16_stream) || algo == TLQ_ALGO_STREAM) {
    const StreamPlan sp = M <= 512 || g_stream_tiles > 0 ? stream_plan_for(M, N, K, group, algo, workspace, workspace_bytes) : StreamPlan{};
    const bool args_ok = stream_args_ok(A, w_packed, scales, zeros, C, M, N, K, in_dtype, out_dtype);
    const bool ws_ok = stream_workspace_ok(sp, M, N, workspace, workspace_bytes);
    if (algo == TLQ_ALGO_AUTO && sp.ok && args_ok) {
      const SmallTile small = w4a16_small_plan(M, N, K, group, scales, zeros, 0, 0, 0);
      if (small_beats_stream(small, sp, M, N, K, group, zeros != nullptr))
        return gemm_w4a16_small(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_W_PLAIN, small, "tlq_gemm_w4a16(small)",
                                (hipStream_t)stream);
    }
    if (algo == TLQ_ALGO_AUTO && !g_w4a16_panel && group > 0 && panel256_beats_stream(M, N, K, group, sp)) {
      const int rc = try_panel256(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_W_PLAIN, workspace,
                                  workspace_bytes, stream, true);
      if (rc >= 0) return rc;
    }
    // What is left, the tile kernel over K slices and the two passes, is behind on 783 of 796 problems (33 .. 512 rows, 2^25 .. 2^29 weights,
    // groups of 32 - 4096, both types): 318 x 24192 x 8576 213 us against 300 and 333, 407 x 19968 x 2048 50 against 80 and 64, 319 x 3200 x 12800
    // in groups of 32 51 against 89 and 74.  On ten of the others the 256-row kernel, asked above, is ahead of all three; the last three (groups of 32;
    // 5, 6 and 17 % ahead) do not carry a rule.
    if (sp.ok && args_ok && ws_ok)
      return gemm_w4a16_stream(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_W_PLAIN, sp, (float*)workspace,
                               (hipStream_t)stream);
    if (algo == TLQ_ALGO_STREAM) {
      set_error("tlq_gemm_w4a16_ws: the streaming kernel needs 17 <= M <= 512, K %% 128 == 0, a power-of-two group >= 32, N %% 4 == 0, "
                "16-byte aligned operands and a workspace of %lld bytes (M=%lld N=%lld K=%lld group=%lld, workspace %lld)",
                (long long)(sp.ok ? (int64_t)sp.split * M * N * 4 : 0), (long long)M, (long long)N, (long long)K, (long long)group,
                (long long)workspace_bytes);
      return 1;
    }
  }
  // Above 512 rows: the 256-row panel kernel (one launch, no dequantised matrix) where its work-groups fill the machine.
  // Measured against the choice without it (two passes, tile kernel over K slices) and against the 128-row panel kernel
  // on ten (N, K) pairs x eleven values of M from 576 to 8192, fp16 with a zero-point tensor and bf16 with a scalar one,
  // groups of 128: wherever its last round of work-groups fills more than half of the CUs it is level or ahead -- by 3 - 16 %
  // from 3072 rows on (4096 x 4096 x 4096 bf16: 104 against 113 - 119 us; 8192 x 8192 x 8192: 1.11 x), by 10 - 56 % between
  // 576 and 2048 rows on wide or long matrices (N = 28672, K = 4096, M = 768: 1.40 - 1.54 x; N = 4096, K = 14336, M = 1280:
  // 1.50 - 1.56 x), 0.98 - 0.99 on a few of the largest fp16 problems -- and 2 - 21 % behind below that fill (N = K = 4096,
  // M <= 1024: 96 work-groups).  The 128-row kernel is ahead of it nowhere by more than 4 % and stays an explicit choice.
  if (algo == TLQ_ALGO_AUTO && !g_w4a16_panel && M > 512 && K > 0 && group > 0 && N >= 1 && N < kMaxDim && K < kMaxDim && M < kMaxDim &&
      !(have && two_passes_beat_panels(M, N, K, group, in_dtype == TLQ_BF16, zeros != nullptr))) {
    // The middle-M kernel's 128-row tiles first where an estimate of both kernels' times says so: rounds of work-groups x
    // (steps per K slice x the time of a step + a fixed part) + the pass over the slices' partial tiles, with the step
    // times measured at a full machine (2.2 us on 128 rows, 3.3 us on 256) and fixed parts of 6 / 8 us.  On ten (N, K)
    // pairs x M = 576 .. 3072, fp16 with a zero-point tensor and bf16 with a scalar one (144 cases where both kernels
    // apply), taking the 128-row kernel where its estimate is below 0.94 of the other's never lost against the choice
    // without it and gains 4 % on average: N = 11008, K = 4096, M = 576 - 640 (5 x 43 tiles fill the machine once, 3 x 43
    // half of it) 69 against 102 - 106 us; N = 8192, K = 2048, M <= 1024 35 - 43 against 50 - 54 us; N = K = 4096, M = 1024
    // 50 against 62 us; N = 2048, K = 8192, M <= 1024 42 - 51 against 47 - 59 us.
    if (panelm_estimate_wins(M, N, K, group)) {
      const int rc = try_panelm(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, workspace, workspace_bytes, stream);
      if (rc >= 0) return rc;
    }
    if (panel256_fills(M, N, K, group)) {
      const int rc = try_panel256(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, TLQ_W_PLAIN, workspace,
                                  workspace_bytes, stream);
      if (rc >= 0) return rc;
    }
  }
  // (above 512 rows only rows of 13312 values and more: below, the plain GEMM of the two passes, in the ring kernel
  // or over uneven slices of K, is ahead: 614 x 1392 x 2304 28.7 -> 20.6 us, 667 x 256 x 12288 36.8 -> 25.3, 682 x 2288 x 11648
  // 76.4 -> 66.3; 656 x 2496 x 3712 level)
  const bool split_region = !(algo == TLQ_ALGO_AUTO && have && M > 512 && K < 13312 && N % 8 == 0 && w4a16_split_forced() == 0) &&
                            w4a16_mid_split(M, N, K, group > 0 ? group : 32) > 1;
  const bool two_pass = algo == TLQ_ALGO_TWO_PASS ||
                        (algo == TLQ_ALGO_AUTO && have && M >= kTwoPassMinM && N % 8 == 0 && !split_region);
  if (!two_pass && (algo == TLQ_ALGO_AUTO || algo == TLQ_ALGO_MFMA) && M > 16 && workspace && aligned16(workspace) &&
      K > 0 && K % 64 == 0 && group > 0 && K % group == 0 && group % 32 == 0 && A && w_packed && C && aligned16(A) &&
      aligned16(w_packed) && aligned16(C) && N % 4 == 0 && (M * N) % 4 == 0 && M < kMaxDim && N < kMaxDim && K < kMaxDim &&
      (in_dtype == TLQ_F16 || in_dtype == TLQ_BF16) && (out_dtype == TLQ_F16 || out_dtype == TLQ_BF16 || out_dtype == TLQ_F32) &&
      fits32(M, K * 2) && fits32(N, K / 2) && ((uintptr_t)scales & 1) == 0 && ((uintptr_t)zeros & 1) == 0) {
    // small and middle M: the tile kernel over K slices, partial sums in the workspace, one pass to add them up
    const int64_t split = w4a16_mid_split(M, N, K, group);
    if (split > 1 && workspace_bytes >= split * M * N * 4)
      return gemm_w4a16_mfma_splitk(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, split,
                                    (float*)workspace, (hipStream_t)stream);
  }
  if (!two_pass)
    return tlq_gemm_w4a16(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype,
                          algo == TLQ_ALGO_TWO_PASS ? TLQ_ALGO_AUTO : algo, stream);
  TLQ_CHECK_DIMS("tlq_gemm_w4a16_ws");
  TLQ_REQUIRE(in_dtype == TLQ_F16 || in_dtype == TLQ_BF16, "tlq_gemm_w4a16_ws: in_dtype must be float16 or bfloat16 (got %d)",
              in_dtype);
  TLQ_REQUIRE(out_dtype == TLQ_F16 || out_dtype == TLQ_BF16 || out_dtype == TLQ_F32,
              "tlq_gemm_w4a16_ws: out_dtype must be float16, bfloat16 or float32 (got %d)", out_dtype);
  if (M == 0 || N == 0) return 0;
  TLQ_REQUIRE(K > 0 && K % 64 == 0, "tlq_gemm_w4a16_ws: K=%lld must be a positive multiple of 64", (long long)K);
  TLQ_REQUIRE(group > 0 && K % group == 0 && group % 32 == 0,
              "tlq_gemm_w4a16_ws: group=%lld must divide K=%lld and be a multiple of 32", (long long)group, (long long)K);
  TLQ_REQUIRE(((uintptr_t)scales & 1) == 0 && ((uintptr_t)zeros & 1) == 0, "tlq_gemm_w4a16_ws: scales / zeros misaligned");
  if (int rc = tlq_dequant_w4(w_packed, scales, zeros, workspace, N, K, group, zero_scalar, in_dtype, stream)) return rc;
  return plain_gemm_on_workspace(A, workspace, workspace_bytes, C, M, N, K, in_dtype, out_dtype, stream);
}

int tlq_gemm_w4a16_layout_ws(const void* A, const void* w_packed, const void* scales, const void* zeros, void* C, int64_t M,
                             int64_t N, int64_t K, int64_t group, float zero_scalar, int in_dtype, int out_dtype, int algo,
                             int w_layout, void* workspace, int64_t workspace_bytes, void* stream) {
  TLQ_REQUIRE(w_layout == TLQ_W_PLAIN || w_layout == TLQ_W_INTERLEAVED_F16, "tlq_gemm_w4a16_layout_ws: bad weight layout %d", w_layout);
  if (w_layout == TLQ_W_PLAIN)
    return tlq_gemm_w4a16_ws(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, algo, workspace,
                             workspace_bytes, stream);
  TLQ_CHECK_DIMS("tlq_gemm_w4a16_layout_ws");
  TLQ_REQUIRE(algo == TLQ_ALGO_AUTO || algo == TLQ_ALGO_GEMV || algo == TLQ_ALGO_STREAM || algo == TLQ_ALGO_TWO_PASS || algo == TLQ_ALGO_DECODE || algo == TLQ_ALGO_PANEL || algo == TLQ_ALGO_PANEL256 ||
                  algo == TLQ_ALGO_SMALL,
              "tlq_gemm_w4a16_layout_ws: interleaved weights are read by the ring GEMV, the decode kernel, the small-tile kernel, the streaming kernel, the panel kernels and the two passes (algo %d)", algo);
  TLQ_REQUIRE(in_dtype == TLQ_F16 || in_dtype == TLQ_BF16, "tlq_gemm_w4a16_layout_ws: in_dtype must be float16 or bfloat16 (got %d)", in_dtype);
  TLQ_REQUIRE(out_dtype == TLQ_F16 || out_dtype == TLQ_BF16 || out_dtype == TLQ_F32, "tlq_gemm_w4a16_layout_ws: bad out_dtype %d", out_dtype);
  if (M == 0 || N == 0) return 0;
  TLQ_REQUIRE(K > 0 && K % 64 == 0, "tlq_gemm_w4a16_layout_ws: K=%lld must be a positive multiple of 64", (long long)K);
  TLQ_REQUIRE(group > 0 && K % group == 0 && group % 32 == 0, "tlq_gemm_w4a16_layout_ws: group=%lld must divide K=%lld and be a multiple of 32",
              (long long)group, (long long)K);
  TLQ_REQUIRE(A && w_packed && C, "tlq_gemm_w4a16_layout_ws: null pointer");
  TLQ_REQUIRE(aligned16(A) && aligned16(w_packed) && aligned16(C), "tlq_gemm_w4a16_layout_ws: A, w_packed and C must be 16-byte aligned");
  TLQ_REQUIRE(((uintptr_t)scales & 1) == 0 && ((uintptr_t)zeros & 1) == 0, "tlq_gemm_w4a16_layout_ws: scales / zeros misaligned");
  TLQ_REQUIRE(fits32(M, K * 2) && fits32(N, K / 2), "tlq_gemm_w4a16_layout_ws: a matrix spans 4 GiB or more");
  if (algo != TLQ_ALGO_TWO_PASS) {  // one scale / zero point per row on rows that are no power of two: as for plain words
    RowValues rv;
    const int wrote = write_out_row_values(scales, zeros, M, N, K, group, in_dtype, workspace, workspace_bytes, stream, rv);
    if (wrote < 0) return 1;
    if (wrote > 0)
      return tlq_gemm_w4a16_layout_ws(A, w_packed, rv.scales, rv.zeros, C, M, N, K, rv.group, zero_scalar, in_dtype, out_dtype, algo, w_layout, workspace,
                                      rv.workspace_bytes, stream);
  }
  if (algo == TLQ_ALGO_AUTO) {  // ragged weight-row counts: as for plain words
    bool taken = false;
    const int rc = run_ragged_rows(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, w_layout, workspace, workspace_bytes, stream, taken);
    if (taken) return rc;
  }
  const bool ws_aligned = workspace && aligned16(workspace);
  if (algo == TLQ_ALGO_SMALL) {
    const SmallTile p = w4a16_small_plan(M, N, K, group, scales, zeros, 0, 0, 0);
    TLQ_REQUIRE(p.ok, TLQ_SMALL_NEEDS("tlq_gemm_w4a16_layout_ws"), (long long)M, (long long)N, (long long)K, (long long)group);
    return gemm_w4a16_small(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, w_layout, p, "tlq_gemm_w4a16(small)", (hipStream_t)stream);
  }
  // one or two activation rows: the ring GEMV where the plain layout takes it too (one row; two fp16 rows on 8192 weight
  // rows or more), or when asked for by name
  if (M <= 2 && (algo == TLQ_ALGO_GEMV || (algo == TLQ_ALGO_AUTO && (M == 1 || N >= 8192)))) {
    const int rc = gemv_w4a16_ring_interleaved(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype,
                                               (hipStream_t)stream);
    if (rc >= 0) return rc;
    TLQ_REQUIRE(algo != TLQ_ALGO_GEMV, "tlq_gemm_w4a16_layout_ws: the GEMV kernel reads interleaved weights for M <= 2 (fp16; bf16 M = 1), "
                "K <= 4096, a power-of-two group with (K / group) %% 8 == 0 and 16-byte aligned scale / zero tensors (M=%lld N=%lld K=%lld "
                "group=%lld)", (long long)M, (long long)N, (long long)K, (long long)group);
  }
  TLQ_REQUIRE(algo != TLQ_ALGO_GEMV, "tlq_gemm_w4a16_layout_ws: the GEMV kernel reads interleaved weights for M <= 2 only (got %lld)", (long long)M);
  if (M <= 32 && (algo == TLQ_ALGO_AUTO || algo == TLQ_ALGO_DECODE)) {
    const DecodePlan dp = w4a16_decode_plan(M, N, K, group, cu_count_or_default());
    const bool dec_ok = dp.ok && (((uintptr_t)scales | (uintptr_t)zeros) & 3) == 0 &&
                        (dp.chunks == 1 || ((M * N) % 4 == 0 && ws_aligned && workspace_bytes >= (int64_t)dp.chunks * M * N * 4));
    if (dec_ok)
      return gemm_w4a16_decode(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, w_layout, dp,
                               (float*)workspace, (hipStream_t)stream);
    TLQ_REQUIRE(algo != TLQ_ALGO_DECODE, "tlq_gemm_w4a16_layout_ws: the decode kernel does not take M=%lld N=%lld K=%lld group=%lld with a "
                "workspace of %lld bytes (K %% 256 == 0, a power-of-two group, dword-aligned scale / zero tensors)", (long long)M, (long long)N,
                (long long)K, (long long)group, (long long)workspace_bytes);
  }
  TLQ_REQUIRE(algo != TLQ_ALGO_DECODE, "tlq_gemm_w4a16_layout_ws: the decode kernel handles M <= 32 (got %lld)", (long long)M);
  if (algo == TLQ_ALGO_PANEL256 || (algo == TLQ_ALGO_AUTO && !g_w4a16_panel && M > 512)) {
    // (the same rule as for plain words: where the 256-row panel kernel's tiles fill the machine)
    if (algo == TLQ_ALGO_PANEL256 || panel256_fills(M, N, K, group)) {
      const int rc = try_panel256(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, w_layout, workspace,
                                  workspace_bytes, stream);
      if (rc >= 0) return rc;
    }
    TLQ_REQUIRE(algo != TLQ_ALGO_PANEL256, "tlq_gemm_w4a16_layout_ws: the 256-row panel kernel does not take M=%lld N=%lld K=%lld group=%lld "
                "with a workspace of %lld bytes (K %% 128 == 0, M %% 4 == 0, N %% 16 == 0, a power-of-two group >= 32)", (long long)M,
                (long long)N, (long long)K, (long long)group, (long long)workspace_bytes);
  }
  if (algo == TLQ_ALGO_PANEL) {
    const PanelPlan pp = w4a16_panel_plan(M, N, K, group, cu_count_or_default());
    if (pp.ok) {
      const int rc = try_panel(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, w_layout, workspace,
                               workspace_bytes, stream);
      if (rc >= 0) return rc;
    }
    TLQ_REQUIRE(false, "tlq_gemm_w4a16_layout_ws: the panel kernel does not take M=%lld N=%lld K=%lld group=%lld with a "
                "workspace of %lld bytes (K %% 128 == 0, M %% 4 == 0, N %% 16 == 0, a power-of-two group with (K / group) %% 8 == 0, 16-byte "
                "aligned scale / zero tensors)", (long long)M, (long long)N, (long long)K, (long long)group, (long long)workspace_bytes);
  }
  if (algo == TLQ_ALGO_AUTO && !g_w4a16_panel && panel_one_round(M, N, K)) {  // (65 .. 128 rows on output-layer widths, as for plain words)
    const int rc = try_panel(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, w_layout, workspace, workspace_bytes, stream);
    if (rc >= 0) return rc;
  }
  if (algo != TLQ_ALGO_TWO_PASS) {
    const StreamPlan sp = M <= 512 ? stream_plan_for(M, N, K, group, algo, workspace, workspace_bytes) : StreamPlan{};
    const bool ws_ok = sp.ok && (M * N) % 4 == 0 && (sp.split == 1 || (ws_aligned && workspace_bytes >= (int64_t)sp.split * M * N * 4));
    // (no tile kernel reads this layout: the alternative is the two passes, which are behind: 512 x 8192 x 4096 39 against 56 us)
    // the small-tile kernel in the place of either, for calls that bring the workspace those want: without it they are refused
    if (algo == TLQ_ALGO_AUTO && sp.ok && (M * N) % 4 == 0 && (ws_ok || (room_for_two_passes(N, K, workspace, workspace_bytes) && N % 8 == 0))) {
      const SmallTile small = w4a16_small_plan(M, N, K, group, scales, zeros, 0, 0, 0);
      if (small_beats_stream(small, sp, M, N, K, group, zeros != nullptr))
        return gemm_w4a16_small(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, w_layout, small, "tlq_gemm_w4a16(small)",
                                (hipStream_t)stream);
    }
    // (129 .. 512 rows: the 256-row kernel where its estimate beats the streaming kernel's, as for the plain layout)
    if (algo == TLQ_ALGO_AUTO && !g_w4a16_panel && group > 0 && panel256_beats_stream(M, N, K, group, sp)) {
      const int rc = try_panel256(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, w_layout, workspace,
                                  workspace_bytes, stream);
      if (rc >= 0) return rc;
    }
    if (ws_ok)
      return gemm_w4a16_stream(A, w_packed, scales, zeros, C, M, N, K, group, zero_scalar, in_dtype, out_dtype, w_layout, sp,
                               (float*)workspace, (hipStream_t)stream);
    TLQ_REQUIRE(algo != TLQ_ALGO_STREAM, "tlq_gemm_w4a16_layout_ws: the streaming kernel does not take M=%lld N=%lld K=%lld group=%lld "
                "with a workspace of %lld bytes", (long long)M, (long long)N, (long long)K, (long long)group, (long long)workspace_bytes);
  }
  TLQ_REQUIRE(M >= 17, "tlq_gemm_w4a16_layout_ws: with M=%lld interleaved weights need the decode kernel's shapes (K %% 256 == 0, power-of-two "
              "group, dword-aligned scale / zero tensors); other decode-sized problems read the plain layout", (long long)M);
  TLQ_REQUIRE(ws_aligned && workspace_bytes >= N * K * 2 && N % 8 == 0,
              "tlq_gemm_w4a16_layout_ws: M=%lld N=%lld K=%lld needs a 16-byte aligned workspace of %lld bytes (got %lld) and N %% 8 == 0",
              (long long)M, (long long)N, (long long)K, (long long)(N * K * 2), (long long)workspace_bytes);
  if (int rc = tlq_dequant_w4_layout(w_packed, scales, zeros, workspace, N, K, group, zero_scalar, in_dtype, w_layout, stream)) return rc;
  return plain_gemm_on_workspace(A, workspace, workspace_bytes, C, M, N, K, in_dtype, out_dtype, stream);
}

int tlq_gemv_w4a16_batched(const void* A, const void* w_packed, const void* scales, const void* zeros, void* C,
                           int64_t batch, int64_t M, int64_t N, int64_t K, int64_t group, float zero_scalar, int in_dtype,
                           int out_dtype, void* stream) {
  TLQ_CHECK_DIMS("tlq_gemv_w4a16_batched");
  TLQ_REQUIRE(batch >= 0 && batch <= 65535, "tlq_gemv_w4a16_batched: batch=%lld must be in 0..65535", (long long)batch);
  TLQ_REQUIRE(in_dtype == TLQ_F16 || in_dtype == TLQ_BF16, "tlq_gemv_w4a16_batched: bad in_dtype %d", in_dtype);
  TLQ_REQUIRE(out_dtype == TLQ_F16 || out_dtype == TLQ_BF16 || out_dtype == TLQ_F32, "tlq_gemv_w4a16_batched: bad out_dtype %d",
              out_dtype);
  if (batch == 0 || M == 0 || N == 0) return 0;
  TLQ_REQUIRE(M <= 16, "tlq_gemv_w4a16_batched: M=%lld must be <= 16", (long long)M);
  TLQ_REQUIRE(K > 0 && K % 64 == 0, "tlq_gemv_w4a16_batched: K=%lld must be a positive multiple of 64", (long long)K);
  TLQ_REQUIRE(group > 0 && K % group == 0 && group % 32 == 0,
              "tlq_gemv_w4a16_batched: group=%lld must divide K=%lld and be a multiple of 32", (long long)group, (long long)K);
  TLQ_REQUIRE(A && w_packed && C, "tlq_gemv_w4a16_batched: null pointer");
  TLQ_REQUIRE(aligned16(A) && aligned16(w_packed), "tlq_gemv_w4a16_batched: A and w_packed must be 16-byte aligned");
  return gemv_w4a16(A, w_packed, scales, zeros, C, batch, M, N, K, group, zero_scalar, in_dtype, out_dtype,
                    (hipStream_t)stream);
}

// What a call takes that cuts K into slices over work-groups and adds them in a further launch, by SmallW kind: 8 - 9 us before
// anything is multiplied.
static double sliced_us(int kind, int64_t batch, int64_t M, int64_t N, int64_t K) {
  const double g = (double)batch * (double)M * (double)N * (double)K * 1e-9, g32 = (double)batch * (double)ceil_div(M, (int64_t)32) * 32.0 * (double)N * (double)K * 1e-9;
  const double nk = (double)batch * (double)N * (double)K * 1e-6, mn = (double)batch * (double)M * (double)N * 1e-6, k = (double)K * 1e-3;
  const double tiles_k = (double)batch * (double)ceil_div(M, (int64_t)128) * (double)ceil_div(N, (int64_t)128) * (double)K * 1e-6;
  switch (kind) {
    case 0: return 8.4 + 0.12 * g + 0.065 * nk + 8.7 * mn + 0.12 * k + 0.65 * g32;
    case 1: return 8.6 + 1.84 * g + 0.073 * nk + 0.97 * mn + 0.073 * k + 1.08 * g32;
    case 2: return 8.3 + 0.049 * nk + 2.2 * mn + 0.17 * k + 2.9 * g32 + 10.9 * tiles_k;
    default: return 8.9 + 2.5 * g + 4.7 * mn + 0.24 * k + 6.2 * tiles_k;
  }
}
// One launch over all of K, or slices of it?  By both estimates (on rows of up to 64 stages 0.91 and 1.0 x what is measured, 13 - 14 % rms); longer rows stay with the
// slices, which they make too dear.  On 3284 random [N, K] 16-bit products that have a cut 2.2 % behind the faster of the two, 2.8 % by a bar of 0.82 on rows of any length
// (496 x 2496 x 11520 47 us in slices, 73 in one launch, which that took; 1111 x 240 x 2496 10.0 in one launch, 13.8 in slices).
static bool tiles_beat_slices(TileKind tile, int kind, int64_t M, int64_t N, int64_t K, int64_t k_bytes) {
  return M > 32 && k_bytes <= 64 * kStageBytes && tile_choice(tile, 1, M, N, k_bytes).us < 0.9 * sliced_us(kind, 1, M, N, K);
}
static double plain_nk_us(int64_t M, int64_t N, int64_t K) {  // one 16-bit matrix of [N, K] weights
  if (f16_split_choice(1, M, N, K) > 1 && !tiles_beat_slices(kTileF16NK, 2, M, N, K, K * 2)) return sliced_us(2, 1, M, N, K);
  return tile_choice(kTileF16NK, 1, M, N, K * 2).us;
}
// The products that may take the small-tile kernel: weights as stored (the first four: SmallW), int32 results, or rescaled ones
// (W8A8), W4A8 where the caller brought the room to unpack the weights first (65 to 256 rows: above, that is what runs; the figures
// below count such problems of any number of rows).
enum SmallUse { kUseI8NK = kSmallNK, kUseI8KN = kSmallKN8, kUseF16KN = kSmallKN16, kUseW4A8 = kSmallW4, kUseW4A8TwoSteps = 4, kUseW8A8NK = 5, kUseW8A8KN = 6,
                // the two of W4A8 with weights multiplied as 16 times their value
                kUseW4A8Times16 = 7, kUseW4A8TwoStepsTimes16 = 8 };
static SmallW small_weights(SmallUse use) {
  return use == kUseW8A8NK ? kSmallNK : use == kUseW8A8KN ? kSmallKN8 : use == kUseW4A8TwoSteps || use >= kUseW4A8Times16 ? kSmallW4 : (SmallW)use;
}
static SmallUse w4a8_use(bool two_steps, int sign_mode, int64_t K) {
  if (small_w4a8_times16(sign_mode, K)) return two_steps ? kUseW4A8TwoStepsTimes16 : kUseW4A8Times16;
  return two_steps ? kUseW4A8TwoSteps : kUseW4A8;
}
// Is the small-tile kernel ahead of what would run in its place?  Two things its own estimate leaves out come on top: the activations' trip from
// memory (at 2.5 TB/s: every tile of weight rows asks for them again) and, with 16-bit weights, that theirs cannot take less than
// a copy.  The other side, by what would run: calls that cut K into slices over work-groups (sliced_us), up to 32 rows a fit to the 32-row
// tiles, else the tiles' own estimates -- plain, of the ring kernel, 256 x 256 --, for W4A8 in two steps behind the unpack pass.
//   * The ring kernel, one round of its tiles: what the small-tile kernel takes is fitted anew (330 - 520 problems per use, those weighted where the two
//     are within 1.7 x); the choice is 0.7 - 1.1 % behind the faster of the two on average, more than 5 % on 15 - 31 of them (with bars of 0.88 - 1.2 on its own
//     estimate 2 - 4 % and 23 - 97).  Behind the unpack pass, and W4A8 by itself, as before.
//   * Up to 32 rows and slices keep bars that were fitted to kernels which are still those that run there; on 190 of those problems 1 % behind.
//   * Rows of one to three stages and more than one round of the ring kernel's tiles: against the estimate of what runs, the rescaled products at 0.9 and 0.95 of it (they store
//     their tiles row by row: 224 x 3216 x 256 [N, K] 7.9 against 5.6 us).  On 2445 random problems of one to three stages 0.7 % behind the faster of the two on average.
struct SmallBars {
  double few_sliced, sliced, few, plain;
  // against the ring kernel: what the small-tile kernel takes, launch + scale x its estimate + trip x the activations' trip + step x stages + out x
  // millions of outputs + weights x millions of weights
  double launch, scale, trip, step, out, weights;
};
static constexpr SmallBars kSmallBars[9] = {
    // <= 32 rows, K slices   K slices   <= 32 rows   tiles   the ring kernel
    {0.84, 1.5, 1.15, 1.0, -1.54, 0.922, 1.03, 0.040, 0.0, 0.0},  // int8 [N, K]
    {0.74, 1.05, 1.05, 1.0, -0.67, 0.815, 0.09, 0.102, 0.0, 0.0},  // int8 [K, N]
    {0.8, 1.04, 1.02, 1.0, 0.55, 0.577, 0.0, 0.071, 1.5, 0.296},    // 16-bit [K, N]
    {1.04, 1.0, 0.93, 1.0, 0.0, 1.08, 1.08, 0.0, 0.0, 0.0},       // W4A8
    {1.04, 1.0, 0.93, 1.0, 0.0, 1.0, 1.0, 0.0, 0.0, 0.0},          // W4A8 in two steps
    {0.84, 0.95, 1.12, 0.9, -1.53, 1.026, 1.0, 0.025, 0.0, 0.0},   // W8A8 [N, K]
    {0.74, 0.9, 1.0, 0.95, -0.52, 0.868, 0.36, 0.093, 0.0, 0.0},   // W8A8 [K, N]
    {1.04, 1.0, 0.93, 1.0, 0.0, 1.08, 1.08, 0.0, 0.0, 0.0},       // W4A8 times 16
    {1.04, 1.0, 0.93, 1.0, 0.0, 1.0, 1.0, 0.0, 0.0, 0.0}};         // the same in two steps
static bool small_tile_wins(const SmallTile& t, SmallUse use, int64_t batch, int64_t M, int64_t N, int64_t K) {
  if (!t.ok || small_tile_forced()) return t.ok;
  const SmallW w = small_weights(use);
  const SmallBars& bar = kSmallBars[use];
  const double g = (double)batch * (double)M * (double)N * (double)K * 1e-9, g32 = (double)batch * (double)ceil_div(M, (int64_t)32) * 32.0 * (double)N * (double)K * 1e-9;
  const double nk = (double)batch * (double)N * (double)K * 1e-6, mn = (double)batch * (double)M * (double)N * 1e-6, k = (double)K * 1e-3;
  const int64_t k_bytes = w == kSmallKN16 ? 2 * K : K, stages = ceil_div(k_bytes, (int64_t)kStageBytes);
  const double trip_us = (double)batch * (double)M * (double)k_bytes / 2.5e6;
  double us = t.us + trip_us;
  if (w == kSmallKN16 && us < 1.05 * nk * 2.0 / 5.0) us = 1.05 * nk * 2.0 / 5.0;
  const bool packed = w == kSmallW4;
  const TileKind tile = w == kSmallKN16 ? kTileF16KN : w == kSmallKN8 ? kTileI8KN : kTileI8NK;
  const bool adds = use == kUseI8NK || use == kUseI8KN;  // (their slices add into the result itself)
  if (packed ? M <= 256 && slice_choice(M, N, k_bytes, true, 2.5, 0) > 1
             : batch == 1 && slice_choice(M, N, k_bytes, !adds, 1.0, 0) > 1 && !tiles_beat_slices(tile, w, M, N, K, k_bytes))
    return us < (M <= 32 ? bar.few_sliced : bar.sliced) * sliced_us(w, batch, M, N, K);
  if (packed && use != kUseW4A8TwoSteps && use != kUseW4A8TwoStepsTimes16) return us < bar.few * (4.9 + 0.069 * nk + 1.44 * mn + 5.7 * k + 0.69 * g32);
  if (M <= 32 && w == kSmallNK) return us < bar.few * (5.1 + 1.4 * g + 0.16 * mn + 2.07 * k);
  if (M <= 32 && w == kSmallKN8) return us < bar.few * (4.8 + 1.22 * g + 0.078 * nk + 0.3 * mn + 2.4 * k + 0.38 * g32);
  if (M <= 32 && w == kSmallKN16) return us < bar.few * (3.8 + 0.08 * nk + 0.6 * mn + 9.4 * k + 12.8 * (double)batch * (double)ceil_div(N, (int64_t)128) * (double)K * 1e-6);
  const double unpack_us = packed ? 2.6 + nk * 1.5 / 4.5 : 0.0;
  if (packed && i8_split_choice(1, M, N, K, false) > 1 && !tiles_beat_slices(kTileI8NK, 0, M, N, K, K))
    return us < bar.sliced * (unpack_us + 2.0 * sliced_us(0, 1, M, N, K));  // (slices that add into the result take twice those with matrices of their own)
  const double mine = bar.launch + bar.scale * t.us + bar.trip * trip_us + bar.step * (double)stages + bar.out * mn + bar.weights * nk;
  const double ring_us = one_round_ring(tile, batch, M, N, k_bytes).us;
  return ring_us > 0.0 ? mine < unpack_us + ring_us : mine < bar.plain * (unpack_us + tile_choice(tile, batch, M, N, k_bytes).us);
}
static SmallTile small_tile_for_i8(int64_t batch, int64_t M, int64_t N, int64_t K, SmallUse use) {
  const SmallTile t{false, 0, 0, 0, 0.0};
  if (batch < 1 || M < 1 || N < 1 || K < 128 || K % 128 != 0 || M >= kMaxDim || N >= kMaxDim || K >= kMaxDim || g_i8_tile || g_i8_split) return t;
  static thread_local PlanTable<SmallTile> known;
  return known.get(M, N, K, use + 16 * batch, [&] {
    SmallTile p = small_tile_plan(use >= kUseW4A8Times16 ? (int)kSmallW4Times16 : (int)small_weights(use), batch, M, N, K);
    p.ok = small_tile_wins(p, use, batch, M, N, K);
    return p;
  });
}
static SmallTile small_tile_for_f16(int64_t batch, int64_t M, int64_t N, int64_t K, int b_layout) {
  const SmallTile t{false, 0, 0, 0, 0.0};
  if (b_layout != TLQ_B_KN || batch < 1 || M < 1 || N < 1 || K < 64 || K % 64 != 0 || N % 8 != 0 || M >= kMaxDim || N >= kMaxDim || K >= kMaxDim || g_gemm_f16_tile || g_gemm_slots == 2)
    return t;
  static thread_local PlanTable<SmallTile> known;
  return known.get(M, N, K, batch, [&] {
    SmallTile p = small_tile_plan(2, batch, M, N, K * 2);
    p.ok = small_tile_wins(p, kUseF16KN, batch, M, N, K);
    return p;
  });
}

// A product whose last round of work-groups is nearly empty runs as two launches: the rows of the tiles that fill whole rounds, then
// the rest by whatever is best for that many rows.  Returns the rows of the first, 0 = one launch.  (4099 rows on 4096 x 4096 int8 are 17 x 16
// tiles of 256 x 256, a round of 256 and one of 16; one launch took 128 x 128 tiles instead, 96 us; 4096 rows and 3 take
// 62 us.)  Not on rows of fewer than six 128-byte stages, where a launch more is a larger part than the 1.5 us below: 300 random problems
// that two launches were estimated to win ran, against one, 0.93 as fast on rows of one to three stages (25 of 33 more than 3 % behind;
// int8 7314 x 2384 x 384 26.7 us for 22.6), 1.01 on four or five (8 of 30 behind), 1.06 on six or seven (1 of 14), 1.1 on eight to
// fifteen (2 of 55) and 1.2 beyond (none of 168).  The tiles between 128 x 128 and 256 x 256 (gemm_core.h) fill most of those rounds in one launch: they are
// taken where they are estimated to be 12 % ahead of two launches.  (Within that both are about level, 4099 x 4096 x 1024 int8 28.3 us in one launch and 26.2 in two; a test
// of the two launches names 7314 x 2384 x 768, 23.5 and 27.4.)
static int64_t rows_of_full_rounds(TileKind kind, int64_t M, int64_t N, int64_t K) {
  if (M <= 512 || N < 256 || K % 128 != 0 || M >= kMaxDim || N >= kMaxDim || K >= kMaxDim || g_gemm_groups || g_gemm_f16_tile || g_i8_tile || g_gemm_slots == 2) return 0;
  static thread_local PlanTable<int64_t> known;
  return known.get(M, N, K, kind + 4 * (g_i8_split != 0), [&]() -> int64_t {  // (forced K slices: small_tile_for_i8 refuses the rest)
    const bool i8 = kind >= kTileI8KN;
    const int64_t k_bytes = i8 ? K : 2 * K, stages = k_bytes / kStageBytes, cus = cu_count_or_default();
    if (stages < 6) return 0;
    auto one_us = [&](int64_t rows) { return tile_choice(kind, 1, rows, N, k_bytes).us; };
    auto rest_us = [&](int64_t rows) {
      const double us = one_us(rows);
      if (kind == kTileF16NK) return us;
      const SmallTile t = i8 ? small_tile_for_i8(1, rows, N, K, kind == kTileI8NK ? kUseI8NK : kUseI8KN) : small_tile_for_f16(1, rows, N, K, TLQ_B_KN);
      return t.ok && t.us < us ? t.us : us;
    };
    // (in one launch the tiles in between fill the rounds as a rule; only the others are asked whether two are ahead of them, and those tiles whether
    // they are ahead of both)
    const double between_us = 1.13 * one_us(M);
    double best = 0.97 * tile_choice(kind, 1, M, N, k_bytes, -1).us;
    if (between_us < best) best = between_us;
    int64_t head = 0;
    for (const int64_t tile : {(int64_t)256, (int64_t)128}) {
      const int64_t across = ceil_div(N, tile), round = tile == 256 ? cus : 2 * cus, rounds = ceil_div(M, tile) * across / round;
      const int64_t rows = rounds * round / across * tile;
      if (rounds == 0 || rows <= 0 || rows >= M) continue;
      const double us = one_us(rows) + 1.5 + rest_us(M - rows);
      if (us < best) best = us, head = rows;
    }
    return head;
  });
}

int tlq_gemm_f16_batched(const void* A, const void* B, void* C, int64_t batch, int64_t M, int64_t N, int64_t K, int in_dtype,
                         int out_dtype, int b_layout, void* stream) {
  TLQ_CHECK_DIMS("tlq_gemm_f16");
  TLQ_REQUIRE(batch >= 0 && batch < kMaxDim, "tlq_gemm_f16: bad batch %lld", (long long)batch);
  TLQ_REQUIRE(in_dtype == TLQ_F16 || in_dtype == TLQ_BF16, "tlq_gemm_f16: in_dtype must be float16 or bfloat16 (got %d)",
              in_dtype);
  TLQ_REQUIRE(out_dtype == TLQ_F16 || out_dtype == TLQ_BF16 || out_dtype == TLQ_F32, "tlq_gemm_f16: bad out_dtype %d",
              out_dtype);
  TLQ_REQUIRE(b_layout == TLQ_B_KN || b_layout == TLQ_B_NK, "tlq_gemm_f16: bad b_layout %d", b_layout);
  if (batch == 0 || M == 0 || N == 0) return 0;
  TLQ_REQUIRE(K > 0 && K % 8 == 0, "tlq_gemm_f16: K=%lld must be a positive multiple of 8", (long long)K);
  TLQ_REQUIRE(N % 8 == 0, "tlq_gemm_f16: N=%lld must be a multiple of 8", (long long)N);
  TLQ_REQUIRE(A && B && C, "tlq_gemm_f16: null pointer");
  TLQ_REQUIRE(aligned16(A) && aligned16(B) && aligned16(C), "tlq_gemm_f16: pointers must be 16-byte aligned");
  TLQ_REQUIRE(fits32(M, K * 2) && fits32(N, K * 2), "tlq_gemm_f16: a matrix spans 4 GiB or more");
  TLQ_REQUIRE(batch == 1 || (((M * K) % 8 == 0) && ((M * N) % 8 == 0)),
              "tlq_gemm_f16: every matrix of a batch must start on a 16-byte boundary (M*K and M*N multiples of 8)");
  if (const SmallTile t = small_tile_for_f16(batch, M, N, K, b_layout); t.ok) return small_f16(t, A, B, C, batch, M, N, K, in_dtype, out_dtype, (hipStream_t)stream);
  if (const int64_t head = batch == 1 ? rows_of_full_rounds(b_layout == TLQ_B_NK ? kTileF16NK : kTileF16KN, M, N, K) : 0; head > 0) {
    if (const int rc = tlq_gemm_f16_batched(A, B, C, 1, head, N, K, in_dtype, out_dtype, b_layout, stream)) return rc;
    return tlq_gemm_f16_batched((const uint8_t*)A + head * K * 2, B, (uint8_t*)C + head * N * (out_dtype == TLQ_F32 ? 4 : 2), 1, M - head, N, K, in_dtype, out_dtype, b_layout,
                                stream);
  }
  return gemm_f16_plain(A, B, C, batch, M, N, K, in_dtype, out_dtype, b_layout, (hipStream_t)stream);
}

int tlq_gemm_f16(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K, int in_dtype, int out_dtype,
                 int b_layout, void* stream) {
  return tlq_gemm_f16_batched(A, B, C, 1, M, N, K, in_dtype, out_dtype, b_layout, stream);
}

int64_t tlq_f16_workspace_bytes(int64_t batch, int64_t M, int64_t N, int64_t K) {
  if (batch != 1 || M <= 0 || N <= 0 || K <= 0 || M >= kMaxDim || N >= kMaxDim || K >= kMaxDim || N % 8 != 0) return 0;
  const int split = f16_split_choice(batch, M, N, K);
  return split > 1 ? (int64_t)split * M * N * 4 : 0;
}

int tlq_gemm_f16_ws(const void* A, const void* B, void* C, void* workspace, int64_t workspace_bytes, int64_t batch, int64_t M,
                    int64_t N, int64_t K, int in_dtype, int out_dtype, int b_layout, void* stream) {
  // One batch, few activation rows: K slices write fp32 matrices into the workspace, a second pass adds them in slice
  // order and rounds once.  As many slices as the workspace holds; none, or a shape that is not cut: tlq_gemm_f16_batched.
  int split = 1;
  if (tlq_f16_workspace_bytes(batch, M, N, K) > 0 && workspace != nullptr && aligned16(workspace)) {
    split = f16_split_choice(batch, M, N, K);
    while (split > 1 && (int64_t)split * M * N * 4 > workspace_bytes) split /= 2;
  }
  if (g_f16_split == 0 && split > 1 && (small_tile_for_f16(batch, M, N, K, b_layout).ok || tiles_beat_slices(b_layout == TLQ_B_NK ? kTileF16NK : kTileF16KN, 2, M, N, K, K * 2)))
    split = 1;
  if (split <= 1) return tlq_gemm_f16_batched(A, B, C, batch, M, N, K, in_dtype, out_dtype, b_layout, stream);
  TLQ_REQUIRE(in_dtype == TLQ_F16 || in_dtype == TLQ_BF16, "tlq_gemm_f16_ws: in_dtype must be float16 or bfloat16 (got %d)",
              in_dtype);
  TLQ_REQUIRE(out_dtype == TLQ_F16 || out_dtype == TLQ_BF16 || out_dtype == TLQ_F32, "tlq_gemm_f16_ws: bad out_dtype %d",
              out_dtype);
  TLQ_REQUIRE(b_layout == TLQ_B_KN || b_layout == TLQ_B_NK, "tlq_gemm_f16_ws: bad b_layout %d", b_layout);
  TLQ_REQUIRE(A && B && C, "tlq_gemm_f16_ws: null pointer");
  TLQ_REQUIRE(aligned16(A) && aligned16(B) && aligned16(C), "tlq_gemm_f16_ws: pointers must be 16-byte aligned");
  TLQ_REQUIRE(fits32(M, K * 2) && fits32(N, K * 2), "tlq_gemm_f16_ws: a matrix spans 4 GiB or more");
  return gemm_f16_slices(A, B, C, (float*)workspace, M, N, K, split, in_dtype, out_dtype, b_layout, (hipStream_t)stream);
}

void tlq_tune_f16_split(int slices) { tlq::tuning_changed(), g_f16_split = slices; }
int tlq_debug_f16_split(int64_t M, int64_t N, int64_t K) { return f16_split_choice(1, M, N, K); }

int tlq_gemm_f16_splitk(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K, int64_t split_k,
                        int in_dtype, int b_layout, void* stream) {
  TLQ_CHECK_DIMS("tlq_gemm_f16_splitk");
  TLQ_REQUIRE(in_dtype == TLQ_F16 || in_dtype == TLQ_BF16,
              "tlq_gemm_f16_splitk: in_dtype must be float16 or bfloat16 (got %d)", in_dtype);
  TLQ_REQUIRE(b_layout == TLQ_B_KN || b_layout == TLQ_B_NK, "tlq_gemm_f16_splitk: bad b_layout %d", b_layout);
  TLQ_REQUIRE(split_k >= 1 && split_k <= 1024, "tlq_gemm_f16_splitk: split_k=%lld out of range 1..1024", (long long)split_k);
  if (M == 0 || N == 0) return 0;
  TLQ_REQUIRE(K > 0 && K % split_k == 0 && (K / split_k) % 8 == 0,
              "tlq_gemm_f16_splitk: K=%lld must split into %lld slices of a multiple of 8", (long long)K, (long long)split_k);
  TLQ_REQUIRE(N % 8 == 0, "tlq_gemm_f16_splitk: N=%lld must be a multiple of 8", (long long)N);
  TLQ_REQUIRE(A && B && C, "tlq_gemm_f16_splitk: null pointer");
  TLQ_REQUIRE(aligned16(A) && aligned16(B) && aligned16(C), "tlq_gemm_f16_splitk: pointers must be 16-byte aligned");
  TLQ_REQUIRE(fits32(M, K * 2) && fits32(N, K * 2), "tlq_gemm_f16_splitk: a matrix spans 4 GiB or more");
  return gemm_f16_splitk(A, B, (float*)C, M, N, K, split_k, in_dtype, b_layout, (hipStream_t)stream);
}

int tlq_gemm_i8(const void* A, const void* B, void* C, int64_t batch, int64_t M, int64_t N, int64_t K, int b_layout,
                void* stream) {
  TLQ_CHECK_DIMS("tlq_gemm_i8");
  TLQ_REQUIRE(batch >= 0 && batch < kMaxDim, "tlq_gemm_i8: bad batch %lld", (long long)batch);
  TLQ_REQUIRE(b_layout == TLQ_B_KN || b_layout == TLQ_B_NK, "tlq_gemm_i8: bad b_layout %d", b_layout);
  if (batch == 0 || M == 0 || N == 0) return 0;
  TLQ_REQUIRE(K > 0 && K % 16 == 0, "tlq_gemm_i8: K=%lld must be a positive multiple of 16", (long long)K);
  TLQ_REQUIRE(N % 16 == 0, "tlq_gemm_i8: N=%lld must be a multiple of 16", (long long)N);
  TLQ_REQUIRE(A && B && C, "tlq_gemm_i8: null pointer");
  TLQ_REQUIRE(aligned16(A) && aligned16(B) && aligned16(C), "tlq_gemm_i8: pointers must be 16-byte aligned");
  TLQ_REQUIRE(fits32(M, K) && fits32(N, K), "tlq_gemm_i8: a matrix spans 4 GiB or more");
  if (const SmallTile t = small_tile_for_i8(batch, M, N, K, b_layout == TLQ_B_NK ? kUseI8NK : kUseI8KN); t.ok) return small_i8(t, A, B, C, batch, M, N, K, b_layout, (hipStream_t)stream);
  // few activation rows: K slices add into C itself (int32, exact in any order)
  if (const int split = i8_split_choice(batch, M, N, K, false);
      split > 1 && (g_i8_split || !tiles_beat_slices(b_layout == TLQ_B_NK ? kTileI8NK : kTileI8KN, b_layout == TLQ_B_NK ? 0 : 1, M, N, K, K)))
    return gemm_i8_i32_splitk(A, B, (int32_t*)C, M, N, K, split, b_layout, (hipStream_t)stream);
  if (const int64_t head = batch == 1 ? rows_of_full_rounds(b_layout == TLQ_B_NK ? kTileI8NK : kTileI8KN, M, N, K) : 0; head > 0) {
    if (const int rc = tlq_gemm_i8(A, B, C, 1, head, N, K, b_layout, stream)) return rc;
    return tlq_gemm_i8((const uint8_t*)A + head * K, B, (int32_t*)C + head * N, 1, M - head, N, K, b_layout, stream);
  }
  return gemm_i8_i32(A, B, C, batch, M, N, K, b_layout, (hipStream_t)stream);
}

int tlq_gemm_w4a8(const void* A, const void* w_packed, void* C, int64_t M, int64_t N, int64_t K, int sign_mode,
                  void* stream) {
  TLQ_CHECK_DIMS("tlq_gemm_w4a8");
  TLQ_REQUIRE(sign_mode >= TLQ_U4 && sign_mode <= TLQ_S4_OFFSET7, "tlq_gemm_w4a8: bad sign_mode %d", sign_mode);
  if (M == 0 || N == 0) return 0;
  TLQ_REQUIRE(K > 0 && K % 32 == 0, "tlq_gemm_w4a8: K=%lld must be a positive multiple of 32", (long long)K);
  TLQ_REQUIRE(N % 4 == 0, "tlq_gemm_w4a8: N=%lld must be a multiple of 4", (long long)N);
  TLQ_REQUIRE(A && w_packed && C, "tlq_gemm_w4a8: null pointer");
  TLQ_REQUIRE(aligned16(A) && aligned16(w_packed) && aligned16(C), "tlq_gemm_w4a8: pointers must be 16-byte aligned");
  TLQ_REQUIRE(fits32(M, K) && fits32(N, K / 2), "tlq_gemm_w4a8: a matrix spans 4 GiB or more");
  if (const SmallTile t = small_tile_for_i8(1, M, N, K, w4a8_use(false, sign_mode, K)); t.ok) return small_w4a8(t, A, w_packed, C, M, N, K, sign_mode, (hipStream_t)stream);
  // few activation rows: K slices add into C (int32, exact in any order)
  if (const int split = i8_split_choice(1, M, N, K, false, 2.5); split > 1)
    return gemm_w4a8_i32_splitk(A, w_packed, C, M, N, K, sign_mode, split, nullptr, (hipStream_t)stream);
  return gemm_w4a8_i32(A, w_packed, C, M, N, K, sign_mode, (hipStream_t)stream);
}

static thread_local int g_w4a8_ws_mode = 0;  // tlq_tune_w4a8_ws: 0 = automatic, 1 = K slices in the workspace, 2 = unpack + int8 GEMM

int tlq_gemm_w4a8_ws(const void* A, const void* w_packed, void* workspace, int64_t workspace_bytes, void* C, int64_t M,
                     int64_t N, int64_t K, int sign_mode, void* stream) {
  // The reference's int8 [N, K] workspace is used in one of two ways.  Many activation rows: the reference's own two
  // steps -- unpack into the workspace, int8 GEMM on it -- each at its own roofline (M = N = K = 4096: 6 + 66 us against
  // 98 us fused; M = 1024: 37 against 65 us).  Few rows (the unpack pass would cost more than the GEMM): the kernel that
  // unpacks on the way into LDS over K slices, the workspace holding one int32 [M, N] matrix per slice.
  const bool usable = workspace != nullptr && aligned16(workspace) && N > 0 && K > 0 && M > 0 && M < kMaxDim && N < kMaxDim &&
                      K < kMaxDim && fits32(N, K / 2) && fits32(M, K);
  const bool two_steps = usable && workspace_bytes >= N * K && K % 16 == 0 && N % 16 == 0 && fits32(N, K) &&
                         (M > 64 || g_w4a8_ws_mode == 2);
  // (above 256 rows the caller finds the unpacked weights in a workspace that holds them, also where the small-tile kernel is faster)
  if (g_w4a8_ws_mode == 0 && !(two_steps && M > 256) && small_tile_for_i8(1, M, N, K, w4a8_use(two_steps, sign_mode, K)).ok)
    return tlq_gemm_w4a8(A, w_packed, C, M, N, K, sign_mode, stream);
  if (usable && K % 32 == 0 && N % 4 == 0 && g_w4a8_ws_mode != 2 && (M <= 256 || g_w4a8_ws_mode == 1)) {
    int split = i8_split_choice(1, M, N, K, true, 2.5);
    while (split > 1 && (int64_t)split * M * N * 4 > workspace_bytes) split /= 2;
    if (split > 1) {
      TLQ_REQUIRE(sign_mode >= TLQ_U4 && sign_mode <= TLQ_S4_OFFSET7, "tlq_gemm_w4a8_ws: bad sign_mode %d", sign_mode);
      TLQ_REQUIRE(A && w_packed && C && aligned16(A) && aligned16(w_packed) && aligned16(C),
                  "tlq_gemm_w4a8_ws: null or misaligned pointer");
      return gemm_w4a8_i32_splitk(A, w_packed, C, M, N, K, sign_mode, split, (int32_t*)workspace, (hipStream_t)stream);
    }
  }
  if (!two_steps) return tlq_gemm_w4a8(A, w_packed, C, M, N, K, sign_mode, stream);
  TLQ_REQUIRE(sign_mode >= TLQ_U4 && sign_mode <= TLQ_S4_OFFSET7, "tlq_gemm_w4a8_ws: bad sign_mode %d", sign_mode);
  TLQ_REQUIRE(A && w_packed && C && aligned16(w_packed), "tlq_gemm_w4a8_ws: null or misaligned pointer");
  if (int rc = tlq_unpack_int4(w_packed, workspace, N, K, TLQ_I8, sign_mode, stream)) return rc;
  return tlq_gemm_i8(A, workspace, C, 1, M, N, K, TLQ_B_NK, stream);
}

void tlq_tune_w4a8_ws(int mode) { g_w4a8_ws_mode = mode; }

int tlq_gemm_w8a8(const void* A, const void* B, const void* scale_a, const void* scale_b, void* C, int64_t batch,
                  int64_t M, int64_t N, int64_t K, int64_t n_scale_b, int b_layout, int out_dtype, void* stream) {
  TLQ_CHECK_DIMS("tlq_gemm_w8a8");
  TLQ_REQUIRE(batch >= 0 && batch < kMaxDim, "tlq_gemm_w8a8: bad batch %lld", (long long)batch);
  TLQ_REQUIRE(b_layout == TLQ_B_KN || b_layout == TLQ_B_NK, "tlq_gemm_w8a8: bad b_layout %d", b_layout);
  TLQ_REQUIRE(out_dtype == TLQ_F16 || out_dtype == TLQ_BF16 || out_dtype == TLQ_F32, "tlq_gemm_w8a8: bad out_dtype %d",
              out_dtype);
  if (batch == 0 || M == 0 || N == 0) return 0;
  TLQ_REQUIRE(K > 0 && K % 16 == 0, "tlq_gemm_w8a8: K=%lld must be a positive multiple of 16", (long long)K);
  TLQ_REQUIRE(N % 16 == 0, "tlq_gemm_w8a8: N=%lld must be a multiple of 16", (long long)N);
  TLQ_REQUIRE(scale_b == nullptr || n_scale_b == 1 || n_scale_b == N,
              "tlq_gemm_w8a8: n_scale_b=%lld must be 1 or N=%lld", (long long)n_scale_b, (long long)N);
  TLQ_REQUIRE(A && B && C, "tlq_gemm_w8a8: null pointer");
  TLQ_REQUIRE(aligned16(A) && aligned16(B) && aligned16(C), "tlq_gemm_w8a8: pointers must be 16-byte aligned");
  TLQ_REQUIRE(((uintptr_t)scale_a & 3) == 0 && ((uintptr_t)scale_b & 3) == 0, "tlq_gemm_w8a8: scales misaligned");
  TLQ_REQUIRE(fits32(M, K) && fits32(N, K), "tlq_gemm_w8a8: a matrix spans 4 GiB or more");
  if (const SmallTile t = small_tile_for_i8(batch, M, N, K, b_layout == TLQ_B_NK ? kUseW8A8NK : kUseW8A8KN); t.ok)
    return small_w8a8(t, A, B, scale_a, scale_b, C, batch, M, N, K, n_scale_b, b_layout, out_dtype, (hipStream_t)stream);
  if (const int64_t head = batch == 1 ? rows_of_full_rounds(b_layout == TLQ_B_NK ? kTileI8NK : kTileI8KN, M, N, K) : 0; head > 0) {
    if (const int rc = tlq_gemm_w8a8(A, B, scale_a, scale_b, C, 1, head, N, K, n_scale_b, b_layout, out_dtype, stream)) return rc;
    return tlq_gemm_w8a8((const uint8_t*)A + head * K, B, scale_a ? (const float*)scale_a + head : nullptr, scale_b,
                         (uint8_t*)C + head * N * (out_dtype == TLQ_F32 ? 4 : 2), 1, M - head, N, K, n_scale_b, b_layout, out_dtype, stream);
  }
  return gemm_w8a8_rescale(A, B, scale_a, scale_b, C, batch, M, N, K, n_scale_b, b_layout, out_dtype,
                           (hipStream_t)stream);
}

static bool w8a8_dims_split(int64_t batch, int64_t M, int64_t N, int64_t K) {
  return batch == 1 && M > 0 && N > 0 && K > 0 && M < kMaxDim && N < kMaxDim && K < kMaxDim && K % 16 == 0 && N % 16 == 0 &&
         fits32(M, K) && fits32(N, K);
}

int64_t tlq_w8a8_workspace_bytes(int64_t batch, int64_t M, int64_t N, int64_t K) {
  if (!w8a8_dims_split(batch, M, N, K)) return 0;
  const int split = i8_split_choice(batch, M, N, K, true);
  return split > 1 ? (int64_t)split * M * N * 4 : 0;
}

int tlq_gemm_w8a8_ws(const void* A, const void* B, const void* scale_a, const void* scale_b, void* C, void* workspace,
                     int64_t workspace_bytes, int64_t batch, int64_t M, int64_t N, int64_t K, int64_t n_scale_b,
                     int b_layout, int out_dtype, void* stream) {
  // One batch, few activation rows: K slices write their int32 tiles into the workspace, a second pass sums and
  // rescales them into C (the reference's own two steps, example_quant_batch_matmul.py:42,66-68, with a matrix per slice).
  int split = 1;
  if (w8a8_dims_split(batch, M, N, K) && workspace != nullptr && aligned16(workspace)) {
    split = i8_split_choice(batch, M, N, K, true);
    while (split > 1 && (int64_t)split * M * N * 4 > workspace_bytes) split /= 2;  // as many slices as the workspace holds
  }
  if (split <= 1 || small_tile_for_i8(batch, M, N, K, b_layout == TLQ_B_NK ? kUseW8A8NK : kUseW8A8KN).ok ||
      (!g_i8_split && tiles_beat_slices(b_layout == TLQ_B_NK ? kTileI8NK : kTileI8KN, b_layout == TLQ_B_NK ? 0 : 1, M, N, K, K)))
    return tlq_gemm_w8a8(A, B, scale_a, scale_b, C, batch, M, N, K, n_scale_b, b_layout, out_dtype, stream);
  TLQ_REQUIRE(b_layout == TLQ_B_KN || b_layout == TLQ_B_NK, "tlq_gemm_w8a8_ws: bad b_layout %d", b_layout);
  TLQ_REQUIRE(out_dtype == TLQ_F16 || out_dtype == TLQ_BF16 || out_dtype == TLQ_F32, "tlq_gemm_w8a8_ws: bad out_dtype %d",
              out_dtype);
  TLQ_REQUIRE(scale_b == nullptr || n_scale_b == 1 || n_scale_b == N,
              "tlq_gemm_w8a8_ws: n_scale_b=%lld must be 1 or N=%lld", (long long)n_scale_b, (long long)N);
  TLQ_REQUIRE(A && B && C, "tlq_gemm_w8a8_ws: null pointer");
  TLQ_REQUIRE(aligned16(A) && aligned16(B) && aligned16(C), "tlq_gemm_w8a8_ws: pointers must be 16-byte aligned");
  TLQ_REQUIRE(((uintptr_t)scale_a & 3) == 0 && ((uintptr_t)scale_b & 3) == 0, "tlq_gemm_w8a8_ws: scales misaligned");
  return gemm_w8a8_rescale_splitk(A, B, scale_a, scale_b, C, (int32_t*)workspace, M, N, K, n_scale_b, split, b_layout,
                                  out_dtype, (hipStream_t)stream);
}

}  // extern "C"
