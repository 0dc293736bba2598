// Per-token (per-row) int8 activation quantiser, the step that feeds the W8A8 matmuls:
//   amax[m]  = max(max_n |x[m, n]|, 1e-4)
//   scale[m] = amax / 127                      (round_scale: the next power of two, 2^ceil(log2(amax / 127)))
//   y[m, n]  = int8( rint( clamp(x[m, n] / scale[m], -127, 127) ) )      rint = round half to even
// HBM bound: one wavefront (many rows) or one work-group (long rows) owns a row, reads it once into registers with 16-byte
// loads, reduces the maximum across lanes, and writes 8 int8 per lane and chunk.  Few long rows are shared by work-groups, each of
// which reads the whole row.  Rows longer than 32768 values, or of a length that is no multiple of 8, are read twice.
#include <type_traits>

#include "tlq_common.h"

namespace tlq {

template <>
__device__ __forceinline__ float to_float<float>(float v) {
  return v;
}

// Eight consecutive values, kept as loaded (16 or 32 bytes) and widened to float on use.  The input is read once:
// non-temporal loads (M = 16384, N = 4096: 38.2 instead of 40.0 us; with the resident grid 36.1 us) -- but for load_shared, whose
// values other work-groups read too.  The output is
// stored normally: non-temporal stores save another microsecond here and cost the W8A8 GEMM that reads the output next
// 4 - 14 us (16384 x 4096 x 4096: quantiser + GEMM 291 against 279 us).
template <typename T>
struct Raw8;
template <>
struct Raw8<half_t> {
  half8_t v;
  __device__ __forceinline__ void load(const half_t* p) { v = __builtin_nontemporal_load((const half8_t*)p); }
  __device__ __forceinline__ void load_shared(const half_t* p) { v = *(const half8_t*)p; }
  __device__ __forceinline__ float get(int i) const { return (float)v[i]; }
};
template <>
struct Raw8<bf16_t> {
  uint32_t w[4];
  __device__ __forceinline__ void load(const bf16_t* p) {
    const uint4_t q = __builtin_nontemporal_load((const uint4_t*)p);
    w[0] = q.x, w[1] = q.y, w[2] = q.z, w[3] = q.w;
  }
  __device__ __forceinline__ void load_shared(const bf16_t* p) {
    const uint4_t q = *(const uint4_t*)p;
    w[0] = q.x, w[1] = q.y, w[2] = q.z, w[3] = q.w;
  }
  __device__ __forceinline__ float get(int i) const {
    return bitcast<float>((i & 1) ? (w[i >> 1] & 0xffff0000u) : (w[i >> 1] << 16));
  }
};
template <>
struct Raw8<float> {
  float4_t a, b;
  __device__ __forceinline__ void load(const float* p) {
    a = __builtin_nontemporal_load((const float4_t*)p);
    b = __builtin_nontemporal_load((const float4_t*)(p + 4));
  }
  __device__ __forceinline__ void load_shared(const float* p) { a = *(const float4_t*)p, b = *(const float4_t*)(p + 4); }
  __device__ __forceinline__ float get(int i) const { return i < 4 ? a[i] : b[i - 4]; }
};

__device__ __forceinline__ float wave_max(float v) {
  // a row of 16 lanes inside the vector unit (lanes swapped in pairs, in fours, halves of a row and rows mirrored), then rows and halves
  // of the wavefront swapped: no trip through LDS
  auto dpp = [&](auto ctrl) { v = fmaxf(v, bitcast<float>(__builtin_amdgcn_update_dpp(0, bitcast<int>(v), decltype(ctrl)::value, 0xf, 0xf, false))); };
  dpp(std::integral_constant<int, 0xb1>{}), dpp(std::integral_constant<int, 0x4e>{}), dpp(std::integral_constant<int, 0x141>{}), dpp(std::integral_constant<int, 0x140>{});
  const auto rows = __builtin_amdgcn_permlane16_swap(bitcast<uint32_t>(v), bitcast<uint32_t>(v), false, false);
  v = fmaxf(bitcast<float>((uint32_t)rows[0]), bitcast<float>((uint32_t)rows[1]));
  const auto halves = __builtin_amdgcn_permlane32_swap(bitcast<uint32_t>(v), bitcast<uint32_t>(v), false, false);
  return fmaxf(bitcast<float>((uint32_t)halves[0]), bitcast<float>((uint32_t)halves[1]));
}

__device__ __forceinline__ float row_scale(float amax, int round_scale) {
  amax = fmaxf(amax, 1e-4f);
  const float s = amax / 127.0f;
  if (!round_scale) return s;
  // 2^ceil(log2(s)) from the bits of s: exponent, plus one when any mantissa bit is set
  const uint32_t bits = bitcast<uint32_t>(s);
  const int e = (int)((bits >> 23) & 0xff) - 127 + ((bits & 0x7fffffu) ? 1 : 0);
  return bitcast<float>((uint32_t)(e + 127) << 23);
}

// x / scale, correctly rounded wherever the quotient matters, from the row's reciprocal
// rcp = fl(1 / scale): q0 = x * rcp is within an ulp, the remainder x - q0 * scale is exact in one
// fma, and one more fma lands on the correctly rounded quotient.  (Only when the remainder
// underflows, |x| < 2^-100 or so, can the last bit differ; such quotients round to 0 either way.)
__device__ __forceinline__ uint32_t quant1(float x, float scale, float rcp) {
  const float q0 = x * rcp;
  const float q1 = __builtin_fmaf(__builtin_fmaf(-q0, scale, x), rcp, q0);
  // bounded (NaN becomes the lower bound), then to the nearest even whole number by the addition, which leaves its two's complement in
  // the low byte
  return bitcast<uint32_t>(__builtin_amdgcn_fmed3f(q1, -127.0f, 127.0f) + 12582912.0f);
}

template <typename R>
__device__ __forceinline__ uint2_t quant8(const R& r, float scale, float rcp) {
  uint2_t o;
  auto four = [&](int i) {
    const uint32_t lo = __builtin_amdgcn_perm(quant1(r.get(i + 1), scale, rcp), quant1(r.get(i), scale, rcp), 0x0c0c0400u);
    return __builtin_amdgcn_perm(__builtin_amdgcn_perm(quant1(r.get(i + 3), scale, rcp), quant1(r.get(i + 2), scale, rcp), 0x0c0c0400u), lo, 0x05040100u);
  };
  o.x = four(0), o.y = four(4);
  return o;
}

// N % 8 == 0.  WPR wavefronts of a 256-lane work-group share one row (1: four rows per work-group,
// 4: one row); a lane keeps CH chunks of 8 values, so the row length is at most 512 * WPR * CH.
template <typename T, int CH, int WPR>
__global__ __launch_bounds__(256) void act_quant_rows_kernel(const T* __restrict__ X, int8_t* __restrict__ Y,
                                                            float* __restrict__ S, int64_t M, int N, int round_scale, int blocks) {
  __shared__ float part[2][4];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  constexpr int RPB = 4 / WPR;  // rows per work-group
  const int sub = WPR == 1 ? 0 : wv, lanes = 64 * WPR;
  const int chunks = N >> 3;
  int it = 0;
  // every wavefront of a work-group runs the same number of iterations (the barrier below needs that)
  for (int64_t m0 = (int64_t)blockIdx.x * RPB; m0 < M; m0 += (int64_t)blocks * RPB, it ^= 1) {
    const int64_t m = m0 + (WPR == 1 ? wv : 0);
    const bool live = m < M;
    const T* x = X + m * N;
    Raw8<T> r[CH];
    float amax = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int ci = c * lanes + sub * 64 + lane;
      if (live && ci < chunks) {
        r[c].load(x + ci * 8);
#pragma unroll
        for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(r[c].get(i)));
      }
    }
    amax = wave_max(amax);
    if constexpr (WPR > 1) {
      if (lane == 0) part[it][wv] = amax;
      __syncthreads();  // part[] alternates between iterations, so one barrier per row is enough
      amax = fmaxf(fmaxf(part[it][0], part[it][1]), fmaxf(part[it][2], part[it][3]));
    }
    const float scale = row_scale(amax, round_scale);
    const float rcp = 1.0f / scale;
    if (live && lane == 0 && sub == 0) S[m] = scale;
    int8_t* y = Y + m * N;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int ci = c * lanes + sub * 64 + lane;
      if (live && ci < chunks) {
        *(uint2_t*)(y + ci * 8) = quant8(r[c], scale, rcp);  // plain store: the GEMM that follows finds the output in the last-level cache
      }
    }
  }
}

// Few long rows: `parts` work-groups (grid y) per row.  Each reads the whole row for its maximum -- from a cache for all but the first: the
// last-level one, or L2 where M is a multiple of eight and the row's work-groups land on one XCD (32 x 14336 2.97 us, 31 rows 3.50) --, two
// vector instructions a value, and quantises chunks part, part + parts, ... of 8 values, ten instructions a value, one or two chunks per lane.  WHOLE: one
// work-group per row (more rows than half the CUs), which quantises the chunks that it holds (256 x 14336 3.95 -> 3.74 us, 512 x 14336 6.7 -> 6.45
// against loading them once more).  One work-group per row left seven of eight CUs idle at M = 32 and each of its lanes 56 values of both kinds:
// 32 x 14336 bf16 4.1 -> 2.9 us, 128 x 16384 7.1 -> 3.6, 256 x 14336 7.1 -> 4.6 and, on rows of one chunk per lane, 512 x 4096 3.9 -> 3.4 (back to
// back in a graph); from three rows per CU on it is level, from four long ones behind (1000 x 14336 11.2 against 11.6).
template <typename T, int CH, int OC, bool WHOLE>
__global__ __launch_bounds__(512) void act_quant_parts_kernel(const T* __restrict__ X, int8_t* __restrict__ Y, float* __restrict__ S, int N, int round_scale, int parts) {
  __shared__ float part[8];
  const int tid = threadIdx.x, chunks = N >> 3;
  const int64_t m = blockIdx.x;
  const T* x = X + m * N;
  const int own = tid * parts + (int)blockIdx.y;  // the first of the lane's chunks
  Raw8<T> r[CH], mine[WHOLE ? 1 : OC];
#pragma unroll
  for (int c = 0; c < CH; ++c)
    if (c * 512 + tid < chunks) r[c].load_shared(x + (c * 512 + tid) * 8);
  if constexpr (!WHOLE) {
#pragma unroll
    for (int c = 0; c < OC; ++c)
      if (c * 512 * parts + own < chunks) mine[c].load_shared(x + (c * 512 * parts + own) * 8);
  }
  float amax = 0.f;
#pragma unroll
  for (int c = 0; c < CH; ++c)
    if (c * 512 + tid < chunks)
#pragma unroll
      for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(r[c].get(i)));
  amax = wave_max(amax);
  if ((tid & 63) == 0) part[tid >> 6] = amax;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 8; ++w) amax = fmaxf(amax, part[w]);
  const float scale = row_scale(amax, round_scale);
  if (tid == 0 && blockIdx.y == 0) S[m] = scale;
  const float rcp = 1.0f / scale;
  if constexpr (WHOLE) {
#pragma unroll
    for (int c = 0; c < CH; ++c)
      if (c * 512 + tid < chunks) *(uint2_t*)(Y + m * N + (c * 512 + tid) * 8) = quant8(r[c], scale, rcp);
  } else {
#pragma unroll
    for (int c = 0; c < OC; ++c)
      if (c * 512 * parts + own < chunks) *(uint2_t*)(Y + m * N + (c * 512 * parts + own) * 8) = quant8(mine[c], scale, rcp);
  }
}

// Any N: two passes over the row, one value per lane and step.
template <typename T>
__global__ __launch_bounds__(256) void act_quant_generic_kernel(const T* __restrict__ X, int8_t* __restrict__ Y,
                                                               float* __restrict__ S, int64_t M, int64_t N,
                                                               int round_scale, int blocks) {
  const int lane = threadIdx.x & 63;
  const int64_t wave = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int64_t waves = (int64_t)blocks * 4;
  for (int64_t m = wave; m < M; m += waves) {
    const T* x = X + m * N;
    float amax = 0.f;
    for (int64_t n = lane; n < N; n += 64) amax = fmaxf(amax, fabsf(to_float(x[n])));
    amax = wave_max(amax);
    const float scale = row_scale(amax, round_scale);
    if (lane == 0) S[m] = scale;
    int8_t* y = Y + m * N;
    for (int64_t n = lane; n < N; n += 64) {
      const float q = __builtin_rintf(fminf(fmaxf(to_float(x[n]) / scale, -127.0f), 127.0f));
      y[n] = (int8_t)(int)q;
    }
  }
}

template <typename T, int WPR>
static void launch_rows(const T* X, int8_t* Y, float* S, int64_t M, int N, int round_scale, int per_lane,
                        hipStream_t st) {
  // a resident grid (eight work-groups per CU: every wavefront slot) that walks the rows, instead of a work-group per
  // four rows: 37.0 instead of 40.0 us at M = 16384, N = 4096 (4 and 12 per CU are slower).  A work-group per row of at most two chunks a
  // lane is in and out too soon for that: up to four times as many, 4099 x 4096 bf16 11.05 -> 10.8 us, 8192 x 4096 20.0 -> 18.4.
  const int64_t want = ceil_div(M, (int64_t)(4 / WPR));
  int cus = tlq_device_cu_count();
  if (cus <= 0) cus = 256;
  const int64_t most = (int64_t)cus * (WPR == 4 && per_lane <= 2 ? 32 : 8);
  const int blocks = (int)(want > most ? most : want);
#define TLQ_AQ(CH) act_quant_rows_kernel<T, CH, WPR><<<blocks, 256, 0, st>>>(X, Y, S, M, N, round_scale, blocks)
  if (per_lane <= 1) TLQ_AQ(1);
  else if (per_lane <= 2) TLQ_AQ(2);
  else if (WPR == 1 || per_lane <= 4) TLQ_AQ(4);  // (one wavefront per row: at most 4, by its caller)
  else if constexpr (WPR == 4) {
    if (per_lane <= 8) TLQ_AQ(8);
    else TLQ_AQ(16);
  }
#undef TLQ_AQ
}

template <typename T>
static int run_act_quant(const void* Xv, void* Yv, void* Sv, int64_t M, int64_t N, int round_scale, hipStream_t st) {
  const T* X = (const T*)Xv;
  int8_t* Y = (int8_t*)Yv;
  float* S = (float*)Sv;
  const bool vec = N % 8 == 0 && ((uintptr_t)X & 15) == 0 && ((uintptr_t)Y & 7) == 0 && N <= 512 * 4 * 16;
  if (vec) {
    // one wavefront per row while a lane then holds at most 4 chunks and there are rows enough to fill the chip that way; otherwise the
    // four wavefronts of a work-group split the row (bf16, one wavefront against four: 8192 x 1024 6.2 / 8.6 us, 8192 x 2048 11.7 / 11.9,
    // 4099 x 4096 12.0 / 10.8, 8192 x 4096 18.9 / 18.4)
    int cus = tlq_device_cu_count();
    if (cus <= 0) cus = 256;
    int parts = 8;
    while (parts > 1 && M * parts > cus) parts /= 2;
    const int64_t chunks = N / 8;
    if (M <= (int64_t)2 * cus && N >= 4096 && chunks <= 512 * 4) {
      const dim3 grid((unsigned)M, (unsigned)parts);
#define TLQ_AQP(CH, OC, WHOLE) act_quant_parts_kernel<T, CH, OC, WHOLE><<<grid, 512, 0, st>>>(X, Y, S, (int)N, round_scale, parts)
      if (chunks <= 512)
        parts == 1 ? TLQ_AQP(1, 1, true) : TLQ_AQP(1, 1, false);
      else if (chunks <= 1024)
        parts == 1 ? TLQ_AQP(2, 2, true) : TLQ_AQP(2, 1, false);
      else
        parts == 1 ? TLQ_AQP(4, 4, true) : (parts == 2 ? TLQ_AQP(4, 2, false) : TLQ_AQP(4, 1, false));
#undef TLQ_AQP
      return check_launch("tlq_act_quant_i8", "act_quant kernel") ? 0 : 1;
    }
    const int per_lane1 = (int)ceil_div(N, (int64_t)512);
    if (per_lane1 <= 4 && M >= 4096)
      launch_rows<T, 1>(X, Y, S, M, (int)N, round_scale, per_lane1, st);
    else
      launch_rows<T, 4>(X, Y, S, M, (int)N, round_scale, (int)ceil_div(N, (int64_t)2048), st);
  } else {
    const int64_t want = ceil_div(M, (int64_t)4);
    const int blocks = (int)(want > 65536 ? 65536 : want);
    act_quant_generic_kernel<T><<<blocks, 256, 0, st>>>(X, Y, S, M, N, round_scale, blocks);
  }
  return check_launch("tlq_act_quant_i8", "act_quant kernel") ? 0 : 1;
}

}  // namespace tlq

using namespace tlq;

extern "C" int tlq_act_quant_i8(const void* X, void* Y, void* S, int64_t M, int64_t N, int in_dtype, int round_scale,
                                void* stream) {
  TLQ_REQUIRE(M >= 0 && N >= 0 && M < ((int64_t)1 << 40) && N < ((int64_t)1 << 31), "tlq_act_quant_i8: bad shape M=%lld N=%lld",
              (long long)M, (long long)N);
  TLQ_REQUIRE(in_dtype == TLQ_F16 || in_dtype == TLQ_BF16 || in_dtype == TLQ_F32,
              "tlq_act_quant_i8: in_dtype must be float16, bfloat16 or float32 (got %d)", in_dtype);
  if (M == 0) return 0;
  TLQ_REQUIRE(N > 0, "tlq_act_quant_i8: rows are empty");
  TLQ_REQUIRE(X && Y && S, "tlq_act_quant_i8: null pointer");
  TLQ_REQUIRE(((uintptr_t)S & 3) == 0 && ((uintptr_t)X & (in_dtype == TLQ_F32 ? 3 : 1)) == 0, "tlq_act_quant_i8: misaligned pointer");
  hipStream_t st = (hipStream_t)stream;
  if (in_dtype == TLQ_F16) return run_act_quant<half_t>(X, Y, S, M, N, round_scale, st);
  if (in_dtype == TLQ_BF16) return run_act_quant<bf16_t>(X, Y, S, M, N, round_scale, st);
  return run_act_quant<float>(X, Y, S, M, N, round_scale, st);
}
