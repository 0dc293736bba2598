// MFMA GEMM of 256 x 256 output tiles on FOUR wavefronts, one per SIMD, each with 128 x 128 outputs and the full register file.
//
// What bounds large products is power: with all CUs multiplying the clock falls until the part stays in its limit, so that a cycle in
// which nothing is multiplied costs leakage and clock, and an operand that is read twice costs its energy.  Against the two-stage kernel of eight
// wavefronts (gemm_core.h):
//   * 128 x 128 outputs a wavefront read a third less from LDS per product than 128 x 64; accumulators fill the accumulation registers, and two
//     sets of fragments the others: those of the next k-step are read between the products of this one.
//   * Loads, fragment reads and address arithmetic stand between the products, one at a time (with one wavefront per SIMD nothing else would fill the
//     matrix pipeline meanwhile).  Compiled, a stage is 128 MFMAs and some 110 other instructions.
//   * LDS is five slots of one operand tile and stage.  One barrier per stage, half way through it: in front of it a wavefront has read all
//     of stage s, behind it stage s + 1 has landed, W(s + 2) is loaded into the slot of A(s), and A(s + 3) into that of W(s).
//   * One work-group per CU takes tile after tile.  The loads ahead run on into the next tile, whose first stages land while this one is finished and
//     stored through the slot that is free just then.  Nothing drains them: the row and column scales of a rescaled result are asked for in one go at a
//     tile's start and taken when its first stage has landed (value by value, with a drain of all loads and stores ahead of the first, and another
//     ahead of the first output, int8 8 x 2048 x 4096 x 4096 took 230 for 227.6 us, 4099 x 4096 x 4096 with the quantiser 70.7 for 70.1).
// bf16 8192 x 14336 x 4096 755 -> 647 us with weights [K, N], 720 -> 631 (1.52 PFLOP/s; vendor library 623 - 632) with [N, K]; 4096^3 102 -> 91; fp16 8192 x
// 4096 x 14336 770 -> 672; int8 8 x 2048 x 4096 x 4096 263 -> 241 (2.28 POP/s).  A work-group per tile instead, with the same loop: 8192 x 8192 x 512
// bf16 76.7 against 69.3, 8192 x 14336 x 4096 653 against 647.
#pragma once
#include "gemm_core.h"

namespace tlq {

// The MFMA as an instruction of its own with the accumulator as an in-out operand in the accumulation registers: left to the compiler, 256
// accumulators spread over both halves of the register file and spill in the main loop.
template <class Mma>
struct QuadMma;
#define TLQ_QUAD_MMA(MMA, INSTRUCTION)                                                                        \
  template <>                                                                                                 \
  struct QuadMma<MMA> {                                                                                       \
    static __device__ __forceinline__ void mma(const uint4_t& a, const uint4_t& b, typename MMA::acc_t& c) {  \
      asm volatile(INSTRUCTION " %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));                                 \
    }                                                                                                         \
    static __device__ __forceinline__ void first(const uint4_t& a, const uint4_t& b, typename MMA::acc_t& c) { \
      asm volatile(INSTRUCTION " %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));                                  \
    }                                                                                                         \
  };
TLQ_QUAD_MMA(MmaF16, "v_mfma_f32_16x16x32_f16")
TLQ_QUAD_MMA(MmaBF16, "v_mfma_f32_16x16x32_bf16")
TLQ_QUAD_MMA(MmaI8, "v_mfma_i32_16x16x64_i8")
#undef TLQ_QUAD_MMA

template <int I, int N, typename F>
__device__ __forceinline__ void quad_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    quad_for<I + 1, N>(f);
  }
}

// KT: stages of 128 bytes of K, whole ones, at least two.  The launch's `grid` work-groups (one to a CU) take tiles blockIdx.x, + grid, ... of `tiles`.
template <class Mma, class WL, class Epi>
__global__ __launch_bounds__(256, 1) void quad_gemm_mfma_kernel(typename RowLoaderDirect<256, 256>::Params pa, typename WL::Params pw, typename Epi::Params pe,
                                                               int M, int N, int KT, int tiles, int grid, int band_rows) {
  constexpr int T = 8, TILE = 256 * kStageBytes;  // MFMA tiles of a wavefront per side; one operand, one stage: 32 KB
  typedef RowLoaderDirect<256, 256> AL;
  static_assert(AL::PER_WAVE == addr::kQuadLoads && WL::PER_WAVE == addr::kQuadLoads && WL::DIRECT, "the waits count the direct loads per wavefront and tile");
  extern __shared__ __align__(16) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave_m0 = (wave & 1) * 128, wave_n0 = (wave >> 1) * 128;
  int tile = blockIdx.x;
  TileCoord tc = tile_of_index<256, 256>(tile, tiles, M, N, band_rows);
  AL al(pa, tc.batch, tc.m0, M, tid);
  WL wl(pw, tc.batch, tc.n0, N, tid);
  const RowFrag fragA(lane, wave_m0);
  const typename WL::Frag fragW(lane, wave_n0);
  typename Mma::acc_t acc[T][T];
  uint4_t af[2][T], wf[2][T];  // fragments by k-step of a stage
  uint8_t* slot[5];  // (addr::quad_tile)
#pragma unroll
  for (int i = 0; i < 5; ++i) slot[i] = smem + i * TILE;
  // The 64 products of k-step KS; between them the reads of the next k-step's fragments from (ra, rw) and the eight loads of stage s of an operand.
  auto phase = [&](auto ks_tag, auto first_tag, const uint8_t* ra, const uint8_t* rw, const auto& loader, int s, uint8_t* to) {
    constexpr int KS = decltype(ks_tag)::value, OTHER = 1 - KS;
    constexpr bool FIRST = decltype(first_tag)::value;
    const uint8_t* const src = loader.stage_src(s);
    const uint32_t dst = loader.stage_dst(to);
    __builtin_amdgcn_sched_barrier(0);
    quad_for<0, T * T>([&](auto ic) {
      constexpr int i = decltype(ic)::value, tn = i / T, tm = i % T;
      if constexpr (FIRST)
        QuadMma<Mma>::first(wf[KS][tn], af[KS][tm], acc[tn][tm]);
      else
        QuadMma<Mma>::mma(wf[KS][tn], af[KS][tm], acc[tn][tm]);
      if constexpr (i % 3 == 1 && i / 3 < 2 * T) {
        constexpr int r = i / 3;  // in the order of their first use
        if constexpr (r == 0)
          wf[OTHER][0] = fragW.read(rw, OTHER, 0);
        else if constexpr (r <= T)
          af[OTHER][r - 1] = fragA.read(ra, OTHER, r - 1);
        else
          wf[OTHER][r - T] = fragW.read(rw, OTHER, r - T);
      }
      // (the second phase's loads are waited for a stage on, the first phase's half a stage later than that; those of a tile's first phase behind it)
      constexpr bool EARLY = KS == 1 || FIRST;
      if constexpr (EARLY ? i % 4 == 2 && i < 32 : i % 8 == 6) loader.load_one(EARLY ? i / 4 : i / 8, src, dst);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  auto wait = [&](auto left) { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(left)::value) : "memory"); };
  auto barrier = [] { __syncthreads(); };

  addr::quad_start(
      slot,
      [&](auto operand, int s, uint8_t* to) {
        auto all = [&](const auto& loader) {
          const uint8_t* const src = loader.stage_src(s);
          const uint32_t dst = loader.stage_dst(to);
#pragma unroll
          for (int j = 0; j < 8; ++j) loader.load_one(j, src, dst);
        };
        if constexpr (decltype(operand)::value == 0) all(al); else all(wl);
      },
      wait, barrier,
      [&](const uint8_t* a, const uint8_t* w) {
        wf[0][0] = fragW.read(w, 0, 0);
#pragma unroll
        for (int t = 0; t < T; ++t) af[0][t] = fragA.read(a, 0, t);
#pragma unroll
        for (int t = 1; t < T; ++t) wf[0][t] = fragW.read(w, 0, t);
      });
  for (;;) {
    const Epi epi(pe, tc.batch);
    const int m_base = tc.m0 + wave_m0, n_base = tc.n0 + wave_n0;
    auto out_scales = fetch_scales<Epi, T, T>(epi, m_base, n_base, lane, M, N);
    tile += grid;
    const bool more = tile < tiles;
    addr::quad_tile(
        KT, slot,
        [&] {  // (behind the last tile the loads are those of its first stages again, for nobody)
          if (!more) return;
          tc = tile_of_index<256, 256>(tile, tiles, M, N, band_rows);
          al = AL(pa, tc.batch, tc.m0, M, tid);
          wl = WL(pw, tc.batch, tc.n0, N, tid);
        },
        [&](auto ks, auto first, const uint8_t* ra, const uint8_t* rw, int s, uint8_t* to) {
          if constexpr (decltype(ks)::value == 0) phase(ks, first, ra, rw, al, s, to); else phase(ks, first, ra, rw, wl, s, to);
        },
        [&](auto left) {
          wait(left);
          if constexpr (decltype(left)::value == 0) out_scales.arrive();  // (the scales are among it; waited for at their use, they would drain the next tile's loads)
        },
        barrier);
    // (the wait states between the last MFMAs, which the compiler does not know for what they are, and the first instruction that reads an accumulator)
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    // the free slot was read for the last time in front of the last barrier: the output staging area, 8 KB for each wavefront
    write_tile_with<Epi, T, T, T / 2>(epi, out_scales, acc, slot[4] + wave * (T / 2 * 16 * kStageBytes), lane, m_base, n_base, M, N);
    if (!more) break;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __syncthreads();  // the next loads overwrite it
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no direct load outlives the work-group
}

// k_bytes (bytes of K per activation row): a multiple of 128, two or more
template <class Mma, class WL, class Epi>
int launch_quad(const typename RowLoaderDirect<256, 256>::Params& pa, const typename WL::Params& pw, const typename Epi::Params& pe, int64_t batch, int64_t M,
                int64_t N, int64_t k_bytes, hipStream_t st, const char* what, int band_rows) {
  auto kern = quad_gemm_mfma_kernel<Mma, WL, Epi>;
  constexpr int lds_bytes = 5 * 256 * kStageBytes;
  static bool attr_set = false;  // per instantiation; idempotent, so a race only repeats the call
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (e != hipSuccess) {
      set_error("%s: cannot reserve %d bytes of LDS: %s", what, lds_bytes, hipGetErrorString(e));
      return 1;
    }
    attr_set = true;
  }
  const int64_t tiles = batch * ceil_div(M, (int64_t)256) * ceil_div(N, (int64_t)256);
  if (tiles <= 0) return 0;
  if (tiles > 0x3fffffff || k_bytes < 2 * kStageBytes || k_bytes % kStageBytes != 0) {
    set_error("%s: %lld tiles, %lld bytes of K", what, (long long)tiles, (long long)k_bytes);
    return 1;
  }
  int cus = tlq_device_cu_count();
  if (cus <= 0) cus = 256;
  const int grid = (int)(tiles < cus ? tiles : cus);
  kern<<<grid, 256, lds_bytes, st>>>(pa, pw, pe, (int)M, (int)N, (int)(k_bytes / kStageBytes), (int)tiles, grid, g_gemm_band_rows > 0 ? g_gemm_band_rows : band_rows);
  return check_launch(what, "quad_gemm_mfma_kernel 256x256 tiles, four wavefronts") ? 0 : 1;
}

}  // namespace tlq
