// MFMA GEMM on FOUR wavefronts, one per SIMD, each with a quarter of the output tile and the full register file: tiles of 256 x 256 down to 128 x 128,
// of which two work-groups share a CU.
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
// What bounds products of a few rounds is how full the last one is, and a round's fixed part (the store of every CU's tile at once): hence the tiles between.  Per
// 128-byte stage of K and round, every CU busy, fp16 [K, N], 256 x 256 1.37 us, 192 x 256 1.15, 256 x 128 0.84, 192 x 128 0.73, two of 128 x 128 0.98 (the two-stage kernel
// 1.09; beside one work-group's store the other multiplies); fixed 6.7, 4.9, 3.0, 1.9, 2.0 us.  2159 x 2080 x 3072 fp16 44.2 -> 31.0 us in 192 x 128 tiles, int8 3428 x 1552 x 7040
// 54.4 -> 37.5, 4 x 3620 x 1312 x 9472 fp16 445 -> 327 in 192 x 256, int8 2 x 1980 x 4432 x 512 25.4 -> 20.7 in 128 x 128; 641 random problems of all operators 1.016 x faster on
// average, the 103 of them that get another kernel by it 1.11 x.
// 256 x 256: bf16 8192 x 14336 x 4096 755 -> 647 us with weights [K, N], 720 -> 631 (1.52 PFLOP/s; vendor library 623 - 632) with [N, K]; 4096^3 102 -> 91; fp16 8192 x
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
template <int BM, int BN>
struct QuadCfg {
  static constexpr int TM = BM / 32, TN = BN / 32;                      // MFMA tiles of a wavefront
  static constexpr int TILE = (BM > BN ? BM : BN) * kStageBytes;  // a slot: either operand, one stage
  static constexpr int LDS = 5 * TILE;
  static constexpr int PER_CU = 160 * 1024 / LDS;  // work-groups that share a CU
  static_assert(BM % 64 == 0 && (BN == 128 || BN == 256) && PER_CU >= 1, "even numbers of tile rows, whole lines of outputs");
};
template <class Mma, class WL, class Epi, int BM, int BN>
__global__ __launch_bounds__(256, (QuadCfg<BM, BN>::PER_CU)) void quad_gemm_mfma_kernel(typename RowLoaderDirect<BM, 256>::Params pa, typename WL::Params pw, typename Epi::Params pe,
                                                                                      int M, int N, int KT, int tiles, int grid, int band_rows) {
  constexpr int TM = QuadCfg<BM, BN>::TM, TN = QuadCfg<BM, BN>::TN, TILE = QuadCfg<BM, BN>::TILE;
  typedef RowLoaderDirect<BM, 256> AL;
  static_assert(AL::PER_WAVE == TM && WL::PER_WAVE == TN && WL::DIRECT, "the waits count the direct loads per wavefront and tile");
  extern __shared__ __align__(16) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave_m0 = (wave & 1) * (BM / 2), wave_n0 = (wave >> 1) * (BN / 2);
  int tile = blockIdx.x;
  TileCoord tc = tile_of_index<BM, BN>(tile, tiles, M, N, band_rows);
  AL al(pa, tc.batch, tc.m0, M, tid);
  WL wl(pw, tc.batch, tc.n0, N, tid);
  const RowFrag fragA(lane, wave_m0);
  const typename WL::Frag fragW(lane, wave_n0);
  typename Mma::acc_t acc[TN][TM];
  uint4_t af[2][TM], wf[2][TN];  // fragments by k-step of a stage
  uint32_t slot[5];  // offsets in LDS (addr::quad_tile; as pointers they became generic ones in the smaller tiles: flat loads, which drain the direct ones)
#pragma unroll
  for (int i = 0; i < 5; ++i) slot[i] = i * TILE;
  // The products of k-step KS; between them the reads of the next k-step's fragments from (ra, rw), over three quarters of them, and the loads of stage s
  // of an operand.
  auto phase = [&](auto ks_tag, auto first_tag, uint32_t ra, uint32_t rw, const auto& loader, int s, uint32_t to) {
    constexpr int KS = decltype(ks_tag)::value, OTHER = 1 - KS;
    constexpr bool FIRST = decltype(first_tag)::value;
    constexpr int READ_EACH = 3 * TN * TM / 4 / (TN + TM);
    // (the second phase's loads are waited for a stage on, the first phase's half a stage later than that; those of a tile's first phase behind it)
    constexpr bool EARLY = KS == 1 || FIRST;
    constexpr int LOADS = KS == 0 ? TM : TN, LOAD_EACH = TN * TM / LOADS / (EARLY ? 2 : 1), LOAD_AT = EARLY ? LOAD_EACH / 2 : LOAD_EACH - 2;
    static_assert(READ_EACH >= 1 && LOAD_EACH >= 2, "reads and loads stand between products");
    const uint8_t* const src = loader.stage_src(s);
    const uint32_t dst = loader.stage_dst(smem + to);
    __builtin_amdgcn_sched_barrier(0);
    quad_for<0, TN * TM>([&](auto ic) {
      constexpr int i = decltype(ic)::value, tn = i / TM, tm = i % TM;
      if constexpr (FIRST)
        QuadMma<Mma>::first(wf[KS][tn], af[KS][tm], acc[tn][tm]);
      else
        QuadMma<Mma>::mma(wf[KS][tn], af[KS][tm], acc[tn][tm]);
      if constexpr (i % READ_EACH == READ_EACH / 2 && i / READ_EACH < TN + TM) {
        constexpr int r = i / READ_EACH;  // in the order of their first use
        if constexpr (r == 0)
          wf[OTHER][0] = fragW.read(smem + rw, OTHER, 0);
        else if constexpr (r <= TM)
          af[OTHER][r - 1] = fragA.read(smem + ra, OTHER, r - 1);
        else
          wf[OTHER][r - TM] = fragW.read(smem + rw, OTHER, r - TM);
      }
      if constexpr (i % LOAD_EACH == LOAD_AT && i / LOAD_EACH < LOADS) loader.load_one(i / LOAD_EACH, src, dst);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  auto wait = [&](auto left) { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(left)::value) : "memory"); };
  auto barrier = [] { __syncthreads(); };

  addr::quad_start<TM, TN>(
      slot,
      [&](auto operand, int s, uint32_t to) {
        auto all = [&](const auto& loader) {
          const uint8_t* const src = loader.stage_src(s);
          const uint32_t dst = loader.stage_dst(smem + to);
#pragma unroll
          for (int j = 0; j < std::decay_t<decltype(loader)>::PER_WAVE; ++j) loader.load_one(j, src, dst);
        };
        if constexpr (decltype(operand)::value == 0) all(al); else all(wl);
      },
      wait, barrier,
      [&](uint32_t a, uint32_t w) {
        wf[0][0] = fragW.read(smem + w, 0, 0);
#pragma unroll
        for (int t = 0; t < TM; ++t) af[0][t] = fragA.read(smem + a, 0, t);
#pragma unroll
        for (int t = 1; t < TN; ++t) wf[0][t] = fragW.read(smem + w, 0, t);
      });
  for (;;) {
    const Epi epi(pe, tc.batch);
    const int m_base = tc.m0 + wave_m0, n_base = tc.n0 + wave_n0;
    auto out_scales = fetch_scales<Epi, TM, TN>(epi, m_base, n_base, lane, M, N);
    tile += grid;
    const bool more = tile < tiles;
    addr::quad_tile<TM>(
        KT, slot,
        [&] {  // (behind the last tile the loads are those of its first stages again, for nobody)
          if (!more) return;
          tc = tile_of_index<BM, BN>(tile, tiles, M, N, band_rows);
          al = AL(pa, tc.batch, tc.m0, M, tid);
          wl = WL(pw, tc.batch, tc.n0, N, tid);
        },
        [&](auto ks, auto first, uint32_t ra, uint32_t rw, int s, uint32_t to) {
          if constexpr (decltype(ks)::value == 0) phase(ks, first, ra, rw, al, s, to); else phase(ks, first, ra, rw, wl, s, to);
        },
        [&](auto left) {
          wait(left);
          if constexpr (decltype(left)::value == 0) out_scales.arrive();  // (the scales are among it; waited for at their use, they would drain the next tile's loads)
        },
        barrier);
    // (the wait states between the last MFMAs, which the compiler does not know for what they are, and the first instruction that reads an accumulator)
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    // the free slot was read for the last time in front of the last barrier: the output staging area, half a wavefront's rows for each
    static_assert(4 * (TM / 2 * 16 * kStageBytes) <= TILE, "the staging areas fit a slot");
    write_tile_with<Epi, TM, TN, TM / 2>(epi, out_scales, acc, smem + slot[4] + wave * (TM / 2 * 16 * kStageBytes), lane, m_base, n_base, M, N);
    if (!more) break;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __syncthreads();  // the next loads overwrite it
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no direct load outlives the work-group
}

// k_bytes (bytes of K per activation row): a multiple of 128, two or more
template <class Mma, class WL, class Epi, int BM = 256, int BN = 256>
int launch_quad(const typename RowLoaderDirect<BM, 256>::Params& pa, const typename WL::Params& pw, const typename Epi::Params& pe, int64_t batch, int64_t M,
                int64_t N, int64_t k_bytes, hipStream_t st, const char* what, int band_rows) {
  auto kern = quad_gemm_mfma_kernel<Mma, WL, Epi, BM, BN>;
  constexpr int lds_bytes = QuadCfg<BM, BN>::LDS;
  static bool attr_set = false;  // per instantiation; idempotent, so a race only repeats the call
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (e != hipSuccess) {
      set_error("%s: cannot reserve %d bytes of LDS: %s", what, lds_bytes, hipGetErrorString(e));
      return 1;
    }
    attr_set = true;
  }
  const int64_t tiles = batch * ceil_div(M, (int64_t)BM) * ceil_div(N, (int64_t)BN);
  if (tiles <= 0) return 0;
  if (tiles > 0x3fffffff || k_bytes < 2 * kStageBytes || k_bytes % kStageBytes != 0) {
    set_error("%s: %lld tiles, %lld bytes of K", what, (long long)tiles, (long long)k_bytes);
    return 1;
  }
  int cus = tlq_device_cu_count();
  if (cus <= 0) cus = 256;
  const int64_t places = (int64_t)cus * QuadCfg<BM, BN>::PER_CU;
  const int grid = (int)(tiles < places ? tiles : places);
  kern<<<grid, 256, lds_bytes, st>>>(pa, pw, pe, (int)M, (int)N, (int)(k_bytes / kStageBytes), (int)tiles, grid, g_gemm_band_rows > 0 ? g_gemm_band_rows : band_rows);
  char detail[96] = "";
  if (launch_log_on()) snprintf(detail, sizeof(detail), "quad_gemm_mfma_kernel %dx%d tiles, four wavefronts", BM, BN);
  return check_launch(what, detail) ? 0 : 1;
}

}  // namespace tlq
