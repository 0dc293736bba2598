// MFMA GEMM over a ring of K stages, for few tiles: launches that give each CU one work-group at most, as a rule (tile_choice in gemm_core.h).
//
// What bounds such a launch (one work-group per CU) is what a CU takes in: a 128 x 128 tile pulls 32 KB per 128-byte stage of K, and a work-group with one stage
// in flight gets 55 KB per us, with two or more 90 - 97 (direct loads alone, 256 work-groups, row pitches of 4 - 16 KB; one stage of
// 256 rows on either side: 66 - 71).  So LDS is a ring of four stages: while stage s is multiplied, s + 1 has landed and s + 2 .. s + 3 or s + 4
// (addr::ring_ahead) are on their way, and the waits count loads instead of draining them.
//   * Two groups of four wavefronts (2 x 2 over the tile) take one MFMA k-step of every stage each, so that every SIMD has two wavefronts and a
//     fragment that is read from LDS still feeds a tile of half the work-group's rows and columns; the groups' sums meet in LDS at the end.
//   * The fragments of stage s + 1 are read into a second register set while stage s is multiplied.  A slot is therefore free one
//     barrier after its stage was read: the barrier at the top of iteration s frees the slot of stage s for stage s + 4.
//   * One barrier per stage: behind it every wavefront's loads of stage s + 1 have landed, and everyone has read stage s.
//   * The loads and the fragment reads of a stage stand between its products.  Issued together behind the barrier, the loads of eight
//     wavefronts hold the issue of all of them until the address unit has taken the last one: 989 cycles a stage instead of 706 of
//     which the products are 523 (128 x 128 tiles, fp16, by the shader's clock).  No more is asked for ahead of the first product than the lead.
// fp16 1000 x 4096 x 4096: 39.5 us with the groups on parts of K in two stages each, which drained the loads in every stage; 37.6 with the ring, 33.6 with
// the loads between the products, 32.9 with a lead of four stages for five.  Over that earlier kernel, the better tile of either, 615 problems: 1.04 x on 4 - 6 stages,
// 1.06 - 1.09 on 7 - 16, 1.17 on 17 - 24, 1.22 beyond.  What is left is power: with the loads between the products the part runs at 1.50 GHz, without the loads at 1.83, without the fragment reads at 1.62,
// the products alone at 1.97 (60, 46, 52 and 38 us of a 64 us call).
#pragma once
#include "gemm_core.h"

namespace tlq {

// Part h of every wavefront tile (tile rows h TH .. h TH + TH - 1) is group h's to write: the other groups leave theirs in LDS,
// [h][from][wave][TN][TH][64 lanes], and group h adds the KG of them in the order of the groups (its own, from its registers,
// among them).  smem: free once every wavefront is here.
template <class Epi, int TM, int TN, int KG, int WAVES, class acc_t>
__device__ __forceinline__ void add_groups_and_write(const Epi& epi, acc_t (&acc)[TN][TM], uint8_t* smem, int group, int wave, int lane, int m_base,
                                                     int n_base, int M, int N) {
  static_assert(TM % KG == 0, "whole tile rows per group");
  constexpr int TH = TM / KG, PART = TN * TH * 64;
  acc_t* const sums = (acc_t*)smem + lane;
  auto part_of = [&](int h, int from) { return ((h * (KG - 1) + (from < h ? from : from - 1)) * WAVES + wave) * PART; };
  __syncthreads();
#pragma unroll
  for (int h = 0; h < KG; ++h)
    if (h != group)
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int t = 0; t < TH; ++t) sums[part_of(h, group) + (tn * TH + t) * 64] = acc[tn][h * TH + t];
  __syncthreads();
  acc_t own[TN][TH];
#pragma unroll
  for (int h = 0; h < KG; ++h)
    if (h == group)
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int t = 0; t < TH; ++t) {
          acc_t sum = h == 0 ? acc[tn][h * TH + t] : sums[part_of(h, 0) + (tn * TH + t) * 64];
#pragma unroll
          for (int from = 1; from < KG; ++from) sum += from == h ? acc[tn][h * TH + t] : sums[part_of(h, from) + (tn * TH + t) * 64];
          own[tn][t] = sum;
        }
  if constexpr (Epi::STAGED) __syncthreads();
  write_tile<Epi, TH, TN>(epi, own, smem + (group * WAVES + wave) * (TH * 16 * kStageBytes), lane, m_base + group * (TH * 16), n_base, M, N);
}

template <int BM, int BN>
struct RingCfg {
  static constexpr int SLOT = (BM + BN) * kStageBytes;
  static constexpr int S = addr::kRingSlots;
  static constexpr int LDS = S * SLOT;
  static constexpr int TM = BM / 32, TN = BN / 32;  // MFMA tiles of a wavefront: 2 x 2 wavefronts in either group
  static_assert(S == 4 && LDS <= 160 * 1024, "slot of stage s: s % 4");
  static_assert(4 * TM * TN * 1024 <= LDS && 8 * (TM / 2) * 16 * kStageBytes <= LDS, "the groups' sums and the staging areas fit the ring");
};

// KT: whole stages (at least one); band_and_tail: 2 x the tile rows of a band, + 1 where a partial stage follows
template <class Mma, class AL, class WL, class Epi, int BM, int BN>
__global__ __launch_bounds__(512, 2) void ring_gemm_mfma_kernel(typename AL::Params pa, typename WL::Params pw, typename Epi::Params pe, int M, int N,
                                                               int KT, int blocks, int band_and_tail) {
  typedef RingCfg<BM, BN> Cfg;
  typedef typename Mma::acc_t acc_t;
  constexpr int S = Cfg::S, TM = Cfg::TM, TN = Cfg::TN;
  constexpr int LOADS = AL::PER_WAVE + WL::PER_WAVE;  // direct loads per wavefront and stage
  static_assert(AL::DIRECT && WL::DIRECT && LOADS * (S - 1) <= 63, "the waits count direct loads");
  extern __shared__ __align__(16) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wave_all >> 2, wave = wave_all & 3;  // group: this wavefront's MFMA k-step of every stage
  const int wave_m0 = (wave & 1) * (BM / 2), wave_n0 = (wave >> 1) * (BN / 2);
  const TileCoord tc = tile_of_block<BM, BN>(blocks, M, N, band_and_tail >> 1);
  AL al(pa, tc.batch, tc.m0, M, tid);
  WL wl(pw, tc.batch, tc.n0, N, tid);
  typename AL::Regs ra;
  typename WL::Regs rw;
  const typename AL::Frag fragA(lane, wave_m0);
  const typename WL::Frag fragW(lane, wave_n0);
  acc_t acc[TN][TM];
#pragma unroll
  for (int tn = 0; tn < TN; ++tn)
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) acc[tn][tm] = acc_t{0, 0, 0, 0};

  uint4_t af[2][TM], wf[2][TN];  // fragments by parity of the stage
  auto issue = [&](int s, int slot) {
    uint8_t* const base = smem + slot * Cfg::SLOT;
    al.template gload<false>(ra, s, base);
    wl.template gload<false>(rw, s, base + BM * kStageBytes);
  };
  auto read = [&](auto par, int slot) {
    constexpr int P = decltype(par)::value;
    const uint8_t* const base = smem + slot * Cfg::SLOT;
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) wf[P][tn] = fragW.read(base + BM * kStageBytes, group, tn);
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) af[P][tm] = fragA.read(base, group, tm);
  };
  // One stage: the products of the fragments of parity P, with the reads of the next stage's (READ, from `slot`) and the loads of
  // stage `ahead` (LOAD, into `free_slot`) between them.
  auto run_stage = [&](auto par, auto read_tag, auto load_tag, int slot, int ahead, int free_slot) {
    constexpr int P = decltype(par)::value, Q = 1 - P;
    constexpr bool READ = decltype(read_tag)::value, LOAD = decltype(load_tag)::value;
    constexpr int PRODUCTS = TN * TM, READS = TN + TM;
    const uint8_t* const from = smem + slot * Cfg::SLOT;
    const uint8_t *src_a = nullptr, *src_w = nullptr;
    uint32_t dst_a = 0, dst_w = 0;
    if constexpr (LOAD) {
      uint8_t* const to = smem + free_slot * Cfg::SLOT;
      src_a = al.stage_src(ahead), src_w = wl.stage_src(ahead);
      dst_a = al.stage_dst(to), dst_w = wl.stage_dst(to + BM * kStageBytes);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < PRODUCTS; ++i) {
      acc[i / TM][i % TM] = Mma::mma(wf[P][i / TM], af[P][i % TM], acc[i / TM][i % TM]);
      if constexpr (READ) {
#pragma unroll
        for (int r = 0; r < READS; ++r)
          if (r * 3 * PRODUCTS / (4 * READS) == i) {  // (over the first three quarters: they are waited for at the end)
            if (r < TN)
              wf[Q][r] = fragW.read(from + BM * kStageBytes, group, r);
            else
              af[Q][r - TN] = fragA.read(from, group, r - TN);
          }
      }
      if constexpr (LOAD) {
#pragma unroll
        for (int j = 0; j < LOADS; ++j)
          if ((2 * j + 1) * PRODUCTS / (2 * LOADS) == i) {
            if (j < AL::PER_WAVE)
              al.load_one(j, src_a, dst_a);
            else
              wl.load_one(j - AL::PER_WAVE, src_w, dst_w);
          }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  typedef std::integral_constant<int, 0> Even;
  typedef std::false_type No;
  auto wait_but = [&](auto stages) {
    if constexpr (std::is_same<decltype(stages), int>::value) {
      switch (stages) {
#define TLQ_WAIT(n) \
  case n: asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LOADS * (n)) : "memory"); break;
        TLQ_WAIT(1) TLQ_WAIT(2) TLQ_WAIT(3)
#undef TLQ_WAIT
        default: asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      }
    } else {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LOADS * decltype(stages)::value) : "memory");
    }
  };
  auto run = [&](auto ahead_tag) {
    constexpr int D = decltype(ahead_tag)::value;
    addr::ring_schedule<D>(
        KT, [&](int s) { issue(s, s); }, wait_but, [] { __syncthreads(); }, [&] { read(Even{}, 0); },
        [&](auto parity, auto reads, auto loads, int s) { run_stage(parity, reads, loads, (s + 1) & (S - 1), s + D, (s + D) & (S - 1)); });
  };
  if (addr::ring_ahead(KT) == 3)
    run(std::integral_constant<int, 3>{});
  else
    run(std::integral_constant<int, 4>{});
  if (band_and_tail & 1) {  // the partial stage, with zeros past K: through registers into slot 0 (every load has landed, every fragment is read)
    __syncthreads();
    al.template gload<true>(ra, KT, smem);
    wl.template gload<true>(rw, KT, smem + BM * kStageBytes);
    al.lstore(ra, smem);
    wl.lstore(rw, smem + BM * kStageBytes);
    __syncthreads();
    read(Even{}, 0);
    run_stage(Even{}, No{}, No{}, 0, 0, 0);
  }
  const Epi epi(pe, tc.batch);
  add_groups_and_write<Epi, TM, TN, 2, 4>(epi, acc, smem, group, wave, lane, tc.m0 + wave_m0, tc.n0 + wave_n0, M, N);
}

template <class Mma, class AL, class WL, class Epi, int BM, int BN>
int launch_ring(const typename AL::Params& pa, const typename WL::Params& pw, const typename Epi::Params& pe, int64_t batch, int64_t M, int64_t N,
                int64_t k_bytes, hipStream_t st, const char* what, int band_rows) {
  auto kern = ring_gemm_mfma_kernel<Mma, AL, WL, Epi, BM, BN>;
  constexpr int lds_bytes = RingCfg<BM, BN>::LDS;
  static bool attr_set = false;  // per instantiation; idempotent, so a race only repeats the call
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (e != hipSuccess) {
      set_error("%s: cannot reserve %d bytes of LDS: %s", what, lds_bytes, hipGetErrorString(e));
      return 1;
    }
    attr_set = true;
  }
  const int64_t tiles_m = ceil_div(M, (int64_t)BM), tiles_n = ceil_div(N, (int64_t)BN), blocks = batch * tiles_m * tiles_n;
  if (blocks <= 0) return 0;
  if (blocks > 0x7fffffff || k_bytes < kStageBytes) {
    set_error("%s: %lld tiles, %lld bytes of K", what, (long long)blocks, (long long)k_bytes);
    return 1;
  }
  kern<<<(unsigned)blocks, 512, lds_bytes, st>>>(pa, pw, pe, (int)M, (int)N, (int)(k_bytes / kStageBytes), (int)blocks,
                                       2 * (g_gemm_band_rows > 0 ? g_gemm_band_rows : band_rows) + (k_bytes % kStageBytes != 0));
  char detail[96] = "";
  if (launch_log_on()) snprintf(detail, sizeof(detail), "ring_gemm_mfma_kernel %dx%d tiles, %d stages, K in groups of wavefronts", BM, BN, RingCfg<BM, BN>::S);
  return check_launch(what, detail) ? 0 : 1;
}

}  // namespace tlq
