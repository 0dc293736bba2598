// W4A16 for small and middle M (17 activation rows and more): the weights are streamed from HBM once per block of up
// to 128 activation rows, and every global access is a full-width direct global -> LDS load into a ring deep enough
// to keep the memory pipeline busy.
//
//   * A work-group of 8 wavefronts owns 32 TB activation rows (TB = 1 .. 4), 256 or 128 weight rows and a slice of K.  A wavefront owns 64
//     weight rows against all of them and half or a quarter of every step's K: two groups of four wavefronts or four of
//     two (KG), which meet in LDS at the end.  Packed weights are read from LDS as packed words and dequantised in registers right
//     into MFMA operands, no weight twice.  Four groups halve the fp32 partial sums of K slices, or need none (256 x 14336 x 4096: 47.6
//     -> 39.8 us): a slice's partial sums cost 0.4 us per MB, and 8 slices of 211 x 4096 were 14 of that call's 37 us.
//   * A step is 128 values of K: the activation tile (32 TB rows x 256 B, shared) and the packed weights (64 B a row); steps live in a
//     ring of D slots.  One barrier per step, two units before its end, publishes step s + 1 and frees step s.
//   * 32 x 32 x 16 MFMAs.  The two wavefronts of a SIMD share one issue port, which an MFMA of either shape holds for 8 cycles and a vector
//     instruction for 4 (v_fma_mixlo / mixhi_f16: 8), while the products take 32 (16) cycles of the matrix pipeline: with 16 x 16 x 32
//     operands the port is the bound, 3745 cycles a step of 128 rows against 2749 (matrix pipeline: 2048).  At full load the clock
//     gives way in turn (1.6 - 1.9 GHz): the step of 128 rows takes 1.8 us, 2.1 before.
//   * The scales and zero points of 32 weight rows are fetched 16 (KG = 2; 32 where a longer slice has room for them) or 32 groups at a time into LDS: a slice longer than that
//     runs in windows, each of which fetches its scales and restarts the ring.
// K slices write fp32 partial sums as [slice][N / 4][M][4] (two runs of 512 bytes per store), added up in slice order by
// w4a16_stream_reduce_kernel.  All together, against the kernel with 16 x 16 operands and no groups: 211 x 4096 x 11008 37.0 -> 33.0 us,
// 128 x 14336 x 4096 30.3 -> 26.3, 64 x 14336 x 4096 23.2 -> 19.6, 64 x 4096 x 14336 24.2 -> 20.4, 512 x 4096 x 4096 31.5 -> 28.2.
//
// k assignment inside a step: lane (row r32, half h) of group kg holds, at MFMA k-step t, the eight values of packed word
// 2 KT kg + KT h + t of its row (KT = 8 / KG k-steps of a wavefront); its words are contiguous bytes (one LDS read), all in one
// quantisation group (groups are >= 32 values), and the activation operand reads the 16-byte chunk of the same number.
// Weights whose 32-bit words went through interleave_weight (tilelang/quantize/utils.py:73-101, fp16 target) are taken
// as they are (LAYOUT 1): the word is still the same eight consecutive k, only the decode differs.
#include "expand8.h"
#include "gemm_core.h"
#include "stream_plan.h"

namespace tlq {

namespace {

typedef float float16_t __attribute__((ext_vector_type(16)));
template <typename T>
struct StreamMma;
template <>
struct StreamMma<half_t> {
  static __device__ __forceinline__ float16_t mma(const uint4_t& a, const uint4_t& b, const float16_t& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(bitcast<half8_t>(a), bitcast<half8_t>(b), c, 0, 0, 0);
  }
};
template <>
struct StreamMma<bf16_t> {
  static __device__ __forceinline__ float16_t mma(const uint4_t& a, const uint4_t& b, const float16_t& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(bitcast<bf16x8_t>(a), bitcast<bf16x8_t>(b), c, 0, 0, 0);
  }
};

// quantisation groups per window of a K slice: what the scale area holds (few weight rows leave room for twice as many).  A slice of several windows (`many`) takes
// twice as many of 256 weight rows too, where that leaves the ring as deep as it is: 19 of 96 random problems with 33 - 511 rows 1.05 x on average (163 x 5888 x 13952
// 48.2 -> 44.9 us, 173 x 19328 x 2688 in groups of 32 41.3 -> 36.6, 36 x 12544 x 11904 in groups of 64 44.0 -> 41.1), the others level but for one plan that this
// moves (296 x 5888 x 6656 in groups of 32 49.6 -> 50.9).
constexpr int stream_max_groups(int kg, int tb = 0, bool many = false) { return kg == 4 || (many && (tb == 2 || tb == 3)) ? 32 : 16; }

// TB: 32-row activation blocks per work-group; KG: groups of wavefronts, each with 128 / KG values of every step; MANY: several windows
template <int TB, int KG, bool MANY>
struct StreamCfg {
  static_assert(TB >= 1 && TB <= 4 && (KG == 2 || KG == 4), "32-row activation blocks and groups of wavefronts");
  static constexpr int WN = 8 / KG, BM = 32 * TB, BN = 64 * WN;
  static constexpr int T = 8 / KG;                            // k-steps of 16 values of a wavefront's share of a step
  static constexpr int NU = 2 * T;                            // units (k-step, weight tile) of a wavefront and step
  static constexpr int A_TILE = BM * 256;                     // bytes of activations per step
  static constexpr int W_TILE = BN * 64;                      // packed weights per step
  static constexpr int SLOT = A_TILE + W_TILE;
  static constexpr int MG = stream_max_groups(KG, TB, MANY);
  static constexpr int SZ = 2 * 32 * MG * 2;                  // per 32 weight rows: scales [32][MG groups], then zero points, 2 bytes each
  static constexpr int FITS = (160 * 1024 - BN / 32 * SZ) / SLOT;
  static constexpr int D = FITS > 6 ? 6 : FITS;               // ring depth, one work-group per CU
  static constexpr int RING = D * SLOT, LDS = RING + BN / 32 * SZ;
  static constexpr int LA = TB;                               // activation load instructions per wavefront and step (8 TB / 8)
  static constexpr int LW = WN / 2;                           // weight load instructions per wavefront and step (16 rows each)
  static constexpr int L = LA + LW;
  // load i of a step is issued in unit i * NU / L of the NU units that start at the barrier, two units before the step's end
  static constexpr int LB = addr::stream_loads_behind(NU, L);  // loads issued in those two
  static_assert(D >= 3 && LDS <= 160 * 1024, "rings fit the CU's LDS");
  static_assert(D * L <= 63, "vmcnt range");
  static_assert(BM * BN * 4 <= RING && (KG == 2 || 2 * BM * BN * 4 <= LDS), "the groups' exchange and the output tile fit the ring");
};
// Eight weights of a packed word.  The matrix and the vector instructions of a SIMD's wavefronts share one issue port here (an MFMA
// takes 8 cycles of it, a vector instruction 4, v_fma_mixlo / mixhi_f16 8): the binary16 weights with integer zero points are
// made with packed arithmetic on byte pairs, 16 instructions (64 cycles) against 13 with the half-rate ones (84).
struct StreamMagic : NibbleMagic {
  uint32_t m_pair, b_pair;  // the low nibble of the lower half, the high nibble of the upper half's byte, onto 1024 and 64
};
template <typename T, bool FOLD, int LAYOUT>
struct StreamExpand : Expand8<T, FOLD, LAYOUT> {
  static constexpr int INSTRUCTIONS = FOLD ? 17 : 23;
  StreamExpand() = default;
  __device__ __forceinline__ StreamExpand(T s, T z, const StreamMagic& mg) : Expand8<T, FOLD, LAYOUT>(s, z, mg) {}
};
template <int LAYOUT>
struct StreamExpand<half_t, true, LAYOUT> {
  static constexpr int INSTRUCTIONS = LAYOUT == 1 ? 13 : 16;
  half2_t s2, b_lo, b_hi, b_pair;
  StreamMagic mg;
  StreamExpand() = default;
  __device__ __forceinline__ StreamExpand(half_t s, half_t z, const StreamMagic& mg_) : mg(mg_) {
    const half_t zl = z + (half_t)1024.0f, zh = z + (half_t)64.0f;  // exact: small integers
    s2 = half2_t{s, s};
    if (LAYOUT == 1)
      b_lo = half2_t{zl, zl}, b_hi = half2_t{zh, zh};
    else
      b_pair = half2_t{zl, zh};
  }
  __device__ __forceinline__ uint4_t operator()(uint32_t v) const {
    half2_t p[4];
    if (LAYOUT == 1) {
      const uint32_t v8 = v >> 8;
      p[0] = bitcast<half2_t>(bfi(mg.m_lo, v, mg.b_lo)) - b_lo;
      p[1] = bitcast<half2_t>(bfi(mg.m_hi, v, mg.b_hi)) - b_hi;
      p[2] = bitcast<half2_t>(bfi(mg.m_lo, v8, mg.b_lo)) - b_lo;
      p[3] = bitcast<half2_t>(bfi(mg.m_hi, v8, mg.b_hi)) - b_hi;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)  // byte j in both halves: its low nibble as 1024 + u below, its high one as 64 + u above
        p[j] = bitcast<half2_t>(bfi(mg.m_pair, __builtin_amdgcn_perm(v, v, (uint32_t)j * 0x01010101u), mg.b_pair)) - b_pair;
    }
    uint4_t o;
    o.x = bitcast<uint32_t>(p[0] * s2);
    o.y = bitcast<uint32_t>(p[1] * s2);
    o.z = bitcast<uint32_t>(p[2] * s2);
    o.w = bitcast<uint32_t>(p[3] * s2);
    return o;
  }
};

template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

// MANY: the slice is longer than one window of the scale area (the common single-window case keeps the simpler control
// flow, which the compiler schedules 3 - 5 % better)
template <typename T, int TB, int KG, int LAYOUT, bool MANY>
__global__ __launch_bounds__(512, 2) void w4a16_stream_kernel(const T* __restrict__ A, const uint8_t* __restrict__ Wp,
                                                             const T* __restrict__ scales, const T* __restrict__ zeros,
                                                             void* __restrict__ C, float* __restrict__ partial, int M, int N, int K,
                                                             int gshift, float zero_scalar, int out_dtype, int slice_steps, int xcd_slices) {
  typedef StreamCfg<TB, KG, MANY> Cfg;
  typedef StreamMma<T> Mma;
  typedef __attribute__((address_space(3))) uint8_t* lptr_t;
  constexpr int D = Cfg::D, LA = Cfg::LA, WN = Cfg::WN, KT = Cfg::T, NU = Cfg::NU, MG = Cfg::MG;
  extern __shared__ __align__(16) uint8_t smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r32 = lane & 31, h = lane >> 5;
  const int kg = wave / WN, wn = wave % WN;  // values 16 KT kg .. of every step; weight rows 64 wn .. 64 wn + 63
  StreamItem item{(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z};
  if (xcd_slices) {  // the launch's K slices, where the order is by XCD
    const int nb = (N + Cfg::BN - 1) / Cfg::BN, mb = (M + Cfg::BM - 1) / Cfg::BM;
    item = stream_item(blockIdx.x + nb * (blockIdx.y + xcd_slices * blockIdx.z), nb, xcd_slices, mb, true);
  }
  const int n0 = item.n * Cfg::BN, m0 = item.m * Cfg::BM, slice = item.slice;
  const int steps_total = K >> 7;
  const int step0 = slice * slice_steps;
  const int steps = steps_total - step0 < slice_steps ? steps_total - step0 : slice_steps;
  const int groups = K >> gshift;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lptr_t)smem);

  // ---- per-lane source offsets of the direct loads (rows past the matrices are clamped; masked at the store) ----
  uint32_t voff[Cfg::L];  // the activation tile's loads, then the packed weights'
#pragma unroll
  for (int j = 0; j < Cfg::LW; ++j) {
    int n = n0 + (wave * Cfg::LW + j) * 16 + addr::sw_row(lane);
    n = n < N ? n : N - 1;
    voff[LA + j] = (uint32_t)n * (uint32_t)(K >> 1) + (uint32_t)(addr::sw_piece(lane) * 16);
  }
#pragma unroll
  for (int j = 0; j < LA; ++j) {
    const int I = j * 8 + wave;
    int m = m0 + addr::sa_row(lane, I);
    m = m < M ? m : M - 1;
    voff[j] = ((uint32_t)m * (uint32_t)K) * 2u + (uint32_t)(addr::sa_chunk(lane, I) * 16);
  }
  const uint8_t* const w_base = Wp + (int64_t)step0 * 64;
  const uint8_t* const a_base = (const uint8_t*)A + (int64_t)step0 * 256;
  auto dma16 = [&](uint32_t lds_addr, uint32_t voff, const uint8_t* sbase) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(voff), "s"(sbase) : "memory");
  };
  auto dma4 = [&](uint32_t lds_addr, uint32_t voff, const uint8_t* sbase) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds_addr), "v"(voff), "s"(sbase) : "memory");
  };
  // load i (of L) of step s of this slice into ring slot `slot`: the activation tile's, then the packed weights'.  Loads of
  // steps past `end` are issued with no lane active: they move nothing, but every step is L loads and the loop has no branch
  // that would cut the schedule.
  auto issue1 = [&](int s, int end, int slot, auto ic) {
    constexpr int i = decltype(ic)::value;
    const uint32_t l0 = lds0 + (uint32_t)(slot * Cfg::SLOT) + (uint32_t)(i < LA ? (i * 8 + wave) * 1024 : Cfg::A_TILE + (wave * Cfg::LW + i - LA) * 1024);
    const uint8_t* const src = i < LA ? uniform_ptr(a_base + (int64_t)s * 256) : uniform_ptr(w_base + (int64_t)s * 64);
    const uint32_t from = voff[i];
    const int lanes = __builtin_amdgcn_readfirstlane((s - end) >> 31);  // -1 or 0
    asm volatile("s_mov_b32 m0, %0\n\ts_mov_b32 exec_lo, %3\n\ts_mov_b32 exec_hi, %3\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1"
                 ::"s"(l0), "v"(from), "s"(src), "s"(lanes)
                 : "memory");
  };

  float16_t acc[2][TB];
  auto clear = [&]() {
#pragma unroll
    for (int tn = 0; tn < 2; ++tn)
#pragma unroll
      for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[tn][tb][i] = 0.0f;
    if constexpr (TB <= 2 && !MANY) {  // (made here and not where they are first used)
#pragma unroll
      for (int tn = 0; tn < 2; ++tn)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) asm volatile("" : "+v"(acc[tn][tb]));
    }
  };
  StreamMagic mg;
  static_cast<NibbleMagic&>(mg) = make_nibble_magic();
  mg.m_pair = 0x00f0000fu, mg.b_pair = 0x54006400u;
  asm volatile("" : "+v"(mg.m_pair), "+v"(mg.b_pair));  // (constants of the instruction otherwise, and two instructions in its place)
  const int w0th = 2 * KT * kg + KT * h;  // the lane's first packed word (and logical activation chunk) of a step
  const uint32_t fo_w = (uint32_t)(Cfg::A_TILE + wn * 4096) + addr::stream_w_frag(r32, w0th >> 2) + (uint32_t)((w0th & 3) * 4);
  uint32_t fo_a[KT];
#pragma unroll
  for (int t = 0; t < KT; ++t) fo_a[t] = addr::stream_a_frag(r32, w0th + t);
  const bool has_s = scales != nullptr, has_z = zeros != nullptr;
  const T one = from_float<T>(1.0f), zs = from_float<T>(zero_scalar);
  // Scales: a wavefront fetches those of 32 weight rows (with four groups of wavefronts half of them the scales, half the zero
  // points) and multiplies by those of its 64.
  const int sz_block = wave & (Cfg::BN / 32 - 1);
  const bool my_s = KG == 2 || wave < 4, my_z = KG == 2 || wave >= 4;
  uint8_t* const sz = smem + Cfg::RING + sz_block * Cfg::SZ;
  const uint8_t* const sz_read = smem + Cfg::RING + 2 * wn * Cfg::SZ;
  int first_group = 0;  // where group 0 of the window lies in this lane's rows of the scale area
  const uint32_t sz_lane = lds0 + (uint32_t)(Cfg::RING + 2 * wn * Cfg::SZ);

  // The slice runs in windows of as many steps as the scale area holds groups for (16 groups: 4, 8, 16 steps for groups
  // of 32, 64, 128 values, more for larger groups; 32 groups, twice as many, with four groups of wavefronts and where stream_max_groups says so).  Every window fetches its scales and restarts the ring: a memory
  // round trip without multiplications per window, which costs less than a further K slice (a partial tile to write
  // and add, and more work-groups than CUs).
  const int window = __builtin_amdgcn_readfirstlane(gshift >= 7 ? MG << (gshift - 7) : MG >> (7 - gshift));
  // fetch: the window's scales and zero points and what a step finds in flight of its first D steps; returns whether the zero points are small integers
  auto fetch = [&](int w0, int wsteps) -> bool {
    if (w0 > 0) __syncthreads();  // every wavefront has multiplied the previous window's last steps: the slots are free

    // ---- scales / zero points of this wavefront's 32 rows for the window, then the first two steps ----
    // Area of 32 rows: [s | z][32 rows][MG groups], 2 bytes each.  A row's groups of the window are contiguous in memory: where they
    // are 16-byte aligned, MG / 16 direct loads per tensor fetch them in 16-byte pieces (past the row's end its last piece again),
    // issued ahead of the ring so that the first step's wait covers them.  Rows of any other length: MG / 4 direct loads of
    // dwords, from the dword that holds the row's first group of the window on -- which is that dword's second value where
    // the row starts at an odd value (first_group) -- and never past the tensor's last dword.  Left over, tensors on odd 2-byte
    // addresses and windows of MG groups that start on an odd value: 2-byte gathers, four groups per instruction (they keep the
    // address unit busy for about a cycle per lane, so they go behind the weight loads, whose trip to HBM they overlap).
    // groups in this window: a slice is a whole number of groups, or a part of ONE group (large groups, K cut below the group
    // size: the plan takes slice lengths that divide the group, so the slice lies inside the group of its first step)
    const int G = ((wsteps << 7) >> gshift) > 0 ? ((wsteps << 7) >> gshift) : 1;
    const int g0 = ((step0 + w0) << 7) >> gshift;
    const bool wide = addr::stream_sz_wide(groups, g0) && (((uintptr_t)scales | (uintptr_t)zeros) & 15) == 0;  // uniform
    const bool dwords = !wide && (((uintptr_t)scales | (uintptr_t)zeros) & 3) == 0 && addr::stream_sz_dwords(MG, N, groups, g0, G);
    // (the same for both weight tiles: 32 rows on, a row starts an even number of values on)
    first_group = dwords ? addr::stream_sz_first(n0 + wn * 64 + r32, groups, g0) : 0;
    const uint32_t l_sz = lds0 + (uint32_t)(Cfg::RING + sz_block * Cfg::SZ);
    if (wide) {
#pragma unroll
      for (int i = 0; i < MG / 16; ++i) {
        const int row = addr::stream_sz_row(MG / 8, i, lane);
        int n = n0 + sz_block * 32 + row;
        n = n < N ? n : N - 1;
        const uint32_t voff = addr::stream_sz_piece_voff(n, groups, g0, addr::stream_sz_piece(MG, lane, row));
        if (has_s && my_s) dma16(l_sz + (uint32_t)(i * 1024), voff, (const uint8_t*)scales);
        if (has_z && my_z) dma16(l_sz + (uint32_t)(Cfg::SZ / 2 + i * 1024), voff, (const uint8_t*)zeros);
      }
    } else if (dwords) {
#pragma unroll
      for (int i = 0; i < MG / 4; ++i) {
        const int row = addr::stream_sz_row(MG / 2, i, lane);
        int n = n0 + sz_block * 32 + row;
        n = n < N ? n : N - 1;
        const uint32_t voff = addr::stream_sz_dword_voff(n, N, groups, g0, addr::stream_sz_dword(MG, lane, row));
        if (has_s && my_s) dma4(l_sz + (uint32_t)(i * 256), voff, (const uint8_t*)scales);
        if (has_z && my_z) dma4(l_sz + (uint32_t)(Cfg::SZ / 2 + i * 256), voff, (const uint8_t*)zeros);
      }
    }
    // Two steps now, the rest behind the barrier: a CU takes the loads in at 64 bytes a cycle, and the wavefronts that issue them wait for
    // that -- with the whole ring ahead of the barrier step 0 had long landed when they got there (2200 - 4700 cycles to issue).
#pragma unroll
    for (int s = 0; s < addr::kStreamAhead; ++s) static_for<0, Cfg::L>([&](auto ic) { issue1(w0 + s, w0 + wsteps, s, ic); });
    __builtin_amdgcn_sched_barrier(0);
    if (wide || dwords) {
      // loads return in issue order: with the two steps' loads still in flight the scales have landed
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(addr::stream_wait_scales(Cfg::L)) : "memory");
      if (!has_s || !has_z) {  // an absent tensor is the constant 1 / the scalar zero point
        const uint32_t ws = (uint32_t)bitcast<uint16_t>(one) * 0x10001u, wz = (uint32_t)bitcast<uint16_t>(zs) * 0x10001u;
        const uint4_t cs{ws, ws, ws, ws}, cz{wz, wz, wz, wz};
#pragma unroll
        for (int i = 0; i < MG / 16; ++i) {
          if (!has_s && my_s) *(uint4_t*)(sz + i * 1024 + lane * 16) = cs;
          if (!has_z && my_z) *(uint4_t*)(sz + Cfg::SZ / 2 + i * 1024 + lane * 16) = cz;
        }
      }
    } else {
      const int r16 = lane & 15, q = lane >> 4;
      T pre_s[2][MG / 4], pre_z[2][MG / 4];
#pragma unroll
      for (int tn = 0; tn < 2; ++tn) {
        int n = n0 + sz_block * 32 + tn * 16 + r16;
        n = n < N ? n : N - 1;
#pragma unroll
        for (int i = 0; i < MG / 4; ++i) {
          pre_s[tn][i] = one;
          pre_z[tn][i] = zs;
          if (4 * i < G) {  // uniform
            int g = q + 4 * i;
            g = g < G ? g : G - 1;
            const int64_t at = (int64_t)n * groups + g0 + g;
            if (has_s && my_s) pre_s[tn][i] = scales[at];
            if (has_z && my_z) pre_z[tn][i] = zeros[at];
          }
        }
      }
#pragma unroll
      for (int tn = 0; tn < 2; ++tn)
#pragma unroll
        for (int i = 0; i < MG / 4; ++i) {
          const int g = q + 4 * i;
          if (my_s) *(T*)(sz + addr::stream_sz_value(MG, tn * 16 + r16, g) * 2) = pre_s[tn][i];
          if (my_z) *(T*)(sz + Cfg::SZ / 2 + addr::stream_sz_value(MG, tn * 16 + r16, g) * 2) = pre_z[tn][i];
        }
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(addr::stream_wait_first(Cfg::L)) : "memory");
    __syncthreads();  // the window's scales and its step 0 are complete for every wavefront
#pragma unroll
    for (int s = addr::kStreamAhead; s < D; ++s)
      static_for<0, Cfg::L>([&](auto ic) {
        if (s < D - 1 || decltype(ic)::value < Cfg::LB) issue1(w0 + s, w0 + wsteps, s, ic);
      });
    // small integer zero points fold exactly into the unpack bias (a quarter of the conversion arithmetic less); decided
    // once per wavefront and window, on the zero points of the 64 rows it multiplies
    uint32_t fraction = 0;  // not zero for a fraction or a NaN
    float largest = 0.0f;
#pragma unroll
    for (int p = 0; p < 2 * (MG / 16); ++p) {
      const uint4_t v = *(const uint4_t*)(sz_read + (p & 1) * Cfg::SZ + Cfg::SZ / 2 + (p >> 1) * 1024 + lane * 16);
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float zf = to_float(bitcast<T>((uint16_t)(w[i] >> (16 * e))));
          fraction |= bitcast<uint32_t>(__builtin_amdgcn_fractf(zf));
          largest = __builtin_fmaxf(largest, __builtin_fabsf(zf));
        }
    }
    const bool integral = fraction == 0 && largest <= 256.0f;
    return __builtin_amdgcn_ballot_w64(integral) == ~0ull;
  };
  // The steps of a window.  A wavefront's step is NU units of TB MFMAs (unit u: k-step u / 2 of its KT, weight tile u % 2): eight with two
  // groups of wavefronts, four with four.  While unit u runs, the operand of unit u + 1 is expanded, a few vector instructions
  // behind every MFMA, and the activation operands of the next k-step are read; the last two units read those of the next step, its
  // packed words and scales.  The step's one barrier stands in front of those two: behind it step s + 1 is complete for everyone, and
  // everyone has read its last of step s, whose slot takes step s + D.
  auto multiply = [&](int w0, int wsteps, auto fold_tag) {
    constexpr bool FOLD = decltype(fold_tag)::value;
    typedef StreamExpand<T, FOLD, LAYOUT> Ex;
    constexpr int V = (Ex::INSTRUCTIONS + 4 + TB - 1) / TB;  // vector instructions behind an MFMA
    Ex ex[2];
    typedef typename std::conditional<KT == 4, uint4_t, uint2_t>::type words_t;
    words_t wq[2];
    T sv[2], zv[2];
    uint4_t af[2][TB], wop[2];
    uint32_t slot = 0;  // byte offset of step s in the ring
    auto word = [&](int tn, int t) -> uint32_t { return ((const uint32_t*)&wq[tn])[t]; };
    typedef __attribute__((address_space(3))) const T* lds_t;
    uint32_t sc_at;  // LDS address of this lane's scale of weight tile 0
    auto locate_scales = [&](int s) {
      const int gl = ((s << 7) + 8 * w0th) >> gshift;  // group of this lane's 8 KT values, relative to the window
      sc_at = sz_lane + (uint32_t)(addr::stream_sz_value(MG, r32, first_group + gl) * 2);
    };
    auto read_weights = [&](uint32_t at_slot, int tn) {
      wq[tn] = *(const words_t*)(smem + at_slot + fo_w + tn * 2048);
      sv[tn] = *(lds_t)(uintptr_t)(sc_at + (uint32_t)(tn * Cfg::SZ));
      zv[tn] = *(lds_t)(uintptr_t)(sc_at + (uint32_t)(tn * Cfg::SZ + Cfg::SZ / 2));
    };
    locate_scales(0);
#pragma unroll
    for (int tn = 0; tn < 2; ++tn) read_weights(slot, tn);
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) af[0][tb] = *(const uint4_t*)(smem + fo_a[0] + tb * 32 * 256);
    ex[0] = Ex(sv[0], zv[0], mg);
    wop[0] = ex[0](word(0, 0));
    int at_slot = 0, prev_slot = D - 1;
    for (int s = 0; s < wsteps; ++s) {
      const int next = at_slot + 1 == D ? 0 : at_slot + 1;
      const uint32_t next_slot = (uint32_t)(next * Cfg::SLOT);
      const int s_next = s + 1 < wsteps ? s + 1 : s;  // (past the end: what is read is not used)
      static_for<0, NU>([&](auto uc) {
        constexpr int u = decltype(uc)::value, t = u >> 1, tn = u & 1, v = (u + 1) % NU;
        if constexpr (u == NU - 2) {
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"(addr::stream_wait_step(D, Cfg::L)) : "memory");  // step s + 1
          __syncthreads();
        }
        // the loads of step s + D, spread over the units behind the barrier
        static_for<0, Cfg::L>([&](auto ic) {
          if constexpr (addr::stream_load_unit(decltype(ic)::value, NU, Cfg::L) == (u + 2) % NU)
            issue1(w0 + (u >= NU - 2 ? s + D : s + D - 1), w0 + wsteps, u >= NU - 2 ? at_slot : prev_slot, ic);
        });
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (v < 2) ex[v] = Ex(sv[v], zv[v], mg);
        wop[v & 1] = ex[v & 1](word(v & 1, v >> 1));
        if constexpr (u == (NU == 4 ? 1 : NU - 3)) locate_scales(s_next);
        if constexpr (u >= NU - 2) read_weights(next_slot, tn);
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
          if (tb * 2 / TB == tn) af[(t + 1) & 1][tb] = *(const uint4_t*)(smem + (t == KT - 1 ? next_slot : slot) + fo_a[(t + 1) % KT] + tb * 32 * 256);
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) acc[tn][tb] = Mma::mma(wop[u & 1], af[t & 1][tb], acc[tn][tb]);
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, V / 2, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, V - V / 2, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      prev_slot = at_slot, at_slot = next, slot = next_slot;
    }
  };
  // One copy of the loops per dequantiser: a choice inside a loop would make the two paths meet with the accumulators
  // in different registers.
  if constexpr (!MANY) {
    if constexpr (TB <= 2) clear();  // (while the first loads are on their way; more sums would not stay in registers across them)
    const bool fold = fetch(0, steps);
    if constexpr (TB > 2) clear();
    if (fold)
      multiply(0, steps, std::true_type{});
    else
      multiply(0, steps, std::false_type{});
  } else {
    // Windows run folded while their zero points allow it; from the first window that does not, the rest of the slice
    // runs unfolded (the two give the same bits).
    clear();
    int w0 = 0;
    bool fetched = false;
    for (; w0 < steps; w0 += window) {
      const int wsteps = steps - w0 < window ? steps - w0 : window;
      fetched = true;
      if (!fetch(w0, wsteps)) break;
      fetched = false;
      multiply(w0, wsteps, std::true_type{});
    }
    for (; w0 < steps; w0 += window) {
      const int wsteps = steps - w0 < window ? steps - w0 : window;
      if (!fetched) fetch(w0, wsteps);
      fetched = false;
      multiply(w0, wsteps, std::false_type{});
    }
  }

  // lane (r32, h) holds, as the four values j of acc[tn][tb], C[m = m0 + 32 tb + r32][n = n0 + 64 wn + 32 tn + 8 j + 4 h + 0..3].
  // The groups of wavefronts meet in LDS (the ring is no longer needed once everyone is past the last step): pairs of groups
  // swap halves of their quarters j and add, with four groups first 0 with 2 and 1 with 3, then 0 with 1 and 2 with 3; always
  // the lower group's sum plus the higher's.  Group kg ends up with 4 / KG quarters of every tile.
  constexpr int CELLS = 2 * TB;  // (tn, tb)
  float4_t sums[CELLS][4];
#pragma unroll
  for (int c = 0; c < CELLS; ++c)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      sums[c][j] = float4_t{acc[c / TB][c % TB][4 * j], acc[c / TB][c % TB][4 * j + 1], acc[c / TB][c % TB][4 * j + 2], acc[c / TB][c % TB][4 * j + 3]};
  // swap: of quarters J0 .. J0 + 2 H - 1 this wavefront keeps the lower H (upper = false) or the upper H
  auto swap = [&](auto j0_tag, auto h_tag, auto upper_tag, int region, int other) {
    constexpr int J0 = decltype(j0_tag)::value, H = decltype(h_tag)::value, GIVE = J0 + (decltype(upper_tag)::value ? 0 : H), KEEP = J0 + (decltype(upper_tag)::value ? H : 0);
    float4_t* const mine = (float4_t*)smem + region * (CELLS * H * 64) + lane;
    const float4_t* const theirs = (const float4_t*)smem + other * (CELLS * H * 64) + lane;
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CELLS; ++c)
#pragma unroll
      for (int i = 0; i < H; ++i) mine[(c * H + i) * 64] = sums[c][GIVE + i];
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CELLS; ++c)
#pragma unroll
      for (int i = 0; i < H; ++i) {
        const float4_t got = theirs[(c * H + i) * 64];
        sums[c][KEEP + i] = decltype(upper_tag)::value ? got + sums[c][KEEP + i] : sums[c][KEEP + i] + got;
      }
  };
  typedef std::integral_constant<int, 0> I0;
  typedef std::integral_constant<int, 1> I1;
  typedef std::integral_constant<int, 2> I2;
  const bool split = steps_total > slice_steps;
  auto store = [&](auto j0_tag) {  // the wavefront's quarters, from J0 on
    constexpr int J0 = decltype(j0_tag)::value, COUNT = 4 / KG;
    if (split) {
      // partial sums as [slice][N / 4][M][4]: from this layout of the accumulators every store is two runs of 512 bytes
      float4_t* const out = (float4_t*)partial + (int64_t)slice * M * (N >> 2);
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) {
        const int m = m0 + 32 * tb + r32;
#pragma unroll
        for (int tn = 0; tn < 2; ++tn)
#pragma unroll
          for (int i = 0; i < COUNT; ++i) {
            const int n4 = (n0 + 64 * wn + 32 * tn) / 4 + 2 * (J0 + i) + h;
            if (m < M && n4 < N / 4) out[(int64_t)n4 * M + m] = sums[tn * TB + tb][J0 + i];
          }
      }
      return;
    }
    EpiFloat::Params pe{C, N, 0, out_dtype};
    const EpiFloat epi(pe, 0);
    const int osz = epi.out_bytes(), row_bytes = Cfg::BN * osz;
    if (((N * osz) & 15) != 0) {
#pragma unroll
      for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int tn = 0; tn < 2; ++tn)
#pragma unroll
          for (int i = 0; i < COUNT; ++i) epi.store(m0 + 32 * tb + r32, n0 + 64 * wn + 32 * tn + 8 * (J0 + i) + 4 * h, sums[tn * TB + tb][J0 + i], M, N);
      return;
    }
    // whole rows of the output tile through LDS, 16-byte chunks swizzled by the row
    __syncthreads();
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
      for (int tn = 0; tn < 2; ++tn)
#pragma unroll
        for (int i = 0; i < COUNT; ++i) {
          const int row = 32 * tb + r32, byte = (64 * wn + 32 * tn + 8 * (J0 + i) + 4 * h) * osz;
          const uint4_t v = epi.pack(0, 0, sums[tn * TB + tb][J0 + i], 0, 0);
          uint8_t* const dst = smem + row * row_bytes + (((byte >> 4) ^ (row & 15)) << 4) + (byte & 15);
          if (osz == 2)
            *(uint2_t*)dst = uint2_t{v.x, v.y};
          else
            *(uint4_t*)dst = v;
        }
    __syncthreads();
    const int chunks = row_bytes >> 4;  // a power of two
    for (int at = threadIdx.x; at < Cfg::BM * chunks; at += 512) {
      const int row = at / chunks, chunk = at & (chunks - 1), m = m0 + row, n = n0 + chunk * (16 / osz);
      if (m < M && n < N) *(uint4_t*)epi.addr_of(m, n) = *(const uint4_t*)(smem + row * row_bytes + ((chunk ^ (row & 15)) << 4));
    }
  };
  if constexpr (KG == 2) {
    if (kg == 0) {
      swap(I0{}, I2{}, std::false_type{}, wn, WN + wn);
      store(I0{});
    } else {
      swap(I0{}, I2{}, std::true_type{}, WN + wn, wn);
      store(I2{});
    }
  } else {
    const int region = wave, across = wave ^ (2 * WN), beside = wave ^ WN;
    if (kg < 2) {
      swap(I0{}, I2{}, std::false_type{}, region, across);
      if (kg == 0) {
        swap(I0{}, I1{}, std::false_type{}, region, beside);
        store(I0{});
      } else {
        swap(I0{}, I1{}, std::true_type{}, region, beside);
        store(I1{});
      }
    } else {
      swap(I0{}, I2{}, std::true_type{}, region, across);
      if (kg == 2) {
        swap(I2{}, I1{}, std::false_type{}, region, beside);
        store(I2{});
      } else {
        swap(I2{}, I1{}, std::true_type{}, region, beside);
        store(std::integral_constant<int, 3>{});
      }
    }
  }
}

// Adds the K slices' partial sums in the order of the slices.  Lanes lie along M, where the sums are contiguous; a work-group's 64
// rows x 16 Q columns go through LDS, so that the outputs leave as whole lines of a row (stored from the sums' own layout, a
// thread per 16 bytes of a row, the pass took twice as long).
template <int Q>
__global__ __launch_bounds__(256) void w4a16_stream_reduce_kernel(const float4_t* __restrict__ partial, void* __restrict__ C, int M, int N, int slices, int out_dtype) {
  constexpr int PITCH = 16 * Q + 4;  // floats per row
  __shared__ __align__(16) float tile[64 * PITCH];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m0 = blockIdx.x * 64, n0 = blockIdx.y * (16 * Q), N4 = N >> 2;
  const int m = m0 + lane < M ? m0 + lane : M - 1;
  const int64_t slice = (int64_t)N4 * M;
  const float4_t* from[Q];
  float4_t sum[Q];
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    int n4 = n0 / 4 + wave * Q + i;
    n4 = n4 < N4 ? n4 : N4 - 1;
    from[i] = partial + (int64_t)n4 * M + m;
    sum[i] = *from[i];
  }
  int s = 1;
  for (; s + 3 <= slices; s += 3) {  // three slices' loads in flight
    float4_t v[3][Q];
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int i = 0; i < Q; ++i) v[j][i] = from[i][(s + j) * slice];
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int i = 0; i < Q; ++i) sum[i] += v[j][i];
  }
  for (; s < slices; ++s)
#pragma unroll
    for (int i = 0; i < Q; ++i) sum[i] += from[i][s * slice];
#pragma unroll
  for (int i = 0; i < Q; ++i) *(float4_t*)(tile + lane * PITCH + (wave * Q + i) * 4) = sum[i];
  __syncthreads();
  EpiFloat::Params pe{C, N, 0, out_dtype};
  const EpiFloat epi(pe, 0);
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const int at = i * 256 + threadIdx.x, row = at / (4 * Q), n = at % (4 * Q) * 4;
    epi.store(m0 + row, n0 + n, *(const float4_t*)(tile + row * PITCH + n), M, N);
  }
}

}  // namespace

thread_local int g_stream_tiles = 0;  // tuning and tests: 16-row activation tiles per work-group (2, 4, 6, 8), + 16 for four groups of wavefronts (0: the estimate below)
thread_local int g_stream_slice_steps = 0;  // tuning and tests: steps of 128 values of K per slice (0: the estimate below)

// The launch with the lowest estimate.  Per round of work-groups, one to a CU: a fixed part and its steps; a further window of scales
// restarts the ring; K slices cost a second launch and their partial sums' way to memory and back; then the products of the padded
// problem (power), the result, the weights and the activations.  Fitted to 1865 timed configurations of 1050 problems (M 17 .. 4096, N 256 ..
// 19200, K 512 .. 14336, groups of 64 - 256, both types, up to 2e11 operations), the choice among the configurations timed of a problem 1.5 % behind
// its best on average (22 % at most, more than 5 % on 19 of 158); on 3338 others (M 17 .. 512, N .. 33000, K .. 18944) 5 % high and 7.9 % rms.
// Rounds are whole: counted half by how full the last one is, as they were, plans with a few work-groups in a second round looked 15 - 20 % shorter
// than they are (188 x 18128 x 3200 284 work-groups in 49.6 us, 142 in 35.0): 575 problems that this moves 1.08 x on average, 27 of them 3 % and more behind.
static double stream_us(int64_t M, int64_t N, int64_t K, int tm, int kg, int64_t m_blocks, int64_t n_blocks, int64_t slice_steps, int64_t slices, double windows, int64_t cus) {
  static const double kStep[2][4] = {{0.73, 0.83, 0.95, 1.15}, {0.355, 0.47, 0.61, 0.68}};  // us per step of 128 values of K: [groups][32-row blocks]
  const int64_t blocks = m_blocks * n_blocks * slices;
  const double rounds = (double)ceil_div(blocks, cus);
  return 1.95 + rounds * ((kg == 4 ? 4.45 : 3.0) + (double)slice_steps * kStep[kg == 4][tm / 2 - 1] + 2.9 * (windows - 1.0)) +
         (slices > 1 ? 2.36 + 1.7e-6 * (double)slices * (double)M * (double)N : 0.0) + 0.385e-9 * (double)(m_blocks * tm * 16) * (double)(n_blocks * (512 / kg)) * (double)K +
         0.6e-6 * (double)M * (double)N + 0.022e-6 * (double)N * (double)K + 0.086e-6 * (double)M * (double)K;
}
// The order by XCD where it keeps enough bytes from going into several L2s: the activations, which go into all eight (fewer with fewer blocks
// of weight rows) instead of the two or so that share a slice, and the weights, which the blocks of activation rows of a slice share.  Blocks of
// 128 weight rows, twice as many as the kernel had before, had made that 403 x 1280 x 12544 30.1 -> 33.9 us (by XCD 25.7) and 482 x 1024 x 16256 34.4 ->
// 40.3 (29.1).  On 1524 problems (M 17 .. 3000, N .. 32000, K .. 17920; the line is from 1491 others) it is 3.4 % ahead on average on the 561 beyond the
// line (4.8 % with K slices, 27 % at most), 3 % and more behind on 5.  Short of the line XCDs whose work-groups all read one slice at a time
// are up to 13 % behind (257 x 640 x 10240 18.5 against 16.1 us); without slices the two are level there.
static bool stream_by_xcd(const StreamPlan& p, int64_t M, int64_t N, int64_t K) {
  auto gcd8 = [](int64_t n) { return n % 8 == 0 ? 8.0 : (n % 4 == 0 ? 4.0 : (n % 2 == 0 ? 2.0 : 1.0)); };
  const double nb = p.n_blocks, sl = p.split, shares = (sl + 8.0 - gcd8(p.split)) / sl;
  const double a = 2e-6 * (double)M * (double)K * ((nb < 8.0 ? nb : 8.0) - (nb < shares ? nb : shares));
  const double meet = 8.0 / gcd8((int64_t)p.n_blocks * p.split), w = 0.5e-6 * (double)N * (double)K * ((p.m_blocks < meet ? p.m_blocks : meet) - 1.0);
  return a + w > (p.split > 1 ? 40.0 : 12.0);  // MB
}
static StreamPlan stream_plan_now(int64_t M, int64_t N, int64_t K, int64_t group, int64_t cus, bool short_windows) {
  StreamPlan best{false, 0, 0, 0, 0, 0, 2, 0.0, false};
  if (M < 17 || M > kStreamMaxRows || N < 1 || K < 128 || K % 128 != 0 || group < 32 || (group & (group - 1)) != 0 || K % group != 0) return best;
  if (N % 4 != 0) return best;
  const int64_t steps_total = K / 128;
  // a slice is a whole number of groups, or -- groups of more than 128 values, e.g. one scale per weight row -- a power-of-two
  // part of one group (K % group == 0: such slices tile K, each inside one group, whose scale every step of the slice uses)
  const int64_t unit = group > 128 ? group / 128 : 1;
  auto whole_or_part = [&](int64_t ss) {
    if (ss >= unit) return ceil_div(ss, unit) * unit;
    int64_t part = 1;
    while (part < ss) part *= 2;
    return part;  // (unit is a power of two: part divides it)
  };
  for (int kg = 2; kg <= 4; kg += 2)
    for (int tm = 2; tm <= 8; tm += 2) {
      if (g_stream_tiles > 0 ? (tm != (g_stream_tiles & 15) || kg != (g_stream_tiles >= 16 ? 4 : 2)) : (tm > 2 && M <= 16 * (tm - 2)) || (tm < 6 && M > 16 * tm)) continue;
      const int64_t m_blocks = ceil_div(M, (int64_t)16 * tm), n_blocks = ceil_div(N, (int64_t)(512 / kg));
      const int64_t window = (int64_t)stream_max_groups(kg) * group / 128;  // steps whose groups the scale area holds; and in a slice of several windows (where those hold
      // more: 0.6 of a restart more, for the control flow of several windows and their longer fetch)
      const int64_t of_many = short_windows ? window : (int64_t)stream_max_groups(kg, tm / 2, true) * group / 128;
      for (int64_t want = 1; want <= 16; ++want) {
        int64_t ss = whole_or_part(ceil_div(steps_total, want));
        if (g_stream_slice_steps > 0) {
          ss = g_stream_slice_steps < unit && unit % g_stream_slice_steps == 0 ? (int64_t)g_stream_slice_steps : ceil_div((int64_t)g_stream_slice_steps, unit) * unit;
          want = 16;
        } else if (ss < 4 && steps_total >= 4) {
          continue;  // at least four steps per work-group
        }
        if (ss > steps_total) ss = steps_total;
        const int64_t slices = ceil_div(steps_total, ss);
        if (slices > 16) continue;  // too many partial sums to add up: the tile kernel with longer slices takes it
        const double us = stream_us(M, N, K, tm, kg, m_blocks, n_blocks, ss, slices, ss <= window ? 1.0 : (double)ceil_div(ss, of_many) + (of_many > window ? 0.6 : 0.0), cus);
        if (!best.ok || us < best.us) best = StreamPlan{true, tm, (int)m_blocks, (int)n_blocks, (int)slices, (int)ss, kg, us, false};
      }
    }
  if (best.ok) best.by_xcd = stream_by_xcd(best, M, N, K);
  return best;
}
StreamPlan w4a16_stream_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus, bool short_windows) {
  static thread_local PlanTable<StreamPlan> known;
  const int64_t n = cus > 0 ? cus : 256;
  return known.get(M, N, K, (group * 2 + short_windows) * 4096 + n, [&] { return stream_plan_now(M, N, K, group, n, short_windows); });
}

template <typename T, int TB, int KG, int LAYOUT, bool MANY>
static int launch_stream(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, float* partial,
                         int64_t M, int64_t N, int64_t K, int gshift, float zero_scalar, int out_dtype, const StreamPlan& p,
                         hipStream_t st) {
  auto kern = w4a16_stream_kernel<T, TB, KG, LAYOUT, MANY>;
  constexpr int lds_bytes = StreamCfg<TB, KG, MANY>::LDS;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (e != hipSuccess) {
      set_error("tlq_gemm_w4a16(stream): cannot reserve %d bytes of LDS: %s", lds_bytes, hipGetErrorString(e));
      return 1;
    }
    attr_set = true;
  }
  kern<<<dim3(p.n_blocks, p.split, p.m_blocks), 512, lds_bytes, st>>>((const T*)A, (const uint8_t*)Wp, (const T*)scales, (const T*)zeros, C, partial, (int)M,
                                                                     (int)N, (int)K, gshift, zero_scalar, out_dtype, p.slice_steps, p.by_xcd ? p.split : 0);
  char detail[80] = "";
  if (launch_log_on()) snprintf(detail, sizeof(detail), "w4a16_stream_kernel, %d activation rows per work-group%s", 32 * TB, p.by_xcd ? ", by XCD" : "");
  return check_launch("tlq_gemm_w4a16(stream)", detail) ? 0 : 1;
}

// partial: fp32 [split][N / 4][M][4] workspace, needed when the plan has more than one K slice
int gemm_w4a16_stream(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t M, int64_t N,
                      int64_t K, int64_t group, float zero_scalar, int in_dtype, int out_dtype, int w_layout, const StreamPlan& p,
                      float* partial, hipStream_t st) {
  int gshift = 0;
  while (((int64_t)1 << gshift) < group) ++gshift;
  const bool many = (int64_t)p.slice_steps * 128 > stream_max_groups(p.kg) * group;  // the slice holds more groups than one window of the scale area
  int rc;
#define TLQ_STREAM4(T, TB, LAY, MANY) (p.kg == 4 ? TLQ_STREAM5(T, TB, 4, LAY, MANY) : TLQ_STREAM5(T, TB, 2, LAY, MANY))
#define TLQ_STREAM5(T, TB, KG, LAY, MANY) launch_stream<T, TB, KG, LAY, MANY>(A, Wp, scales, zeros, C, partial, M, N, K, gshift, zero_scalar, out_dtype, p, st)
#define TLQ_STREAM3(T, TB, LAY) (many ? TLQ_STREAM4(T, TB, LAY, true) : TLQ_STREAM4(T, TB, LAY, false))
#define TLQ_STREAM(T, TB) (w_layout == TLQ_W_INTERLEAVED_F16 ? TLQ_STREAM3(T, TB, 1) : TLQ_STREAM3(T, TB, 0))
#define TLQ_STREAM_TM(TB) (in_dtype == TLQ_F16 ? TLQ_STREAM(half_t, TB) : TLQ_STREAM(bf16_t, TB))
  rc = p.tm == 2 ? TLQ_STREAM_TM(1) : (p.tm == 4 ? TLQ_STREAM_TM(2) : (p.tm == 6 ? TLQ_STREAM_TM(3) : TLQ_STREAM_TM(4)));
#undef TLQ_STREAM_TM
#undef TLQ_STREAM3
#undef TLQ_STREAM4
#undef TLQ_STREAM5
#undef TLQ_STREAM
  if (rc) return rc;
  if (p.split == 1) return 0;
  const int64_t m64 = ceil_div(M, (int64_t)64);
  if (m64 * ceil_div(N, (int64_t)64) >= 512)  // two work-groups per CU
    w4a16_stream_reduce_kernel<4><<<dim3((unsigned)m64, (unsigned)ceil_div(N, (int64_t)64)), 256, 0, st>>>((const float4_t*)partial, C, (int)M, (int)N, p.split, out_dtype);
  else
    w4a16_stream_reduce_kernel<2><<<dim3((unsigned)m64, (unsigned)ceil_div(N, (int64_t)32)), 256, 0, st>>>((const float4_t*)partial, C, (int)M, (int)N, p.split, out_dtype);
  return check_launch("tlq_gemm_w4a16(stream, reduce)", "w4a16_stream_reduce_kernel") ? 0 : 1;
}

}  // namespace tlq
