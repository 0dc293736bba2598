// Small-tile GEMM: tiles of 16 MT activation rows x 16 RT columns of the result (MT, RT = 1, 2, 4), one per work-group, whose
// wavefronts split K and add their partial tiles through LDS -- one launch, nothing in memory between.  For the int8, W4A8 and
// plain 16-bit products whose 128-wide tiles would leave most of the machine idle: those run 6 us + 0.35 us per 128-byte stage of
// K on a handful of CUs, or cut K over work-groups and pay a second launch for the sums.  (The W4A16 form of the same
// kernel, with scales and zero points, is gemm_w4a16_small.hip; what bounds small problems is explained there.)
//
// A step is 128 bytes of K of an activation row (128 int8 or 64 16-bit values).  Every global access is a full-width direct
// global -> LDS load into a ring of D slots that only this wavefront uses (no barrier, only counters); the MFMA operands are read back
// with the layouts of gemm_addr.h.  At step i the loads of steps i + 1 .. i + D are in flight or about to be.
//   activations, and weights stored [N, K]:  [16 rows][128 B] per tile, two loads of 8 rows
//   packed int4 weights [N, K/2]:            [16 rows][64 B] per tile, one load; a lane's 16 bytes are 32 consecutive values,
//                                            expanded in registers, so the activation chunk of MFMA ks is 2 q + ks
//   weights stored [K, N] (RT = 4):          [128 or 64 k rows][64 columns] as they are, eight loads, transposed by the read
#pragma once
#include "gemm_core.h"
#include "small_tiles.h"

namespace tlq {

template <SmallW W, int RT, int MT>
struct SmallCfg {
  static constexpr int A_TILE = MT * 2048;
  static constexpr int W_TILE = addr::small_w_tile(W, RT);
  static constexpr int SLOT = addr::small_slot_bytes(W, RT, MT);
  static constexpr int D = addr::small_depth(SLOT);  // steps in the ring
  static_assert(SLOT == A_TILE + W_TILE, "the two parts of a slot");
  static constexpr int LDS = D * SLOT;                                  // per wavefront
  static constexpr int LOADS = SLOT / 1024;                             // direct loads per step
  static constexpr int MAX_WAVES = RT * MT <= 4 ? 16 : 8;
  static_assert(W == kSmallNK || W == kSmallW4 || RT == 4, "[K, N] weights come in tiles of 64 columns");
  static_assert(LOADS * (D - 1) <= 63, "vmcnt range");
  static_assert(LDS >= RT * MT * 1024, "the partial tiles fit the ring");
};

struct SmallParams {
  const uint8_t* a;
  const uint8_t* w;
  int64_t a_batch, w_batch;  // bytes between the batches
  int a_row, w_row;          // bytes between rows ([K, N] weights: between k rows)
  int steps;                 // of 128 bytes of K
  uint16_t sign_mode;        // packed weights
  uint16_t waves;            // of a work-group
};

// four nibbles held one per byte (0 .. 15) -> four int8 under the sign convention; a word of eight -> k order
__device__ __forceinline__ uint32_t small_sign4(uint32_t x, int sign_mode) {
  if (sign_mode == TLQ_U4) return x;
  if (sign_mode == TLQ_S4_TWOS) x ^= 0x08080808u;  // two's complement == offset-8 of (u ^ 8)
  const uint32_t c = sign_mode == TLQ_S4_OFFSET7 ? 0x07070707u : 0x08080808u;
  return ((x | 0x80808080u) - c) ^ 0x80808080u;  // per byte, no borrows between bytes
}
__device__ __forceinline__ uint2_t small_expand8(uint32_t v, int sign_mode) {
  const uint32_t lo = small_sign4(v & 0x0f0f0f0fu, sign_mode), hi = small_sign4((v >> 4) & 0x0f0f0f0fu, sign_mode);
  return uint2_t{__builtin_amdgcn_perm(hi, lo, 0x05010400u), __builtin_amdgcn_perm(hi, lo, 0x07030602u)};
}
// Two's complement nibbles as int8 of 16 times their value -- a nibble in the upper half of its byte is its own sign extension: 5
// instructions a word against 11 - 13 -- ; `flip` turns offset-8 nibbles into two's complement (u ^ 8 == u - 8).  The sums are
// 16 times the result, and exact, while 16 x 8 x 128 K < 2^31 (small_w4a8_times16).  Expanding was what bounded the tiles: 128 x 4096 x 11008 (86 steps per CU)
// 20.3 us before, 14.7 now; the other two conventions stay as they were.
__device__ __forceinline__ uint2_t small_expand8_times16(uint32_t v, uint32_t flip) {
  v ^= flip;
  const uint32_t lo = (v << 4) & 0xf0f0f0f0u, hi = v & 0xf0f0f0f0u;
  return uint2_t{__builtin_amdgcn_perm(hi, lo, 0x05010400u), __builtin_amdgcn_perm(hi, lo, 0x07030602u)};
}

// TIMES16 (packed weights): small_expand8_times16; the epilogue divides.
template <class Mma, SmallW W, class Epi, int RT, int MT, bool TIMES16>
__global__ __launch_bounds__(RT* MT <= 4 ? 1024 : 512) void gemm_small_kernel(SmallParams p, typename Epi::Params pe, int M, int N) {
  typedef SmallCfg<W, RT, MT> Cfg;
  typedef __attribute__((address_space(3))) uint8_t* lptr_t;
  typedef typename Mma::acc_t acc_t;
  constexpr int D = Cfg::D, L = Cfg::LOADS;
  extern __shared__ __align__(16) uint8_t smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int waves = p.waves;
  const int r16 = lane & 15, q = lane >> 4;
  uint8_t* const mine = smem + wave * Cfg::LDS;
  const uint32_t mine_lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lptr_t)mine);
  const int n_base = blockIdx.x * (16 * RT), m_base = blockIdx.y * (16 * MT), batch = blockIdx.z;
  const int s0 = addr::small_first(wave, waves, p.steps), s1 = addr::small_first(wave + 1, waves, p.steps);
  const int n_steps = s1 - s0;
  const uint8_t* const a_base = p.a + batch * p.a_batch;
  const uint8_t* const w_base = p.w + batch * p.w_batch;

  // ---- per-lane source offsets (rows and columns past the matrices are clamped; masked at the store) ----
  uint32_t voff_a[2 * MT], voff_w[Cfg::W_TILE / 1024];
#pragma unroll
  for (int j = 0; j < 2 * MT; ++j) voff_a[j] = addr::rd_voff(lane, 0, j, 1, M - m_base, (uint32_t)p.a_row) + (uint32_t)m_base * (uint32_t)p.a_row;
  int64_t w_step;  // bytes from a step of the weights to the next
  if constexpr (W == kSmallNK) {
    w_step = 128;
#pragma unroll
    for (int j = 0; j < 2 * RT; ++j) voff_w[j] = addr::rd_voff(lane, 0, j, 1, N - n_base, (uint32_t)p.w_row) + (uint32_t)n_base * (uint32_t)p.w_row;
  } else if constexpr (W == kSmallW4) {
    w_step = 64;
#pragma unroll
    for (int j = 0; j < RT; ++j) {
      int n = n_base + j * 16 + addr::sw_row(lane);
      n = n < N ? n : N - 1;
      voff_w[j] = (uint32_t)n * (uint32_t)p.w_row + (uint32_t)(addr::sw_piece(lane) * 16);
    }
  } else {
    constexpr int KR = W == kSmallKN8 ? 128 : 64;  // k rows per step
    w_step = (int64_t)KR * p.w_row;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      voff_w[j] = (W == kSmallKN8 ? addr::kn_voff<64>(lane, 0, j, 1, N - n_base, (uint32_t)p.w_row)
                                  : addr::kn16_voff<64>(lane, 0, j, 1, N - n_base, (uint32_t)p.w_row)) +
                  (uint32_t)(n_base * (W == kSmallKN8 ? 1 : 2));
  }
  auto dma16 = [&](uint32_t lds_addr, uint32_t voff, const uint8_t* sbase) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(voff), "s"(sbase) : "memory");
  };
  auto issue = [&](int s, int slot) {
    const uint8_t* asb = uniform_ptr(a_base + (int64_t)s * 128);
    const uint8_t* wsb = uniform_ptr(w_base + (int64_t)s * w_step);
    const uint32_t l0 = mine_lds + (uint32_t)(slot * Cfg::SLOT);
#pragma unroll
    for (int j = 0; j < Cfg::W_TILE / 1024; ++j) dma16(l0 + Cfg::A_TILE + j * 1024, voff_w[j], wsb);
#pragma unroll
    for (int j = 0; j < 2 * MT; ++j) dma16(l0 + j * 1024, voff_a[j], asb);
  };

  // ---- per-lane LDS offsets of the operand reads ----
  uint32_t fo_a[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) fo_a[ks] = (uint32_t)lds_off(r16, W == kSmallW4 ? 2 * q + ks : q + 4 * ks);
  uint32_t fo_w[4];
  if constexpr (W == kSmallW4) {
    fo_w[0] = addr::sw_frag_off(lane);
  } else if constexpr (W == kSmallKN8 || W == kSmallKN16) {
#pragma unroll
    for (int t = 0; t < 4; ++t) fo_w[t] = W == kSmallKN8 ? addr::knfrag_off<64>(lane, 0, t) : addr::kn16frag_off<64>(lane, 0, t);
  }

  const uint32_t flip = p.sign_mode == TLQ_S4_OFFSET8 ? 0x88888888u : 0u;
  acc_t acc[RT][MT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = acc_t{0, 0, 0, 0};

#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d < n_steps) issue(s0 + d, d);
  int slot = 0;
  for (int i = 0; i < n_steps; ++i) {
    const int younger = addr::small_younger(i, n_steps, D);  // steps issued behind this one
    if (D >= 4 && younger == 3)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(D >= 4 ? 3 * L : 0) : "memory");
    else if (D >= 3 && younger == 2)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(D >= 3 ? 2 * L : 0) : "memory");
    else if (younger == 1)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const uint8_t* const tile = mine + slot * Cfg::SLOT;
    uint4_t af[MT][2], wf[RT][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) af[mt][ks] = *(const uint4_t*)(tile + fo_a[ks] + mt * 2048);
    const uint8_t* const wt = tile + Cfg::A_TILE;
    if constexpr (W == kSmallNK) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) wf[rt][ks] = *(const uint4_t*)(wt + fo_a[ks] + rt * 2048);
    } else if constexpr (W == kSmallW4) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) wf[rt][0] = *(const uint4_t*)(wt + fo_w[0] + rt * 1024);
    } else if constexpr (W == kSmallKN8) {
      typedef int v2i_t __attribute__((ext_vector_type(2)));
      typedef __attribute__((address_space(3))) v2i_t* lds_ptr;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const uint8_t* b = wt + fo_w[rt] + ks * 64 * 64;
          const v2i_t lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_ptr)(b)), hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_ptr)(b + 8 * 64));
          wf[rt][ks] = uint4_t{(uint32_t)lo.x, (uint32_t)lo.y, (uint32_t)hi.x, (uint32_t)hi.y};
        }
    } else {
      typedef short v4s_t __attribute__((ext_vector_type(4)));
      typedef __attribute__((address_space(3))) v4s_t* lds_ptr;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const uint8_t* b = wt + fo_w[rt] + ks * 32 * 128;
          const uint2_t lo = bitcast<uint2_t>(__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(b)));
          const uint2_t hi = bitcast<uint2_t>(__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(b + 4 * 128)));
          wf[rt][ks] = uint4_t{lo.x, lo.y, hi.x, hi.y};
        }
    }
    // the slot may be overwritten once its contents are in registers
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (i + D < n_steps) issue(s0 + i + D, slot);
    slot = slot + 1 == D ? 0 : slot + 1;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      if constexpr (W == kSmallW4) {
        const uint4_t v = wf[rt][0];
        uint2_t e0, e1, e2, e3;
        if constexpr (TIMES16) {
          e0 = small_expand8_times16(v.x, flip), e1 = small_expand8_times16(v.y, flip);
          e2 = small_expand8_times16(v.z, flip), e3 = small_expand8_times16(v.w, flip);
        } else {
          e0 = small_expand8(v.x, p.sign_mode), e1 = small_expand8(v.y, p.sign_mode);
          e2 = small_expand8(v.z, p.sign_mode), e3 = small_expand8(v.w, p.sign_mode);
        }
        wf[rt][0] = uint4_t{e0.x, e0.y, e1.x, e1.y};
        wf[rt][1] = uint4_t{e2.x, e2.y, e3.x, e3.y};
      }
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = Mma::mma(wf[rt][ks], af[mt][ks], acc[rt][mt]);
    }
  }

  // add the partial tiles of the wavefronts (the rings are dead once everyone is here)
  Epi epi(pe, batch);
  auto finished = [](acc_t sum) {
    if constexpr (TIMES16) sum >>= 4;
    return sum;
  };
  if (waves == 1) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) epi.store(m_base + mt * 16 + r16, n_base + rt * 16 + 4 * q, finished(acc[rt][mt]), M, N);
    return;
  }
  __syncthreads();
  acc_t* const red = (acc_t*)smem;  // [waves][RT * MT][64 lanes]
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) red[(wave * (RT * MT) + rt * MT + mt) * 64 + lane] = acc[rt][mt];
  __syncthreads();
  for (int item = threadIdx.x; item < RT * MT * 64; item += waves * 64) {
    acc_t sum = red[item];
    if (waves == 8) {  // (all asked for at once: one by one the reads wait for each other)
      acc_t part[7];
#pragma unroll
      for (int w = 1; w < 8; ++w) part[w - 1] = red[w * (RT * MT * 64) + item];
#pragma unroll
      for (int w = 1; w < 8; ++w) sum += part[w - 1];
    } else {
#pragma unroll 4
      for (int w = 1; w < waves; ++w) sum += red[w * (RT * MT * 64) + item];
    }
    const int tile = item >> 6, l = item & 63;  // lane l of a tile holds C[m = l % 16][n = 4 (l / 16) .. + 3]
    const int rt = tile / MT, mt = tile - rt * MT;
    epi.store(m_base + mt * 16 + (l & 15), n_base + rt * 16 + 4 * (l >> 4), finished(sum), M, N);
  }
}

constexpr int small_lds(SmallW w, int rt, int mt) {
  const int slot = addr::small_slot_bytes(w, rt, mt);
  return slot * addr::small_depth(slot);
}

template <class Mma, SmallW W, class Epi, int RT, int MT, bool TIMES16>
int launch_one(SmallParams p, const typename Epi::Params& pe, int64_t batch, int64_t M, int64_t N, int waves, const char* what, hipStream_t st) {
  typedef SmallCfg<W, RT, MT> Cfg;
  static_assert(Cfg::LDS == small_lds(W, RT, MT), "the plan's LDS");
  auto kern = gemm_small_kernel<Mma, W, Epi, RT, MT, TIMES16>;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) {
      set_error("%s: cannot reserve LDS: %s", what, hipGetErrorString(e));
      return 1;
    }
    attr_set = true;
  }
  p.waves = (uint16_t)waves;
  const dim3 blocks((unsigned)ceil_div(N, (int64_t)16 * RT), (unsigned)ceil_div(M, (int64_t)16 * MT), (unsigned)batch);
  kern<<<blocks, waves * 64, (size_t)waves * Cfg::LDS, st>>>(p, pe, (int)M, (int)N);
  return check_launch(what, "gemm_small_kernel") ? 0 : 1;
}

template <class Mma, SmallW W, class Epi, bool TIMES16 = false>
int launch_tile(const SmallTile& t, const SmallParams& p, const typename Epi::Params& pe, int64_t batch, int64_t M, int64_t N, const char* what, hipStream_t st) {
#define TLQ_ONE(RT, MT) \
  if (t.rt == RT && t.mt == MT) return launch_one<Mma, W, Epi, RT, MT, TIMES16>(p, pe, batch, M, N, t.waves, what, st);
  if constexpr (W == kSmallNK || W == kSmallW4) {
    TLQ_ONE(1, 1) TLQ_ONE(2, 1) TLQ_ONE(1, 2) TLQ_ONE(2, 2) TLQ_ONE(1, 4) TLQ_ONE(2, 4)
  }
  TLQ_ONE(4, 1) TLQ_ONE(4, 2) TLQ_ONE(4, 4)
#undef TLQ_ONE
  set_error("%s: no such tile", what);
  return 1;
}

inline SmallParams small_params(const void* A, const void* B, int64_t M, int64_t N, int64_t row_bytes, int64_t w_row, int64_t w_bytes) {
  return SmallParams{(const uint8_t*)A, (const uint8_t*)B, M * row_bytes, w_bytes, (int)row_bytes, (int)w_row, (int)(row_bytes / 128), 0, 0};
}

// W4A8 with weights multiplied as 16 times their value (gemm_small_w4a8.hip)
int small_w4a8_times16_launch(const SmallTile& t, const SmallParams& p, const EpiInt32::Params& pe, int64_t M, int64_t N, hipStream_t st);

}  // namespace tlq
