// W4A16 for problems too small to fill the machine with large tiles: tiles of 16 MT activation rows x 16 RT weight rows
// (MT, RT = 1, 2, 4), one per work-group, whose wavefronts split K and add their partial tiles through LDS -- one launch,
// no partial sums in memory, as many work-groups as there are small tiles.
//
// What bounds a small problem is latency: the launch, a round trip to memory, and -- with K cut over work-groups, as the
// streaming and tile kernels do to fill the machine -- a second launch that adds the slices' partial tiles.  Those kernels take
// 13 - 16 us for 100 rows on 1024 x 3072 or 2304 x 640; this one 5.5 - 6.5.  The price is that every work-group pulls all of
// its activation rows through its CU (K x (2 BM + BN / 2) bytes per tile), so with more rows and wider matrices the kernels
// with large tiles are ahead; where the line lies is decided by estimates (w4a16_small_plan and its callers).
//
// Every global access is a full-width direct global -> LDS load (1 KB per wavefront instruction, adjacent lanes adjacent
// addresses): per k-block of 128 values RT loads of a [16 rows][64 B] packed-weight tile and 4 MT loads of [4 rows][256 B] of
// activations, into one of two slots of LDS that only this wavefront uses (so there is no barrier, only counters).  The
// MFMA-shaped fragments are then read back with ds_read_b128 (swizzles as in the streaming kernel: no bank conflicts).  Scales
// and zero points come in as dword gathers that cover four consecutive groups of the 16 rows at once, i.e. once per four
// k-blocks at groups of 128.  While k-block i is dequantised and multiplied, the loads of i + 1 and i + 2 are in flight.
//
// k assignment: lane (row r16, k-group q) holds the packed words 4 q .. 4 q + 3 of its weight row = values 32 q .. 32 q + 31 of the
// k-block, one word per MFMA; the activation operand of MFMA j is chunk 4 q + j.  LAYOUT 1: words repacked by
// interleave_weight (tilelang/quantize/utils.py:73-101, fp16 target); the same sums, so the same bits.
#include "expand8.h"
#include "gemm_core.h"
#include "small_tiles.h"

namespace tlq {

template <typename T>
struct SmallMma;
template <>
struct SmallMma<half_t> {
  typedef MmaF16 type;
};
template <>
struct SmallMma<bf16_t> {
  typedef MmaBF16 type;
};

constexpr int small_wave_lds(int rt, int mt) { return 2 * addr::smallw_slot_bytes(rt, mt) + 2 * addr::smallw_sc_bytes(rt); }
constexpr int small_max_waves(int mt) { return mt == 1 ? 16 : 8; }

template <typename T, bool FOLD, int LAYOUT, int RT, int MT>
__global__ __launch_bounds__(MT == 1 ? 1024 : 512) void w4a16_small_kernel(const T* __restrict__ A, const uint8_t* __restrict__ Wp,
                                                                const T* __restrict__ scales, const T* __restrict__ zeros,
                                                                void* __restrict__ C, int M, int N, int K, int gshift,
                                                                float zero_scalar, int out_dtype, int waves) {
  typedef typename SmallMma<T>::type Mma;
  typedef __attribute__((address_space(3))) uint8_t* lptr_t;
  constexpr int SLOT = addr::smallw_slot_bytes(RT, MT);  // RT weight tiles + MT activation tiles
  constexpr int SC = addr::smallw_sc_bytes(RT);          // [rt][scale | zero][64 dwords]
  constexpr int WAVE_LDS = 2 * SLOT + 2 * SC;
  constexpr int NI = RT + 4 * MT;         // direct loads per k-block
  extern __shared__ __align__(16) uint8_t smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, q = lane >> 4;
  uint8_t* const mine = smem + wave * WAVE_LDS;
  const uint32_t mine_lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lptr_t)mine);
  const int n_base = blockIdx.x * (16 * RT), m_base = blockIdx.y * (16 * MT);
  const int groups = K >> gshift;
  const int KB = K >> 7;
  const int kb0 = addr::small_first(wave, waves, KB), kb1 = addr::small_first(wave + 1, waves, KB);
  const int nkb = kb1 - kb0;
  const bool has_s = scales != nullptr, has_z = zeros != nullptr;
  const int NS = RT * ((has_s ? 1 : 0) + (has_z ? 1 : 0));  // gathers per scale period (uniform)
  const T one = from_float<T>(1.0f), zs = from_float<T>(zero_scalar);
  const NibbleMagic mg = make_nibble_magic();

  // ---- per-lane source offsets of the direct loads ----
  uint32_t voff_w[RT], voff_a[4 * MT], row_g[RT];
  {
    const int rho = addr::sw_row(lane), piece = addr::sw_piece(lane);  // lands on row lane/4, physical piece lane%4
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      int n = n_base + rt * 16 + rho;
      n = n < N ? n : N - 1;
      voff_w[rt] = (uint32_t)n * (uint32_t)(K >> 1) + (uint32_t)(piece * 16);
      int ng = n_base + rt * 16 + r16;  // the row this lane gathers scales for / dequantises
      ng = ng < N ? ng : N - 1;
      row_g[rt] = (uint32_t)ng * (uint32_t)groups;
    }
#pragma unroll
    for (int i = 0; i < 4 * MT; ++i) {
      const int row = m_base + addr::sa_row(lane, i);
      const int m = row < M ? row : M - 1;
      voff_a[i] = ((uint32_t)m * (uint32_t)K) * 2u + (uint32_t)(addr::sa_chunk(lane, i) * 16);
    }
  }
  // ---- per-lane LDS offsets of the fragment reads ----
  const uint32_t fo_w = addr::sw_frag_off(lane);
  uint32_t fo_a[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) fo_a[j] = (uint32_t)(RT * 1024) + addr::sa_frag_off(lane, 0, j);

  auto dma16 = [&](uint32_t lds_addr, uint32_t voff, const uint8_t* sbase) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(voff), "s"(sbase) : "memory");
  };
  auto issue_kb = [&](int kb, int slot) {
    const uint8_t* wsb = uniform_ptr(Wp + (int64_t)kb * 64);
    const uint8_t* asb = uniform_ptr((const uint8_t*)A + (int64_t)kb * 256);
    const uint32_t l0 = mine_lds + (uint32_t)(slot * SLOT);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) dma16(l0 + rt * 1024, voff_w[rt], wsb);
#pragma unroll
    for (int i = 0; i < 4 * MT; ++i) dma16(l0 + RT * 1024 + i * 1024, voff_a[i], asb);
  };
  // four consecutive groups (base .. base+3) of the 16 rows of every tile: lane (row r16, group q)
  auto issue_sc = [&](int base, int buf) {
    const uint32_t l0 = mine_lds + (uint32_t)(2 * SLOT + buf * SC);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const uint64_t e2 = addr::smallw_sc_elem(lane, base, row_g[rt], groups) * 2u;
      if (has_s) {
        const uint64_t a = ((uint64_t)(uintptr_t)scales + e2) & ~(uint64_t)3;
        asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, off" ::"s"(l0 + (rt * 2 + 0) * 256), "v"(a) : "memory");
      }
      if (has_z) {
        const uint64_t a = ((uint64_t)(uintptr_t)zeros + e2) & ~(uint64_t)3;
        asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, off" ::"s"(l0 + (rt * 2 + 1) * 256), "v"(a) : "memory");
      }
    }
  };
  auto sc_base = [&](int kb) { return addr::smallw_sc_base(kb, gshift); };
  auto new_period = [&](int kb) { return NS > 0 && addr::smallw_new_period(kb, kb0, gshift); };
  auto sc_buf = [&](int kb) { return addr::smallw_sc_buf(kb, gshift); };

  typename Mma::acc_t acc[RT][MT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = typename Mma::acc_t{0, 0, 0, 0};

  if (nkb > 0) {
    if (new_period(kb0)) issue_sc(sc_base(kb0), sc_buf(kb0));
    issue_kb(kb0, 0);
    if (nkb > 1) {
      if (new_period(kb0 + 1)) issue_sc(sc_base(kb0 + 1), sc_buf(kb0 + 1));
      issue_kb(kb0 + 1, 1);
    }
  }
  // The k-blocks from i0 on, dequantised with the zero points folded into the unpack bias (a quarter of the conversion
  // arithmetic less) while they are small integers in every lane (the usual case, the same bits): returns the first block
  // that is not, whose operands have landed and are still in its slot.  One copy of the loop per dequantiser: a choice inside
  // would make the two paths meet with the accumulators in different registers.
  auto run = [&](int i0, auto fold_tag) -> int {
    constexpr bool F = decltype(fold_tag)::value;
    for (int i = i0; i < nkb; ++i) {
      const int kb = kb0 + i;
      // everything issued for this k-block has landed once only the next k-block's loads are outstanding
      if (i + 1 < nkb) {
        if (new_period(kb + 1)) {
          if (NS == 1 * RT)
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI + RT) : "memory");
          else
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI + 2 * RT) : "memory");
        } else {
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI) : "memory");
        }
      } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      const uint8_t* slot = mine + (i & 1) * SLOT;
      T sv[RT], zv[RT];
      {
        const int g = addr::smallw_group(lane, kb, gshift);
        const uint8_t* sc = mine + 2 * SLOT + sc_buf(kb) * SC + addr::smallw_sc_cell(lane, kb, gshift) * 4;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          const uint32_t sh = (((uint32_t)row_g[rt] + (uint32_t)g) & 1u) * 16u;
          const uint32_t sa = (uint32_t)(((uintptr_t)scales >> 1) & 1), za = (uint32_t)(((uintptr_t)zeros >> 1) & 1);
          sv[rt] = one;
          zv[rt] = zs;
          if (has_s) {
            const uint32_t dw = *(const uint32_t*)(sc + (rt * 2 + 0) * 256);
            sv[rt] = bitcast<T>((uint16_t)(dw >> (sh ^ (sa * 16u))));
          }
          if (has_z) {
            const uint32_t dw = *(const uint32_t*)(sc + (rt * 2 + 1) * 256);
            zv[rt] = bitcast<T>((uint16_t)(dw >> (sh ^ (za * 16u))));
          }
        }
      }
      if (F && !FOLD) {
        bool ok = true;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          const float zf = to_float(zv[rt]);
          ok = ok && zf == __builtin_rintf(zf) && zf >= -256.0f && zf <= 256.0f;
        }
        if (__builtin_amdgcn_ballot_w64(ok) != ~0ull) return i;
      }
      uint4_t wf[RT], af[MT][4];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) wf[rt] = *(const uint4_t*)(slot + rt * 1024 + fo_w);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int j = 0; j < 4; ++j) af[mt][j] = *(const uint4_t*)(slot + fo_a[j] + mt * 4096);
      // the slot may be overwritten once its contents are in registers
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (i + 2 < nkb) {
        if (new_period(kb + 2)) issue_sc(sc_base(kb + 2), sc_buf(kb + 2));
        issue_kb(kb + 2, i & 1);
      }
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const Expand8<T, F, LAYOUT> ex(sv[rt], zv[rt], mg);
        const uint32_t w[4] = {wf[rt].x, wf[rt].y, wf[rt].z, wf[rt].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint4_t wop = ex(w[j]);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = Mma::mma(wop, af[mt][j], acc[rt][mt]);
        }
      }
    }
    return nkb;
  };
  const int done = run(0, std::true_type{});
  if (!FOLD && done < nkb) run(done, std::false_type{});

  // add the partial tiles of the wavefronts (the private regions are dead now)
  __syncthreads();
  float4_t* const red = (float4_t*)smem;  // [waves][RT * MT][64 lanes]
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) red[(wave * (RT * MT) + rt * MT + mt) * 64 + lane] = acc[rt][mt];
  __syncthreads();
  for (int item = threadIdx.x; item < RT * MT * 64; item += waves * 64) {
    float4_t sum = red[item];
    if (waves == 8) {  // (all asked for at once: one by one the reads wait for each other)
      float4_t part[7];
#pragma unroll
      for (int w = 1; w < 8; ++w) part[w - 1] = red[w * (RT * MT * 64) + item];
#pragma unroll
      for (int w = 1; w < 8; ++w) sum += part[w - 1];
    } else {
#pragma unroll 4
      for (int w = 1; w < waves; ++w) sum += red[w * (RT * MT * 64) + item];
    }
    const int tile = item >> 6, l = item & 63;
    const int rt = tile / MT, mt = tile - rt * MT;
    const int m = m_base + mt * 16 + (l & 15);
    const int n = n_base + rt * 16 + 4 * (l >> 4);
    if (m >= M || n >= N) continue;
    const int64_t idx = (int64_t)m * N + n;
    if (n + 3 < N && (N & 3) == 0) {
      if (out_dtype == TLQ_F32) {
        *(float4_t*)((float*)C + idx) = sum;
      } else if (out_dtype == TLQ_F16) {
        half_t h[4] = {(half_t)sum[0], (half_t)sum[1], (half_t)sum[2], (half_t)sum[3]};
        *(uint2_t*)((half_t*)C + idx) = bitcast<uint2_t>(h);
      } else {
        uint2_t o;
        o.x = pack_bf16x2(sum[0], sum[1]);
        o.y = pack_bf16x2(sum[2], sum[3]);
        *(uint2_t*)((uint16_t*)C + idx) = o;
      }
    } else {
      for (int i = 0; i < 4 && n + i < N; ++i) store_out(C, idx + i, sum[i], out_dtype);
    }
  }
}

// Tile, wavefronts per work-group (the cut of K) and an estimate of the call's time, or ok = false where the kernel does not
// apply.  The estimate: a launch, then rounds of the work-groups the machine holds at once (LDS and registers) x the longest
// chain of k-blocks in a wavefront, plus what a CU does for its share of the tiles: dequantising (the vector rate) and
// operand traffic and multiplications per 16 x 16 tile and k-block.  Fitted to 520 problems (M 2 .. 700, N 256 .. 14400,
// K 256 .. 14336, both types, groups of 64 and 128, zero-point tensor or scalar) x up to 24 forced variants each: 12 % rms over all
// variants; the variant it picks is 2.4 % behind the fastest on average.
static SmallTile small_plan_now(int64_t M, int64_t N, int64_t K, int force_waves, int force_rt, int force_mt);
SmallTile w4a16_small_plan(int64_t M, int64_t N, int64_t K, int64_t group, const void* scales, const void* zeros, int force_waves, int force_rt, int force_mt) {
  SmallTile best{false, 0, 0, 0, 0.0};
  if (M < 1 || N < 1 || K < 128 || K % 128 != 0 || group < 32 || (group & (group - 1)) != 0 || K % group != 0) return best;
  // (the scale / zero gathers read aligned dwords: the tensors must start and end on a dword boundary; 32-bit offsets)
  if ((((uintptr_t)scales | (uintptr_t)zeros) & 3) != 0 || ((N * (K / group)) & 1) != 0) return best;
  if (M * K * 2 >= ((int64_t)1 << 32) || N * (K / 2) >= ((int64_t)1 << 32) || N * (K / group) >= ((int64_t)1 << 31)) return best;
  static thread_local PlanTable<SmallTile> known;
  return known.get(M, N, K, force_waves * 100 + force_rt * 10 + force_mt, [&] { return small_plan_now(M, N, K, force_waves, force_rt, force_mt); });
}
static SmallTile small_plan_now(int64_t M, int64_t N, int64_t K, int force_waves, int force_rt, int force_mt) {
  SmallTile best{false, 0, 0, 0, 0.0};
  int cus = tlq_device_cu_count();
  if (cus <= 0) cus = 256;
  const int64_t KB = K / 128;
  for (int mt = 1; mt <= 4; mt *= 2) {
    if (force_mt ? mt != force_mt : mt > 1 && mt * 8 >= M) continue;  // (half of the tile would be padding)
    for (int rt = 1; rt <= 4; rt *= 2) {
      if (force_rt && rt != force_rt) continue;
      const int lds = small_wave_lds(rt, mt), most = 160 * 1024 / lds < small_max_waves(mt) ? 160 * 1024 / lds : small_max_waves(mt);
      const int64_t blocks = ceil_div(M, (int64_t)16 * mt) * ceil_div(N, (int64_t)16 * rt);
      if (blocks > 1 << 20) continue;
      for (int want = force_waves ? force_waves : 2; want <= (force_waves ? force_waves : 16); want *= 2) {
        int64_t w = want < most ? want : most;
        if (w > KB) w = KB;
        int64_t held = 160 * 1024 / (w * lds);
        const int64_t by_registers = mt == 1 ? 32 / w : 12 / w;
        if (held > by_registers) held = by_registers;
        if (held < 1) held = 1;
        const double rounds = (double)ceil_div(blocks, cus * held), per_cu = (double)ceil_div(blocks, (int64_t)cus) * (double)KB;
        const double us = 2.8 + rounds * (1.15 + 0.163 * (double)ceil_div(KB, w) + 0.034 * (double)w) + per_cu * (0.027 * rt + 0.0298 * rt * mt);
        if (!best.ok || us < best.us * 0.995) best = SmallTile{true, mt, rt, (int)w, us};
      }
    }
  }
  if (best.us < 5.0) best.us = 5.0;  // (the launch)
  return best;
}

struct SmallArgs {
  const void *A, *Wp, *scales, *zeros;
  void* C;
  int M, N, K, gshift;
  float zero_scalar;
  int out_dtype;
  const char* what;
  hipStream_t st;
};

template <typename T, bool FOLD, int LAYOUT, int RT, int MT>
static int launch_small(const SmallArgs& a, int waves) {
  auto kern = w4a16_small_kernel<T, FOLD, LAYOUT, RT, MT>;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) {
      set_error("%s: cannot reserve LDS: %s", a.what, hipGetErrorString(e));
      return 1;
    }
    attr_set = true;
  }
  const dim3 blocks((unsigned)ceil_div((int64_t)a.N, (int64_t)16 * RT), (unsigned)ceil_div((int64_t)a.M, (int64_t)16 * MT));
  kern<<<blocks, waves * 64, (size_t)waves * small_wave_lds(RT, MT), a.st>>>((const T*)a.A, (const uint8_t*)a.Wp, (const T*)a.scales, (const T*)a.zeros, a.C,
                                                                          a.M, a.N, a.K, a.gshift, a.zero_scalar, a.out_dtype, waves);
  return check_launch(a.what, LAYOUT == 1 ? "w4a16_small_kernel, interleaved words" : "w4a16_small_kernel") ? 0 : 1;
}

template <typename T, bool FOLD, int LAYOUT>
static int dispatch_small(const SmallArgs& a, const SmallTile& p) {
#define TLQ_SMALL(RT, MT) \
  if (p.rt == RT && p.mt == MT) return launch_small<T, FOLD, LAYOUT, RT, MT>(a, p.waves);
  TLQ_SMALL(1, 1) TLQ_SMALL(2, 1) TLQ_SMALL(4, 1) TLQ_SMALL(1, 2) TLQ_SMALL(2, 2) TLQ_SMALL(4, 2) TLQ_SMALL(1, 4) TLQ_SMALL(2, 4) TLQ_SMALL(4, 4)
#undef TLQ_SMALL
  set_error("%s: no such tile", a.what);
  return 1;
}

int gemm_w4a16_small(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t M, int64_t N, int64_t K, int64_t group,
                     float zero_scalar, int in_dtype, int out_dtype, int w_layout, const SmallTile& p, const char* what, hipStream_t st) {
  // An integer zero point shared by the whole matrix folds exactly into the unpack bias.
  const bool fold = zeros == nullptr && zero_scalar == (float)(int)zero_scalar && zero_scalar >= -256.0f && zero_scalar <= 256.0f;
  int gshift = 0;
  while (((int64_t)1 << gshift) < group) ++gshift;
  const SmallArgs a{A, Wp, scales, zeros, C, (int)M, (int)N, (int)K, gshift, zero_scalar, out_dtype, what, st};
#define TLQ_SMALL(T) \
  return fold ? (w_layout == TLQ_W_INTERLEAVED_F16 ? dispatch_small<T, true, 1>(a, p) : dispatch_small<T, true, 0>(a, p)) \
              : (w_layout == TLQ_W_INTERLEAVED_F16 ? dispatch_small<T, false, 1>(a, p) : dispatch_small<T, false, 0>(a, p));
  if (in_dtype == TLQ_F16) TLQ_SMALL(half_t)
  TLQ_SMALL(bf16_t)
#undef TLQ_SMALL
}

}  // namespace tlq
