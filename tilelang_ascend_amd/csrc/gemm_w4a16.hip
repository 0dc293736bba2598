// W4A16 prefill GEMM: packed-int4 weights are dequantised on their way from global memory
// into the LDS weight tile, then fp16 / bf16 MFMA with fp32 accumulation.
//
//   W[n, k] = rn_T( rn_T(T(u) - z) * s ),  C[m, n] = rn_out( sum_k A[m, k] * W[n, k] )
//
// The dequantised tile holds exactly the values of the stand-alone dequantisation kernel
// (one rounding per operation), so the GEMM result equals "dequantise, then fp32-accumulated
// matmul" up to summation order.
//
// One stage is 64 values of K: 32 packed bytes per weight row.  A thread loads 16 packed
// bytes (32 weights of one quantisation group) plus that group's scale / zero, and later
// expands them to four 16-byte LDS chunks.
//
// fp16 expansion, per 32-bit word (8 nibbles k0..k7):
//   (x    & 0x000f000f) | 0x64006400 -> half2 (1024+k0, 1024+k4)     one v_bfi_b32 each
//   (x    & 0x00f000f0) | 0x54005400 -> half2 (  64+k1,   64+k5)
//   (x>>8 & ...) likewise             -> (k2, k6), (k3, k7)
//   packed subtract of the bias (and of an integer zero point folded into it, exact), packed
//   multiply by the scale, then four v_perm_b32 put the halves back into k order.
// bf16 expansion: v_cvt_f32_ubyteN on the masked nibbles, fp32 fma / sub+mul with explicit
// bfloat16 roundings, v_cvt_pk_bf16_f32 to pack pairs in k order.
#include "gemm_core.h"
#include "expand8.h"
#include "small_tiles.h"

namespace tlq {

template <typename T, bool FOLD, int ROWS, int NT>
struct W4Loader {
  typedef RowFrag Frag;
  static constexpr bool DIRECT = false;
  static constexpr bool PREFETCH2 = true;  // convert from registers loaded one stage earlier
  static constexpr int SLOTS = ROWS * 2;  // 16-byte packed loads per stage
  static constexpr int PASSES = (SLOTS + NT - 1) / NT;
  static constexpr bool PARTIAL = SLOTS % NT != 0;
  static constexpr int UNITS = PASSES * 4;  // one unit = one 32-bit word -> one 16-byte LDS chunk
  static_assert(PASSES == 1 || (NT / 2) % 8 == 0, "pass stride must keep the swizzle phase");
  struct Params {
    const uint8_t* wp;
    const T* scales;  // never null: the host passes a dummy readable pointer when there are no scales
    const T* zeros;
    int row_bytes;    // K / 2
    int slice_bytes;  // split-K: packed bytes of one K slice (whole groups) within a row, 0 without a split; slice z is the kernel's "batch" z
    float zero_scalar;
    uint8_t group_shift;  // log2(group); group is a power of two here
    uint8_t has_scales, has_zeros;
  };
  struct Regs {
    uint4_t v[PASSES];
    uint32_t sz[PASSES];  // scale in the low half, zero point in the high half: 16-bit members of a struct that crosses
                          // a stage boundary are passed through scratch memory by the compiler (a round trip per stage)
  };
  const uint8_t* base;  // uniform: first packed row of the tile
  const T* sbase;       // uniform: scales / zeros row of the tile's first row
  const T* zbase;
  uint32_t voff[PASSES];  // per lane: row * row_bytes + half * 16
  uint32_t goff[PASSES];  // per lane: row * groups + (lane-fixed part of the group index)
  uint32_t loff[4];       // per lane: LDS offsets of the four chunks this lane writes (pass 0)
  int group_shift;
  bool has_s, has_z, active;
  T one, zs;
  NibbleMagic mg;

  __device__ __forceinline__ W4Loader(const Params& p, int batch, int row0, int rows_total, int tid)
      : base(p.wp + (int64_t)row0 * p.row_bytes + (int64_t)batch * p.slice_bytes), group_shift(p.group_shift),
        has_s(p.has_scales != 0), has_z(p.has_zeros != 0), one(from_float<T>(1.0f)), zs(from_float<T>(p.zero_scalar)),
        mg(make_nibble_magic()) {
    const int rows_valid = rows_total - row0;
    const int groups = 2 * p.row_bytes >> p.group_shift, slice_groups = 2 * p.slice_bytes >> p.group_shift;
    sbase = p.scales + (has_s ? (int64_t)row0 * groups + batch * slice_groups : 0);
    zbase = p.zeros + (has_z ? (int64_t)row0 * groups + batch * slice_groups : 0);
    const int half = tid & 1;
#pragma unroll
    for (int ps = 0; ps < PASSES; ++ps) {
      int row = (ps * NT + tid) >> 1;
      row = row < rows_valid ? row : rows_valid - 1;  // clamp: loads stay in bounds, results are masked later
      voff[ps] = (uint32_t)row * (uint32_t)p.row_bytes + (uint32_t)(half * 16);
      goff[ps] = (uint32_t)row * (uint32_t)groups + (uint32_t)((half * 32) >> group_shift);
    }
    const int r0 = tid >> 1;
#pragma unroll
    for (int j = 0; j < 4; ++j) loff[j] = (uint32_t)lds_off(r0, half * 4 + j);
    active = !PARTIAL || ((PASSES - 1) * NT + tid) < SLOTS;
  }

  // K is a multiple of 64 on this path, so every stage is complete (TAIL is never needed).
  // Group index of element (kt*64 + half*32) = ((kt*64) >> shift) + ((half*32) >> shift) for every
  // power-of-two group >= 32.
  template <bool TAIL>
  __device__ __forceinline__ void gload(Regs& r, int kt, uint8_t* /*lds_next*/ = nullptr) const {
    const uint8_t* sb = base + (int64_t)kt * 32;
    const uint32_t gk = (uint32_t)((kt * 64) >> group_shift);
#pragma unroll
    for (int ps = 0; ps < PASSES; ++ps) {
      r.v[ps] = *(const uint4_t*)(sb + voff[ps]);
      const T sv = sbase[has_s ? goff[ps] + gk : 0u];
      const T zv = zbase[has_z ? goff[ps] + gk : 0u];
      r.sz[ps] = (uint32_t)bitcast<uint16_t>(has_s ? sv : one) | ((uint32_t)bitcast<uint16_t>(has_z ? zv : zs) << 16);
    }
  }
  __device__ __forceinline__ void lstore_piece(const Regs& r, uint8_t* lds, int pc, int np) const {
#pragma unroll
    for (int ps = 0; ps < PASSES; ++ps) {
      if (PARTIAL && ps == PASSES - 1 && !active) continue;
      const Expand8<T, FOLD> ex(bitcast<T>((uint16_t)(r.sz[ps] & 0xffffu)), bitcast<T>((uint16_t)(r.sz[ps] >> 16)), mg);
      const uint32_t w[4] = {r.v[ps].x, r.v[ps].y, r.v[ps].z, r.v[ps].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if ((ps * 4 + j) * np / UNITS != pc) continue;
        *(uint4_t*)(lds + loff[j] + ps * (NT / 2) * kStageBytes) = ex(w[j]);
      }
    }
  }
  __device__ __forceinline__ void lstore(const Regs& r, uint8_t* lds) const { lstore_piece(r, lds, 0, 1); }
};

template <typename T>
struct MmaOf;
template <>
struct MmaOf<half_t> {
  typedef MmaF16 type;
};
template <>
struct MmaOf<bf16_t> {
  typedef MmaBF16 type;
};

template <int ROWS, int NT>
using W4LoaderF16Fold = W4Loader<half_t, true, ROWS, NT>;
template <int ROWS, int NT>
using W4LoaderF16Gen = W4Loader<half_t, false, ROWS, NT>;
template <int ROWS, int NT>
using W4LoaderBF16Fold = W4Loader<bf16_t, true, ROWS, NT>;
template <int ROWS, int NT>
using W4LoaderBF16Gen = W4Loader<bf16_t, false, ROWS, NT>;

struct W4Args {
  const void *A, *Wp, *scales, *zeros;
  void* C;
  int64_t M, N, K, group;
  float zero_scalar;
  int out_dtype;
  hipStream_t st;
  int64_t split = 1;         // K slices handled by different work-groups (the MFMA tile kernel only)
  float* partial = nullptr;  // [split][M][N] fp32 partial sums when split > 1
};

template <typename T, bool FOLD, int ROWS, int NT>
static typename W4Loader<T, FOLD, ROWS, NT>::Params w4_params(const W4Args& a) {
  int shift = 0;
  while (((int64_t)1 << shift) < a.group) ++shift;
  const T* dummy = (const T*)a.A;  // readable placeholder for absent scale / zero tensors
  return {(const uint8_t*)a.Wp,
          a.scales ? (const T*)a.scales : dummy,
          a.zeros ? (const T*)a.zeros : dummy,
          (int)(a.K / 2),
          a.split > 1 ? (int)(a.K / a.split / 2) : 0,
          a.zero_scalar,
          (uint8_t)shift,
          (uint8_t)(a.scales != nullptr),
          (uint8_t)(a.zeros != nullptr)};
}

template <typename T, bool FOLD, int BM, int BN, int WM, int WN>
static int run_w4a16(const W4Args& a) {
  constexpr int NT = WM * WN * 64;
  // activations travel global -> LDS directly whenever the tile splits into whole wavefront loads
  constexpr bool DIRECT = BM % 8 == 0 && (BM / 8) % (NT / 64) == 0;
  typedef typename std::conditional<DIRECT, RowLoaderDirect<DIRECT ? BM : 8 * (NT / 64), NT>, RowLoader<BM, NT>>::type AL;
  typedef W4Loader<T, FOLD, BN, NT> WL;
  auto pw = w4_params<T, FOLD, BN, NT>(a);
  if (a.split > 1) {
    // slice z of K is "batch" z of the loaders; every slice writes its own fp32 partial matrix
    const int64_t ks = a.K / a.split;
    typename AL::Params pa{(const uint8_t*)a.A, a.K * 2, ks * 2, ks * 2};
    EpiFloat::Params pe{a.partial, a.N, a.M * a.N, TLQ_F32};
    return launch_gemm<typename MmaOf<T>::type, AL, WL, EpiFloat, BM, BN, WM, WN>(pa, pw, pe, a.split, a.M, a.N, ks * 2, a.st,
                                                                                 "tlq_gemm_w4a16(mfma, split K)", 8);
  }
  typename AL::Params pa{(const uint8_t*)a.A, a.K * 2, 0, a.K * 2};
  EpiFloat::Params pe{a.C, a.N, 0, a.out_dtype};
  return launch_gemm<typename MmaOf<T>::type, AL, WL, EpiFloat, BM, BN, WM, WN>(pa, pw, pe, 1, a.M, a.N, a.K * 2, a.st,
                                                                               "tlq_gemm_w4a16(mfma)", 8);
}

// tile override for tuning runs (0 = automatic)
static thread_local int g_w4a16_tile = 0;

template <typename T, bool FOLD>
static int dispatch_w4a16(const W4Args& a) {
  int tile = g_w4a16_tile;
  const int64_t M = a.M, N = a.N;
  if (tile == 0) {
    if (M <= 16)
      tile = 16;
    else if (M <= 32)
      tile = 32;
    else if (M <= 64)
      tile = 64;
    else if (M <= 128 || (a.split <= 1 && prefer_small_tiles(1, M, N, 0.65)))
      tile = 128;  // few large tiles: smaller ones fill more CUs, unless K is being cut for that purpose
    else
      tile = 256;
  }
  switch (tile) {
    case 16:
      return run_w4a16<T, FOLD, 16, 64, 1, 4>(a);
    case 32:
      return run_w4a16<T, FOLD, 32, 128, 1, 4>(a);
    case 64:
      return run_w4a16<T, FOLD, 64, 256, 1, 4>(a);
    case 128:
      return run_w4a16<T, FOLD, 128, 128, 2, 2>(a);
    default:
      return run_w4a16<T, FOLD, 256, 256, 2, 4>(a);
  }
}

// ---- skinny kernel: a few activation rows (M <= 64) against a large weight matrix ---------------
// HBM bound: every packed weight is read once and goes straight from global memory through the
// dequantiser into an MFMA operand register; there is no LDS tile.  A wavefront owns RT tiles of 16
// weight rows and a slice of K; per 128 values of K ("k-block") lane (row r = lane % 16, k-group
// q = lane / 16) loads the 16 packed bytes of k = 128*kb + 32*q .. +31 of its row (one quantisation
// group, so one scale / zero per lane and k-block), expands them into four 8-value operands, and
// feeds four MFMAs whose activation operand holds A[m = lane % 16][the same 8 k] (the MFMA does not
// care which k a k-group holds as long as both operands agree).  The wavefronts of a work-group
// split K between them and add their partial tiles through LDS, so no global reduction is needed.
template <typename T, bool FOLD, int RT, int MT>
__global__ __launch_bounds__(MT >= 4 ? 512 : 1024) void w4a16_skinny_kernel(const T* __restrict__ A, const uint8_t* __restrict__ Wp,
                                                            const T* __restrict__ scales, const T* __restrict__ zeros,
                                                            void* __restrict__ C, int M, int N, int K, int group,
                                                            float zero_scalar, int out_dtype, int waves) {
  typedef typename MmaOf<T>::type Mma;
  extern __shared__ __align__(16) uint8_t smem[];
  float4_t* const red = (float4_t*)smem;  // [waves][RT * MT][64 lanes]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, q = lane >> 4;
  const int n_base = blockIdx.x * (16 * RT);
  const int groups = K / group;
  const int KB = K >> 7;
  const int kb0 = addr::small_first(wave, waves, KB), kb1 = addr::small_first(wave + 1, waves, KB);
  const bool has_s = scales != nullptr, has_z = zeros != nullptr;
  const T one = from_float<T>(1.0f), zs = from_float<T>(zero_scalar);
  const NibbleMagic mg = make_nibble_magic();

  uint32_t woff[RT], goff[RT], aoff[MT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    int n = n_base + rt * 16 + r16;
    n = n < N ? n : N - 1;  // clamp: loads stay in bounds, the rows are masked at the store
    woff[rt] = (uint32_t)n * (uint32_t)(K >> 1) + (uint32_t)(q * 16);
    goff[rt] = (uint32_t)n * (uint32_t)groups;
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    int m = mt * 16 + r16;
    m = m < M ? m : M - 1;
    aoff[mt] = ((uint32_t)m * (uint32_t)K + (uint32_t)(q * 32)) * 2u;
  }
  const T* const sp = has_s ? scales : A;  // absent tensors: read a valid dummy location, discard the value
  const T* const zp = has_z ? zeros : A;

  struct Block {
    uint4_t w[RT];
    uint32_t sz[RT];  // scale | zero point << 16 (16-bit struct members would travel through scratch memory)
    uint4_t a[MT][4];
  };
  auto load = [&](Block& b, int kb) {
    const uint32_t gi = (uint32_t)((kb * 128 + q * 32) / group);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      b.w[rt] = *(const uint4_t*)(Wp + woff[rt] + (uint32_t)kb * 64u);
      const T sv = sp[has_s ? goff[rt] + gi : 0u];
      const T zv = zp[has_z ? goff[rt] + gi : 0u];
      b.sz[rt] = (uint32_t)bitcast<uint16_t>(has_s ? sv : one) | ((uint32_t)bitcast<uint16_t>(has_z ? zv : zs) << 16);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int j = 0; j < 4; ++j) b.a[mt][j] = *(const uint4_t*)((const uint8_t*)A + aoff[mt] + (uint32_t)kb * 256u + j * 16);
  };

  typename Mma::acc_t acc[RT][MT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = typename Mma::acc_t{0, 0, 0, 0};
  auto compute = [&](const Block& b) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const Expand8<T, FOLD> ex(bitcast<T>((uint16_t)(b.sz[rt] & 0xffffu)), bitcast<T>((uint16_t)(b.sz[rt] >> 16)), mg);
      const uint32_t w[4] = {b.w[rt].x, b.w[rt].y, b.w[rt].z, b.w[rt].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint4_t wf = ex(w[j]);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = Mma::mma(wf, b.a[mt][j], acc[rt][mt]);
      }
    }
  };

  // A wavefront's slice of K is only a few k-blocks long, and one k-block of arithmetic is far
  // shorter than a trip to memory: issue the loads of DEPTH k-blocks at once, then compute them.
  // (Other wavefronts of the CU cover the time between chunks.)
  constexpr int DEPTH = MT == 1 ? 4 : (MT == 2 ? 2 : 1);
  Block b[DEPTH];
  for (int kb = kb0; kb < kb1; kb += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      const int k = kb + d < kb1 ? kb + d : kb1 - 1;  // past the slice: reload the last block, skip its arithmetic
      load(b[d], k);
    }
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
      if (kb + d < kb1) compute(b[d]);
  }

  // add the partial tiles of the wavefronts (they hold different slices of K)
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) red[(wave * (RT * MT) + rt * MT + mt) * 64 + lane] = acc[rt][mt];
  __syncthreads();
  for (int item = threadIdx.x; item < RT * MT * 64; item += waves * 64) {
    float4_t sum = red[item];
    for (int w = 1; w < waves; ++w) {
      const float4_t v = red[w * (RT * MT * 64) + item];
      sum[0] += v[0];
      sum[1] += v[1];
      sum[2] += v[2];
      sum[3] += v[3];
    }
    // lane l of a tile holds D[n = 4 * (l / 16) + i][m = l % 16]
    const int tile = item >> 6, l = item & 63;
    const int rt = tile / MT, mt = tile - rt * MT;
    const int m = mt * 16 + (l & 15);
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

static thread_local int g_skinny_waves = 0, g_skinny_rt = 0, g_skinny_mt = 0;  // tuning overrides (0 = automatic)

template <typename T, bool FOLD, int RT, int MT>
static int launch_skinny(const W4Args& a, int waves) {
  auto kern = w4a16_skinny_kernel<T, FOLD, RT, MT>;
  const int blocks = (int)ceil_div(a.N, 16 * RT);
  const size_t lds = (size_t)waves * RT * MT * 64 * sizeof(float4_t);
  kern<<<blocks, waves * 64, lds, a.st>>>((const T*)a.A, (const uint8_t*)a.Wp, (const T*)a.scales, (const T*)a.zeros, a.C,
                                          (int)a.M, (int)a.N, (int)a.K, (int)a.group, a.zero_scalar, a.out_dtype, waves);
  return check_launch("tlq_gemm_w4a16(skinny)", "w4a16_skinny_kernel") ? 0 : 1;
}

static thread_local int g_skinny_lds = -1;  // tuning override: 0 = never, 1 = whenever possible, -1 = automatic

template <typename T, bool FOLD>
static int dispatch_skinny(const W4Args& a) {
  const int64_t row_tiles = ceil_div(a.N, 16);
  const int KB = (int)(a.K / 128);
  // up to 16 rows and power-of-two groups: operands staged through wavefront-private LDS, which is the small-tile kernel with
  // tiles of 16 activation rows (more rows: only where a tuning hook asks for it)
  if (g_skinny_lds == 1 || (a.M <= 16 && g_skinny_lds != 0)) {
    const SmallTile p = w4a16_small_plan(a.M, a.N, a.K, a.group, a.scales, a.zeros, g_skinny_waves, g_skinny_rt, g_skinny_mt);
    if (p.ok)
      return gemm_w4a16_small(a.A, a.Wp, a.scales, a.zeros, a.C, a.M, a.N, a.K, a.group, a.zero_scalar, std::is_same<T, half_t>::value ? TLQ_F16 : TLQ_BF16, a.out_dtype,
                              TLQ_W_PLAIN, p, "tlq_gemm_w4a16(skinny)", a.st);
  }
  // enough wavefronts to keep every CU streaming: about 24 per CU over the whole grid, at least two k-blocks each
  // two row tiles per wavefront halve the activation loads per weight; worth it once there are plenty of rows
  int rt = g_skinny_rt ? g_skinny_rt : (row_tiles >= 512 ? 2 : 1);
  int waves = g_skinny_waves;
  if (!waves) {
    static int cus = 0;  // cached: one attribute query per process
    if (cus == 0) {
      int dev = 0;
      if (hipGetDevice(&dev) != hipSuccess ||
          hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    }
    const int64_t want = (int64_t)cus * 24;
    waves = 1;
    while (waves < 16 && row_tiles / rt * waves < want && KB / (waves * 2) >= 2) waves *= 2;
  }
  if (waves > KB) waves = KB < 1 ? 1 : KB;
  const int mt = a.M <= 16 ? 1 : (a.M <= 32 ? 2 : 4);
  const int max_waves = mt >= 4 ? 8 : 16;  // four activation tiles need 256 registers per lane
  if (waves > max_waves) waves = max_waves;
#define TLQ_SK(RTT, MTT) return launch_skinny<T, FOLD, RTT, MTT>(a, waves)
  if (rt == 2) {
    if (mt == 1) TLQ_SK(2, 1);
    if (mt == 2) TLQ_SK(2, 2);
    TLQ_SK(2, 4);
  }
  if (mt == 1) TLQ_SK(1, 1);
  if (mt == 2) TLQ_SK(1, 2);
  TLQ_SK(1, 4);
#undef TLQ_SK
}

int gemm_w4a16_skinny(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t M, int64_t N,
                      int64_t K, int64_t group, float zero_scalar, int in_dtype, int out_dtype, hipStream_t st) {
  const bool fold = zeros == nullptr && zero_scalar == (float)(int)zero_scalar && zero_scalar >= -256.0f &&
                    zero_scalar <= 256.0f;
  const W4Args a{A, Wp, scales, zeros, C, M, N, K, group, zero_scalar, out_dtype, st};
  if (in_dtype == TLQ_F16) return fold ? dispatch_skinny<half_t, true>(a) : dispatch_skinny<half_t, false>(a);
  return fold ? dispatch_skinny<bf16_t, true>(a) : dispatch_skinny<bf16_t, false>(a);
}

// C[i] = round(sum over the K slices of partial[z][i]), slices added in index order (so the result does not
// depend on which work-group finished first)
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float4_t* __restrict__ partial, void* __restrict__ C,
                                                           int64_t n4, int split, int out_dtype, int blocks) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (int64_t)blocks * 256) {
    float4_t v = partial[i];
#pragma unroll 8  // loads of eight slices in flight (with few outputs the pass is paced by their latency); same order of adds
    for (int z = 1; z < split; ++z) v += partial[(int64_t)z * n4 + i];
    if (out_dtype == TLQ_F16) {
      half_t h[4] = {(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
      ((uint2_t*)C)[i] = bitcast<uint2_t>(h);
    } else if (out_dtype == TLQ_BF16) {
      ((uint2_t*)C)[i] = uint2_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    } else {
      ((float4_t*)C)[i] = v;
    }
  }
}

// K slices for the tile kernel at small M, where the output tiles alone leave most of the chip idle and a
// work-group's run of stages is latency bound: aim at one to two work-groups per CU (measured best on the
// MLP shapes), slices of at least 512 values that are whole stages and whole quantisation groups.  1 = no split.
static thread_local int g_w4a16_split = 0;  // forced number of K slices for tuning runs (0 = automatic)
int w4a16_split_forced() { return g_w4a16_split; }
bool w4a16_tile_forced() { return g_w4a16_tile != 0; }
bool w4a16_skinny_forced() { return g_skinny_waves != 0 || g_skinny_rt != 0 || g_skinny_lds >= 0; }

int f16_split_choice(int64_t batch, int64_t M, int64_t N, int64_t K);  // gemm_f16.hip

int64_t w4a16_mid_split(int64_t M, int64_t N, int64_t K, int64_t group) {
  // Where cutting K pays (measured against the two passes on the MLP shapes): up to M = 512 always, up to
  // M = 2048 while the 256 x 256 output tiles would fill at most a quarter of the chip.
  const bool region = M > 16 && (M <= 512 || (M < 2048 && ceil_div(M, (int64_t)256) * ceil_div(N, (int64_t)256) <= 64));
  if (!region || (group & (group - 1)) != 0 || N % 4 != 0) return 1;
  // Above 512 rows the two passes are the alternative, and where their plain GEMM cuts K itself (few output tiles) they
  // are ahead of this kernel: M = 768, N = K = 5120: 66 against 89 us.
  // (Not where that GEMM would only halve rows of 13312 values or more: this kernel over four slices is 7 - 16 % ahead
  // there -- N = 4096, K = 14336, M = 1024: 146 against 163 us; N = 5120, K = 13824, M = 768: 136 against 159 us.)
  if (M > 512 && g_w4a16_split == 0) {
    const int plain_slices = f16_split_choice(1, M, N, K);
    if (plain_slices > 2 || (plain_slices == 2 && K < 13312)) return 1;
  }
  if (g_w4a16_split > 0) {
    const int64_t s = g_w4a16_split, unit0 = group > 64 ? group : 64;
    return (s <= 16 && K % s == 0 && (K / s) % unit0 == 0) ? s : 1;
  }
  const int64_t bm = M <= 32 ? 32 : (M <= 64 ? 64 : (M <= 128 ? 128 : 256)), bn = (M <= 32 || (M > 64 && M <= 128)) ? 128 : 256;
  const int64_t tiles = ceil_div(M, bm) * ceil_div(N, bn);
  const int64_t want = ceil_div((int64_t)(bm == 256 ? 256 : 512), tiles);  // one 256-row work-group fills a CU, two smaller ones do
  const int64_t unit = group > 64 ? group : 64;
  // a cut that leaves more than a third of the work-groups' places empty is not worth the partial sums (M = 1024,
  // N = 4096, K = 11008 = 2 x 43 x 128 can only be halved: 128 work-groups, 173 us against 147 us for the two passes)
  const int64_t places = bm == 256 ? 256 : 512;
  for (int64_t s = want < 16 ? want : 16; s >= 2; --s)
    if (K % s == 0 && (K / s) % unit == 0 && K / s >= 512) return (M > 256 && tiles * s * 3 < places * 2) ? 1 : s;
  return 1;
}

void launch_splitk_reduce(const float* partial, void* C, int64_t M, int64_t N, int split, int out_dtype, hipStream_t st) {
  const int64_t n4 = M * N / 4, want = ceil_div(n4, (int64_t)256);
  const int blocks = (int)(want > 65536 ? 65536 : want);
  splitk_reduce_kernel<<<blocks, 256, 0, st>>>((const float4_t*)partial, C, n4, split, out_dtype, blocks);
}

int gemm_w4a16_mfma_splitk(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t M,
                           int64_t N, int64_t K, int64_t group, float zero_scalar, int in_dtype, int out_dtype,
                           int64_t split, float* partial, hipStream_t st) {
  const bool fold = zeros == nullptr && zero_scalar == (float)(int)zero_scalar && zero_scalar >= -256.0f &&
                    zero_scalar <= 256.0f;
  W4Args a{A, Wp, scales, zeros, C, M, N, K, group, zero_scalar, out_dtype, st};
  a.split = split;
  a.partial = partial;
  int rc;
  if (in_dtype == TLQ_F16)
    rc = fold ? dispatch_w4a16<half_t, true>(a) : dispatch_w4a16<half_t, false>(a);
  else
    rc = fold ? dispatch_w4a16<bf16_t, true>(a) : dispatch_w4a16<bf16_t, false>(a);
  if (rc) return rc;
  launch_splitk_reduce(partial, C, M, N, (int)split, out_dtype, st);
  return check_launch("tlq_gemm_w4a16(split-K reduce)") ? 0 : 1;
}

int gemm_w4a16_mfma(const void* A, const void* Wp, const void* scales, const void* zeros, void* C, int64_t M, int64_t N,
                    int64_t K, int64_t group, float zero_scalar, int in_dtype, int out_dtype, hipStream_t st) {
  if ((group & (group - 1)) != 0) {
    set_error("tlq_gemm_w4a16(mfma): group=%lld must be a power of two", (long long)group);
    return 1;
  }
  // An integer zero point shared by the whole matrix folds exactly into the unpack bias.
  const bool fold = zeros == nullptr && zero_scalar == (float)(int)zero_scalar && zero_scalar >= -256.0f &&
                    zero_scalar <= 256.0f;
  const W4Args a{A, Wp, scales, zeros, C, M, N, K, group, zero_scalar, out_dtype, st};
  if (in_dtype == TLQ_F16) return fold ? dispatch_w4a16<half_t, true>(a) : dispatch_w4a16<half_t, false>(a);
  return fold ? dispatch_w4a16<bf16_t, true>(a) : dispatch_w4a16<bf16_t, false>(a);
}

}  // namespace tlq

extern "C" {
// Tuning hook used by the benchmark sweeps: forces the activation-tile height (16, 32, 64,
// 128, 256) of the W4A16 MFMA kernel; 0 restores the automatic choice.
void tlq_tune_w4a16_tile(int block_m) { tlq::g_w4a16_tile = block_m; }
// K slices of the tile kernel for 16 < M < 256 when a workspace is given (2..16, must divide K into whole
// stages and groups); 0 restores the automatic choice.
void tlq_tune_w4a16_split(int slices) { tlq::tuning_changed(), tlq::g_w4a16_split = slices < 0 ? 0 : slices; }
// Wavefronts per work-group (1..16, the in-group split of K) and 16-row weight tiles per wavefront
// (1 | 2) of the skinny W4A16 kernel; 0 restores the automatic choice.
void tlq_tune_w4a16_skinny(int waves, int row_tiles) {
  tlq::g_skinny_waves = (waves < 0 || waves > 16) ? 0 : waves;
  tlq::g_skinny_mt = row_tiles / 100 == 1 || row_tiles / 100 == 2 || row_tiles / 100 == 4 ? row_tiles / 100 : 0;
  row_tiles %= 100;
  tlq::g_skinny_rt = (row_tiles % 10 == 4) ? 4 : (row_tiles % 10 == 2) ? 2 : (row_tiles % 10 == 1 ? 1 : 0);
  tlq::g_skinny_lds = row_tiles >= 20 ? 1 : (row_tiles >= 10 ? 0 : -1);  // +10: registers only, +20: small tiles
}
}
