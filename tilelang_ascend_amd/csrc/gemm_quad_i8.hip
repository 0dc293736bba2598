// The four-wavefront kernel (gemm_quad.h) on tiles other than 256 x 256, int8 operands: kernels in a file of their own, so that the build compiles them
// beside the others.
#include "gemm_quad.h"

namespace tlq {

template <class Epi, int BM, int BN>
static int run(const void* A, const void* B, const typename Epi::Params& pe, int64_t batch, int64_t M, int64_t N, int64_t K, int b_layout, hipStream_t st, const char* what) {
  const typename RowLoaderDirect<BM, 256>::Params pa((const uint8_t*)A, K, M * K, K);
  if (b_layout == TLQ_B_NK) {
    typedef RowLoaderDirect<BN, 256> WL;
    return launch_quad<MmaI8, WL, Epi, BM, BN>(pa, typename WL::Params((const uint8_t*)B, K, N * K, K), pe, batch, M, N, K, st, what, 2);
  }
  return launch_quad<MmaI8, I8KNLoaderDirect<BN, 256>, Epi, BM, BN>(pa, KNParams((const uint8_t*)B, N, K * N, K), pe, batch, M, N, K, st, what, 2);
}

// variant: kQuad*; K a multiple of 128, two stages or more
template <class Epi>
int quad_gemm_i8(int variant, const void* A, const void* B, const typename Epi::Params& pe, int64_t batch, int64_t M, int64_t N, int64_t K, int b_layout, hipStream_t st,
                 const char* what) {
#define TLQ_RUN(BM, BN) return run<Epi, BM, BN>(A, B, pe, batch, M, N, K, b_layout, st, what);
  TLQ_QUAD_TILES(variant, TLQ_RUN)
#undef TLQ_RUN
}
template int quad_gemm_i8<EpiInt32>(int, const void*, const void*, const EpiInt32::Params&, int64_t, int64_t, int64_t, int64_t, int, hipStream_t, const char*);
template int quad_gemm_i8<EpiRescale>(int, const void*, const void*, const EpiRescale::Params&, int64_t, int64_t, int64_t, int64_t, int, hipStream_t, const char*);

}  // namespace tlq
