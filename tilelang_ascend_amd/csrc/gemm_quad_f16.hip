// The four-wavefront kernel (gemm_quad.h) on tiles other than 256 x 256, 16-bit operands: kernels in a file of their own, so that the build compiles them
// beside the others.
#include "gemm_quad.h"

namespace tlq {

template <class Mma, int BM, int BN>
static int run(const void* A, const void* B, void* C, int64_t batch, int64_t M, int64_t N, int64_t K, int out_dtype, int b_layout, hipStream_t st) {
  const typename RowLoaderDirect<BM, 256>::Params pa((const uint8_t*)A, K * 2, M * K * 2, K * 2);
  const EpiFloat::Params pe(C, N, M * N, out_dtype);
  if (b_layout == TLQ_B_NK) {
    typedef RowLoaderDirect<BN, 256> WL;
    return launch_quad<Mma, WL, EpiFloat, BM, BN>(pa, typename WL::Params((const uint8_t*)B, K * 2, N * K * 2, K * 2), pe, batch, M, N, K * 2, st, "tlq_gemm_f16", 4);
  }
  return launch_quad<Mma, H16KNLoaderDirect<BN, 256>, EpiFloat, BM, BN>(pa, KNParams((const uint8_t*)B, N * 2, K * N * 2, K), pe, batch, M, N, K * 2, st, "tlq_gemm_f16", 4);
}

// variant: kQuad*; K a multiple of 64, two stages or more; N a multiple of 8 with weights [K, N]
int quad_gemm_f16(int variant, const void* A, const void* B, void* C, int64_t batch, int64_t M, int64_t N, int64_t K, int in_dtype, int out_dtype, int b_layout,
                  hipStream_t st) {
#define TLQ_RUN(BM, BN)                                                                                    \
  return in_dtype == TLQ_F16 ? run<MmaF16, BM, BN>(A, B, C, batch, M, N, K, out_dtype, b_layout, st)      \
                             : run<MmaBF16, BM, BN>(A, B, C, batch, M, N, K, out_dtype, b_layout, st);
  TLQ_QUAD_TILES(variant, TLQ_RUN)
#undef TLQ_RUN
}

}  // namespace tlq
