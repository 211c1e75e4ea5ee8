// The close of a sublayer -- norm of its output, sum with the float32 residual stream, norm in front of the next sublayer -- in
// the launch of the product that reads it: y[N] = norm(x').w[N, K]^T (+ bias, GLU), x' = x + norm(o + bias), for one row.
//
// A close of one row is a launch of one workgroup, 2.0-2.3 us for a round trip to memory and two sums behind it.  Here every
// workgroup of the product makes the row for itself, in waves of its own beside those that already stream the weights (4 waves:
// gemm_stream.h, CloseRow), and keeps it in LDS; workgroup 0 writes the new stream (to another buffer: the others still read the
// old one).  What is left of the close is the two sums and the barriers, behind a round trip that the first weights pay as well.
// The sums are in the order of the two launches (the row's places, and as many product waves with the same K-tiles as gemm_stream
// has), so that the new stream and the product have their bits.  (Twice the product waves under a GLU of up to 128 rows a workgroup:
// other bits, 4096 x 2560 8.3 for 8.9, but 8192 and 16384 x 2048 14.2 and 22.9 for 10.4 and 15.3.)
// The product's waves wait (a barrier) until the row's loads are issued: a CU's requests for lines are served in their order, and the row
// came behind the first weights, 0.4 to 1.2 us later.
// us, close + product -> this with weights and row issued together -> as it is, cold weights, RMS norms with a clipped GLU or without,
// layer norms with a gelu GLU or without:
//   K  512:  512 / 2048 4.4 / 4.7 -> 3.2 / 3.5 -> 3.0 / 3.1, + GLU 3072 5.4 -> 4.1 -> 3.7;  4.8 / 5.1 -> 3.6 / 3.9 -> 3.4 / 3.6, 5.5 -> 4.4 -> 3.8
//   K 1024:  2048 / 8192 5.1 / 7.1 -> 3.9 / 6.1 -> 3.3 / 5.4, + GLU 6144 7.0 -> 5.9 -> 5.2;  1536 5.4 -> 4.1 -> 3.6, 7.1 -> 6.2 -> 5.1
//   K 1536:  1536 / 4608 5.5 / 7.4 -> 5.1 / 6.4 -> 4.4 / 5.3, + GLU 9216 10.5 -> 9.7 -> 8.9;  6.0 / 7.7 -> 5.7 / 7.1 -> 5.0 / 5.9, 10.7 -> 10.1 -> 8.9
//   K 2048:  2048 / 6144 6.6 / 9.2 -> 5.8 / 8.3 -> 4.8 / 7.0;  7.0 / 9.6 -> 6.3 / 8.9 -> 5.4 / 7.3
//   K 2560:  2560 / 5120 7.7 / 9.8 -> 6.3 / 8.4 -> 5.5 / 7.4, + GLU 15360 19.0 -> 17.3 -> 16.6;  8.2 / 10.2 -> 7.0 / 9.1 -> 6.0 / 8.0, 19.2 -> 17.9 -> 16.6
//   K 3072:  3072 / 9216 8.4 / 15.1 -> 7.1 / 13.1 -> 6.2 / 12.7, + GLU 8192 / 16384 13.7 / 22.3 -> 12.2 / 20.6 -> 11.4 / 19.6;  8.9 / 15.5 -> 7.8 /
//   14.0 -> 6.8 / 13.0, 22.5 -> 21.0 -> 19.5
// A GLU with rows of 4 KiB is the exception: waves that start together ask a part of the memory channels (16384 x 2048 17.3 -> 14.6 -> 14.8,
// 17.4 -> 14.7 -> 15.4).
// Before that barrier every size between and past these that was tried (160, to 96 Mi weights) was as fast as the two launches at least.  Wider
// rows, in four pieces, won as
// much in most products (4096 x 4096 10.9 -> 10.3, 22016 x 4096 + GLU 35.7 -> 33.4), but some GLUs, where a few CUs have a second
// workgroup, lost: 18432 x 3584 26.7 -> 29.5, 14336 / 16384 / 18432 x 4096 27.0 / 28.9 / 31.0 -> 29.3 / 31.3 / 32.2.
// More rows cost each workgroup as many times the arithmetic: 4 rows at best equal (6144 x 1024 7.1 / 7.1), 2560 wide slower (15360
// 19.3 / 19.8), so that the launch of its own is kept for them.
#include "gemm_stream.h"
#include "launchers.h"

namespace dllm {

template <int RG, int GLU, bool NT, int WAVES, int CLOSE, int KMAX>
__global__ void __launch_bounds__((WAVES + CV) * 64) gemm_close_kernel(bf16* __restrict__ Y, const bf16* __restrict__ W,
                                                                       const bf16* __restrict__ bias, int N, int K, float limit,
                                                                       CloseArgs close) {
  gemm_stream_body<RG, 1, GLU, NT, WAVES, CLOSE, KMAX>(Y, nullptr, W, bias, 1, N, K, limit, close);
}

int stream_rows(int ncols, int K, bool glu, int xg);
bool stream_wide(int m, int ncols, int rg);

// kind 1: RMS norms * (offset + w) (glu 0 or 2), 2: layer norms * w + b (glu 0 or 3); ob, bias: may be 0; nt: nontemporal weight
// loads.  Rows of one piece of 4 elements per lane (K <= 1024) or of up to three (3072).
void gemm_close(uintptr_t y, uintptr_t w, uintptr_t bias, int N, int K, int glu, int nt, float limit, int kind, uintptr_t x, uintptr_t o,
                uintptr_t ob, uintptr_t wp, uintptr_t bp, uintptr_t wn, uintptr_t bn, uintptr_t xo, float eps, float mult,
                float offset, uintptr_t stream) {
  DLLM_HOST_CHECK(kind == kRmsClose || kind == kLayerClose, "kind 1 or 2");
  DLLM_HOST_CHECK(K >= SK && K % SK == 0 && K <= 3072, "K: multiples of 64 up to 3072");
  DLLM_HOST_CHECK(glu == 0 || glu == (kind == kRmsClose ? 2 : 3), "a clipped GLU behind RMS norms, a gelu GLU behind layer norms");
  DLLM_HOST_CHECK(N >= 1 && (glu == 0 || N % 2 == 0), "N");
  DLLM_HOST_CHECK(x && o && wp && wn && xo && x != xo && (kind != kLayerClose || (bp && bn)), "close operands");
  DLLM_HOST_CHECK(w % 16 == 0 && y % 8 == 0 && (x | xo) % 16 == 0 && (o | ob | wp | bp | wn | bn) % 8 == 0, "operand alignment");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int ncols = glu ? N / 2 : N, rg = stream_rows(ncols, K, glu != 0, 1);
  const bool wide = glu == 0 && stream_wide(1, ncols, rg);
  const CloseArgs c{(const float*)x, (const bf16*)o, (const bf16*)ob, (const bf16*)wp, (const bf16*)bp, (const bf16*)wn,
                    (const bf16*)bn, (float*)xo, eps, mult, offset};
  const auto go = [&](auto kern, int per, int waves) {
    hipLaunchKernelGGL(kern, dim3((ncols + per - 1) / per), dim3((waves + CV) * 64), 0, s, (bf16*)y, (const bf16*)w,
                       (const bf16*)bias, N, K, limit, c);
  };
#define DLLM_CL_R(RG_, GLU_, CL_, KM_, WV_)                                                                               \
  do {                                                                                                                    \
    if (nt) go(gemm_close_kernel<RG_, GLU_, true, WV_, CL_, KM_>, GLU_ ? RG_ * 4 : RG_ * 8, WV_);                         \
    else go(gemm_close_kernel<RG_, GLU_, false, WV_, CL_, KM_>, GLU_ ? RG_ * 4 : RG_ * 8, WV_);                           \
  } while (0)
#define DLLM_CL_P(CL_, KM_)                                                                                               \
  do {                                                                                                                    \
    if (rg == 1) DLLM_CL_R(1, 0, CL_, KM_, 8);                       /* (a second round is never worth eight rows) */     \
    else if (rg == 2 && wide) DLLM_CL_R(2, 0, CL_, KM_, 8);                                                               \
    else if (rg == 2) DLLM_CL_R(2, 0, CL_, KM_, 4);                                                                       \
    else if (rg == 3 && wide) DLLM_CL_R(3, 0, CL_, KM_, 8);                                                               \
    else if (rg == 3) DLLM_CL_R(3, 0, CL_, KM_, 4);                                                                       \
    else DLLM_CL_R(4, 0, CL_, KM_, 4);                                                                                    \
  } while (0)
#define DLLM_CL_G(GLU_, CL_, KM_)                                                                                         \
  do {                                                                                                                    \
    if (rg == 2) DLLM_CL_R(2, GLU_, CL_, KM_, 4);                                                                         \
    else if (rg == 3) DLLM_CL_R(3, GLU_, CL_, KM_, 4);                                                                    \
    else if (rg == 4) DLLM_CL_R(4, GLU_, CL_, KM_, 4);                                                                    \
    else if (rg == 6) DLLM_CL_R(6, GLU_, CL_, KM_, 4);                                                                    \
    else DLLM_CL_R(8, GLU_, CL_, KM_, 4);                                                                                 \
  } while (0)
#define DLLM_CL_K(CL_, GLU_)                                                                                              \
  do {                                                                                                                    \
    if (glu == 0 && K <= 1024) DLLM_CL_P(CL_, 1024);                                                                      \
    else if (glu == 0) DLLM_CL_P(CL_, 3072);                                                                              \
    else if (K <= 1024) DLLM_CL_G(GLU_, CL_, 1024);                                                                       \
    else DLLM_CL_G(GLU_, CL_, 3072);                                                                                      \
  } while (0)
  if (kind == kRmsClose) DLLM_CL_K(kRmsClose, 2);
  else DLLM_CL_K(kLayerClose, 3);
#undef DLLM_CL_K
#undef DLLM_CL_G
#undef DLLM_CL_P
#undef DLLM_CL_R
  DLLM_HIP_CHECK(hipGetLastError());
}

}  // namespace dllm
