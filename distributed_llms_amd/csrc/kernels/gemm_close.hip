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
// us, close + product -> this, cold weights: RMS norms 2048 x 1024 5.3 -> 4.0, 6144 x 1024 + clipped GLU 7.5 -> 6.1, 5120 x 2560
// 9.9 -> 8.8, 15360 x 2560 + GLU 19.5 -> 18.1; layer norms 1536 x 1024 5.4 -> 4.2, 6144 x 1024 + gelu GLU 7.2 -> 6.3, 15360 x
// 2560 19.4 -> 18.5.  More rows cost each workgroup as many times the arithmetic: 4 rows at best equal (6144 x 1024 7.1 / 7.1),
// 2560 wide slower (15360 19.3 / 19.8), so that the launch of its own is kept for them.
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

// kind 1: RMS norms * (offset + w) (glu 0 or 2), 2: layer norms * w + b (glu 0 or 3); ob, bias: may be 0
void gemm_close(uintptr_t y, uintptr_t w, uintptr_t bias, int N, int K, int glu, float limit, int kind, uintptr_t x, uintptr_t o,
                uintptr_t ob, uintptr_t wp, uintptr_t bp, uintptr_t wn, uintptr_t bn, uintptr_t xo, float eps, float mult,
                float offset, uintptr_t stream) {
  DLLM_HOST_CHECK(kind == kRmsClose || kind == kLayerClose, "kind 1 or 2");
  DLLM_HOST_CHECK(K >= SK && K % SK == 0 && K <= 2560, "K: multiples of 64 up to 2560");
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
  // nontemporal weights as ops/gemm asks for them elsewhere: not where the whole of a model's stays in the Infinity Cache
#define DLLM_CL_R(RG_, GLU_, CL_, KM_, WV_)                                                                                  go(gemm_close_kernel<RG_, GLU_, (GLU_ != 0 || KM_ > 1024), WV_, CL_, KM_>, GLU_ ? RG_ * 4 : RG_ * 8, WV_)
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
    if (rg == 2) DLLM_CL_R(2, GLU_, CL_, KM_, 4);                                                                            \
    else if (rg == 3) DLLM_CL_R(3, GLU_, CL_, KM_, 4);                                                                       \
    else if (rg == 4) DLLM_CL_R(4, GLU_, CL_, KM_, 4);                                                                       \
    else if (rg == 6) DLLM_CL_R(6, GLU_, CL_, KM_, 4);                                                                       \
    else DLLM_CL_R(8, GLU_, CL_, KM_, 4);                                                                                    \
  } while (0)
#define DLLM_CL_K(CL_, GLU_)                                                                                              \
  do {                                                                                                                    \
    if (glu == 0 && K <= 1024) DLLM_CL_P(CL_, 1024);                                                                      \
    else if (glu == 0) DLLM_CL_P(CL_, 2560);                                                                              \
    else if (K <= 1024) DLLM_CL_G(GLU_, CL_, 1024);                                                                       \
    else DLLM_CL_G(GLU_, CL_, 2560);                                                                                      \
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
