// Weight-streaming GEMM for decode batches of up to 64 rows: y[M, N] = x[M, K] . w[N, K]^T, bf16 in, f32 sums, with
// the bias, the SiLU, clipped or gelu GLU in the epilogue -- one launch where the wide kernel's K-split grid needs a
// second one to sum its slabs and (behind a bias) a third for the activation.
//
// At these sizes a projection of a 1k-4k wide model is a few microseconds of weight bytes, and every further launch
// (a slab sum, a gate kernel) costs 2-4 us: the end of one kernel to the start of the next inside a graph, plus its first
// load's round trip.  Where it is the faster route: ops/gemm.stream_fits.
//
//  * one workgroup owns 8 RG weight rows (stream_rows) and all of K, so nothing is left to sum in memory; its waves take the
//    64-deep K-tiles in turn (wave v: tiles v, v + WAVES, ...), so that together they read 512-byte or 1 KiB runs of
//    every row;
//  * a wave stages its tiles -- weights and x -- through an LDS ring of its OWN (two slots, global_load_lds_dwordx4 in
//    whole 128-byte lines, the chunk swizzle c ^ ((row >> 1) & 7) on the source address and on the read): no barrier
//    in the K loop, the only waits are the wave's counted vmcnt.  x fragments straight from global memory touch 16
//    half lines per load and took 1.3-2x as long at 16-64 rows (2560 x 2560: 8.1 / 12.4 / 19.2 us at M = 16 / 32 / 64
//    against 5.9 / 7.4 / 9.7);
//  * the waves' sums meet in LDS (wave 0 first: the same result on every run), behind the only two barriers.
// Measured, cold weights, M = 1 / 16 / 32 / 64, us (wide: gemm_wide's K split, without the reduction behind it):
//   1024 x 1024  3.0 / 3.5 / 4.0 / 5.1 (wide 5.0 / 5.4 / 5.5 / 5.6)    2560 x 2560  4.6 / 5.8 / 7.4 / 9.7 (6.7 / 7.2 / 7.7 / 8.2)
//   5120 x 2560  7.0 / 7.5 / 9.7 / 12.5 (7.9 / 8.5 / 9.0 / 9.6)        15360 x 2560 + GLU  14.6 / 14.8 / 16.2 / 19.7 (15.8 / 16.5 / 17.5 / 18.5)
//   4096 x 4096  7.6 / 8.6 / 10.0 / 13.2 (7.8 / 8.1 / 8.5 / 8.9)       6144 x 4096  10.4 / 10.1 (10.7 / 11.0)
// bound by the weight bytes and the launch below 16 rows, by staging x once per workgroup above.
#include "gemm_stream.h"
#include "launchers.h"

namespace dllm {

template <int RG, int XG, int GLU, bool NT, int WAVES>
__global__ void __launch_bounds__(WAVES * 64) gemm_stream_kernel(bf16* __restrict__ Y, const bf16* __restrict__ X,
                                                                 const bf16* __restrict__ W,
                                                                 const bf16* __restrict__ bias, int M, int N, int K,
                                                                 float limit) {
  gemm_stream_body<RG, XG, GLU, NT, WAVES, kNoClose, 64>(Y, X, W, bias, M, N, K, limit, CloseArgs{});
}

// Groups of 8 weight rows per workgroup up to 16 rows of x: the fewest rows (weights and x) that a CU has to stage.  What a CU
// takes in does not grow with its waves, so the time is that of the CU with the most rows:
// ceil(workgroups / 256) (RG + XG).  Where a weight row is a multiple of 4 KiB the lines of 32 and, more so, 64 rows that walk
// K in step fall on few memory channels: their rows count 1.24 and 1.6 times.  us, M = 1 / 16, 16-row tiles (32 from 256 tiles
// on) -> this: 1024 x 3072 4.8 / 6.1 -> 4.4 / 5.3, 2048 x 2048 4.5 / 5.1 -> 4.1 / 4.6, 2048 x 8192 10.5 / 12.0 -> 8.3 / 9.5,
// 5120 x 2560 8.0 / 8.2 -> 7.0 / 7.5, 6144 x 4096 13.0 / 13.8 -> 10.3 / 10.1; GLU 8192 x 2048 9.0 / 9.3 -> 8.0 / 9.3, 10240 x
// 2560 11.7 / 12.7 -> 10.9 / 11.3, 16384 x 4096 28.3 / 28.1 -> 23.6 / 25.6, 22016 x 4096 39.9 / 39.6 -> 30.0 / 29.7.
int stream_rows(int ncols, int K, bool glu, int xg) {
  int best = 0;
  float at = 0.f;
  for (const int rg : {8, 6, 4, 3, 2, 1}) {
    if (glu ? rg == 1 : rg > 4) continue;
    const int cols = glu ? rg * 4 : rg * 8, wgs = (ncols + cols - 1) / cols;
    const float t = (float)((wgs + 255) / 256) * (float)(rg + xg) * (K % 2048 ? 1.f : rg == 8 ? 1.6f : rg == 4 ? 1.24f : 1.f);
    if (best == 0 || t < at) best = rg, at = t;
  }
  return best;
}

// 8 waves for a plain product where up to three groups of its rows have a CU each: their K loop is over in one or two rounds; else
// 4 (several workgroups per CU).  Which wave has which K-tiles is the order of the sums.
bool stream_wide(int m, int ncols, int rg) {
  return m <= 16 ? rg <= 3 && (ncols + rg * 8 - 1) / (rg * 8) <= 256 : rg == 2 && m <= 32;
}

// glu 0: y [M, N] = x w^T (+ bias);  1 / 2 / 3: y [M, N / 2], SiLU / clipped / gelu GLU of w = [gate; up] (+ bias).
// 4: y [M, N] in float32, cap tanh(z / cap) of the rounded product z with cap = limit, z itself where that is not positive.
// (A launch of their own read the rounded logits back and wrote 4 bytes each: 1.6 to 2 us of a step whose head's product takes
// 12.4; the epilogue's threads have them in registers.  The sums keep their order, so the logits their bits.)
// nt: nontemporal weight loads.
void gemm_stream(uintptr_t y, uintptr_t x, uintptr_t w, uintptr_t bias, int M, int N, int K, int glu, int nt, float limit,
                 uintptr_t stream) {
  DLLM_HOST_CHECK(M >= 1 && M <= 64, "1 <= M <= 64");
  DLLM_HOST_CHECK(K >= SK && K % SK == 0, "K must be a positive multiple of 64");
  DLLM_HOST_CHECK(glu >= 0 && glu <= 4, "glu 0..4");
  const bool pair = glu >= 1 && glu <= 3;
  DLLM_HOST_CHECK(N >= 1 && (!pair || N % 2 == 0), "N");
  DLLM_HOST_CHECK(x % 16 == 0 && w % 16 == 0 && y % (glu == 4 ? 16 : 8) == 0, "operand alignment");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int ncols = pair ? N / 2 : N;
  const bool one = M <= 16;
  const int xg = M <= 8 ? 1 : M <= 16 ? 2 : M <= 32 ? 4 : 8;
  int rg;
  if (one) {
    rg = stream_rows(ncols, K, pair, xg);
  } else {
    // twice the weight rows per workgroup (half the x staging) once that still leaves a workgroup for most CUs
    const bool two = (ncols + 15) / 16 > 256;
    rg = (pair ? 4 : 2) * (two ? 2 : 1);
  }
  const int per = pair ? rg * 4 : rg * 8;
  const dim3 grid((ncols + per - 1) / per);
  const bool wide = !pair && stream_wide(M, ncols, rg);
#define DLLM_ST_GO(RG_, XG_, GLU_, WV_)                                                                             \
  do {                                                                                                              \
    if (nt) hipLaunchKernelGGL((gemm_stream_kernel<RG_, XG_, GLU_, true, WV_>), grid, dim3(WV_ * 64), 0, s,         \
                               (bf16*)y, (const bf16*)x, (const bf16*)w, (const bf16*)bias, M, N, K, limit);          \
    else hipLaunchKernelGGL((gemm_stream_kernel<RG_, XG_, GLU_, false, WV_>), grid, dim3(WV_ * 64), 0, s,           \
                            (bf16*)y, (const bf16*)x, (const bf16*)w, (const bf16*)bias, M, N, K, limit);             \
  } while (0)
#define DLLM_ST_P(RG_, XG_)                                                                                         \
  do {                                                                                                              \
    constexpr int W8 = RG_ <= 3 && XG_ <= 4 ? 8 : 4;                                                                  \
    if (wide) DLLM_ST_GO(RG_, XG_, 0, W8); else DLLM_ST_GO(RG_, XG_, 0, 4);                                            \
  } while (0)
#define DLLM_ST_C(RG_, XG_)                                                                                         \
  do {                                                                                                              \
    constexpr int W8 = RG_ <= 3 && XG_ <= 4 ? 8 : 4;                                                                  \
    if (wide) DLLM_ST_GO(RG_, XG_, 4, W8); else DLLM_ST_GO(RG_, XG_, 4, 4);                                            \
  } while (0)
#define DLLM_ST_G(RG_, XG_)                                                                                         \
  do {                                                                                                              \
    if (glu == 1) DLLM_ST_GO(RG_, XG_, 1, 4); else if (glu == 2) DLLM_ST_GO(RG_, XG_, 2, 4); else DLLM_ST_GO(RG_, XG_, 3, 4); \
  } while (0)
#define DLLM_ST_X(DO_, RG_)                                                                                         \
  do {                                                                                                              \
    if (xg == 1) DO_(RG_, 1); else DO_(RG_, 2);                                                                       \
  } while (0)
#define DLLM_ST_M(DO_, RG_)                                                                                         \
  do {                                                                                                              \
    if (xg == 1) DO_(RG_, 1); else if (xg == 2) DO_(RG_, 2); else if (xg == 4) DO_(RG_, 4); else DO_(RG_, 8);            \
  } while (0)
  if (glu == 0) {
    if (rg == 1) DLLM_ST_X(DLLM_ST_P, 1);
    else if (rg == 2) DLLM_ST_M(DLLM_ST_P, 2);
    else if (rg == 3) DLLM_ST_X(DLLM_ST_P, 3);
    else DLLM_ST_M(DLLM_ST_P, 4);
  } else if (glu == 4) {
    if (rg == 1) DLLM_ST_X(DLLM_ST_C, 1);
    else if (rg == 2) DLLM_ST_M(DLLM_ST_C, 2);
    else if (rg == 3) DLLM_ST_X(DLLM_ST_C, 3);
    else DLLM_ST_M(DLLM_ST_C, 4);
  } else {
    if (rg == 2) DLLM_ST_X(DLLM_ST_G, 2);
    else if (rg == 3) DLLM_ST_X(DLLM_ST_G, 3);
    else if (rg == 4) DLLM_ST_M(DLLM_ST_G, 4);
    else if (rg == 6) DLLM_ST_X(DLLM_ST_G, 6);
    else DLLM_ST_M(DLLM_ST_G, 8);
  }
#undef DLLM_ST_M
#undef DLLM_ST_X
#undef DLLM_ST_G
#undef DLLM_ST_C
#undef DLLM_ST_P
#undef DLLM_ST_GO
  DLLM_HIP_CHECK(hipGetLastError());
}

}  // namespace dllm
