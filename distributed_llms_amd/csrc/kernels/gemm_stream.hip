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
#include "common.h"
#include "launchers.h"

namespace dllm {

namespace {
typedef __attribute__((address_space(3))) void* lds_vptr_s;
typedef __attribute__((address_space(1))) void* glb_vptr_s;
constexpr int SK = 64;                    // K-tile
constexpr int D = 2;                      // slots of a wave's ring

__device__ __forceinline__ int sswz(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }
}  // namespace

// GLU 0: y [M, N] (+ bias [N]);  1 / 2 / 3: SiLU / clipped (`limit`) / gelu GLU, w = [gate; up], y [M, N / 2], bias
// gate | up.  A workgroup's RG groups of 8 weight rows are its output columns, under a GLU CW gate rows and then the same
// columns' up rows; XG groups of 8 rows of x.  An odd last group fills half an MFMA tile, its other half repeats it.
template <int RG, int XG, int GLU, bool NT, int WAVES>
__global__ void __launch_bounds__(WAVES * 64) gemm_stream_kernel(bf16* __restrict__ Y, const bf16* __restrict__ X,
                                                                 const bf16* __restrict__ W,
                                                                 const bf16* __restrict__ bias, int M, int N, int K,
                                                                 float limit) {
  static_assert(GLU == 0 || RG % 2 == 0 || RG == 3, "a GLU's CW is a multiple of 4");
  constexpr int RT = (RG + 1) / 2, MT = (XG + 1) / 2;
  constexpr int SLOT = (RG + XG) * 8 * SK;                      // bf16 elements of one ring slot: weights, then x
  constexpr int G = RG + XG;                                    // loads per K-tile
  constexpr int RING = WAVES * D * SLOT * 2, RED = WAVES * RT * MT * 1024;
  static_assert(G <= 63, "vmcnt");
  __shared__ __attribute__((aligned(16))) char smem[RING > RED ? RING : RED];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fq = lane >> 4;
  const int half = N / 2, ncols = GLU ? half : N;
  constexpr int CW = GLU ? RG * 4 : RG * 8;                     // output columns
  const int c0 = blockIdx.x * CW;
  bf16* ring = reinterpret_cast<bf16*>(smem) + wv * (D * SLOT);

  // weight row of row r of the workgroup; rows past the matrix repeat its last row
  auto wrow = [&](int r) {
    const bool up = GLU && r >= CW;
    return (up ? half : 0) + min(c0 + (up ? r - CW : r), ncols - 1);
  };
  // The bias of the epilogue: of the GLU that has one in its models, loaded here, so that no round trip is left for the end, off
  // a place that is there and in its stored form, since a load behind a branch or next to its conversion is waited for at
  // once.  (The others load theirs behind one branch: loads that nobody needs cost 0.1 us.)  us, behind a `bias ?` of its own
  // for each of a thread's eight loads -> this, M = 1 / 16: 6144 x 1024 + clipped GLU 5.18 / 5.55 -> 4.79 / 5.18, 15360 x 2560
  // 16.5 / 15.9 -> 16.2 / 15.6; 2560 x 2560 plain 4.96 / 6.15 -> 4.80 / 5.92.
  constexpr int TH = WAVES * 64, EL = CW / 4 * MT * 16, NE = (EL + TH - 1) / TH;
  bf16 eb[NE][GLU ? 8 : 4] = {};
  auto load_bias = [&](const bf16* bs, int n) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int cc = min(c0 + 4 * (((tid + n * TH) >> 4) % (CW / 4)) + v, ncols - 1);
      eb[n][v] = bs[bias ? cc : 0];
      if constexpr (GLU != 0) eb[n][4 + v] = bs[bias ? half + cc : 0];
    }
  };
  if constexpr (GLU == 2) {
#pragma unroll
    for (int n = 0; n < NE; ++n) load_bias(bias ? bias : X, n);
    __builtin_amdgcn_sched_barrier(0);
  }
  const bf16* src[G];
#pragma unroll
  for (int q = 0; q < G; ++q) {
    const int r = 8 * (q < RG ? q : q - RG) + (lane >> 3);
    const bf16* row = q < RG ? W + (size_t)wrow(r) * K : X + (size_t)min(r, M - 1) * K;
    src[q] = row + wv * SK + sswz(r, lane & 7) * 8;
  }
  const int nk = K / SK, cnt = (nk - wv + WAVES - 1) / WAVES;     // this wave's K-tiles (0 for a short K)
  f32x4 acc[RT][MT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto load = [&](int slot, int i) {
    const int ko = i * (WAVES * SK);
#pragma unroll
    for (int q = 0; q < RG; ++q)
      __builtin_amdgcn_global_load_lds((glb_vptr_s)(src[q] + ko), (lds_vptr_s)(ring + slot * SLOT + q * 512), 16, 0,
                                       NT ? 2 : 0);
#pragma unroll
    for (int q = RG; q < G; ++q)
      __builtin_amdgcn_global_load_lds((glb_vptr_s)(src[q] + ko), (lds_vptr_s)(ring + slot * SLOT + q * 512), 16, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int u = 0; u < D; ++u)
    if (u < cnt) load(u, u);
  for (int i0 = 0; i0 < cnt; i0 += D) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      const int i = i0 + u;                                       // wave-uniform
      if (i < cnt) {
        // tile i has landed when only the younger tile's loads are left, if there is one
        if (i + 1 < cnt) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(G) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const bf16* b = ring + u * SLOT;
        bf16x8 wa[RT][2], xa[MT][2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
          for (int t = 0; t < RT; ++t) {
            const int r = 2 * t + 1 < RG ? fr : fr & 7;
            wa[t][s] = *reinterpret_cast<const bf16x8*>(b + t * 1024 + r * SK + sswz(r, 4 * s + fq) * 8);
          }
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            const int r = 2 * m + 1 < XG ? fr : fr & 7;
            xa[m][s] = *reinterpret_cast<const bf16x8*>(b + RG * 512 + m * 1024 + r * SK + sswz(r, 4 * s + fq) * 8);
          }
        }
        // every fragment of the slot is in registers before its refill goes out
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (i + D < cnt) load(u, i + D);
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int m = 0; m < MT; ++m)
              acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[t][s], xa[m][s], acc[t][m], 0, 0, 0);
      }
    }
  }
  __syncthreads();
  // acc[t][m]: lane holds weight rows 4 fq + v of tile t, x row m 16 + fr
  f32x4* red = reinterpret_cast<f32x4*>(smem);
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) red[(wv * RT * MT + t * MT + m) * 64 + lane] = acc[t][m];
  __syncthreads();
  // four columns of one row each: rows R .. R + 3 of the workgroup in tile R / 16, lane group R / 4 % 4
#pragma unroll
  for (int n = 0; n < NE; ++n) {
    const int e = tid + n * TH;
    if (e >= EL) break;
    const int m = e / (CW * 4), R = 4 * ((e >> 4) % (CW / 4)), U = CW + R;
    const int at = ((R >> 4) * MT + m) * 64 + ((R >> 2) & 3) * 16 + (e & 15);
    f32x4 a = red[at], b = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 1; w < WAVES; ++w) a += red[w * RT * MT * 64 + at];
    if constexpr (GLU != 0) {
      const int up = ((U >> 4) * MT + m) * 64 + ((U >> 2) & 3) * 16 + (e & 15);
#pragma unroll
      for (int w = 0; w < WAVES; ++w) b += red[w * RT * MT * 64 + up];
    }
    const int row = m * 16 + (e & 15), c = c0 + R;
    if (row >= M || c >= ncols) continue;
    bf16x4 o;
    if (GLU != 2 && bias) load_bias(bias, n);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float z = a[v] + (bias ? bf2f(eb[n][v]) : 0.f);
      if constexpr (GLU != 0) {
        const float up = b[v] + (bias ? bf2f(eb[n][4 + v]) : 0.f);
        // (a projection, a bias and a gate kernel until they met here: the gate kernels' arithmetic)
        z = GLU == 1 ? silu_f(z) * up : GLU == 2 ? clipped_glu_exact_f(z, up, limit, kGluAlpha) : gelu_glu_exact_f(z, up);
      }
      o[v] = f2bf(z);
    }
    bf16* dst = Y + (size_t)row * ncols + c;
    if (c + 4 <= ncols && ncols % 4 == 0) {
      *reinterpret_cast<bf16x4*>(dst) = o;
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (c + v < ncols) dst[v] = o[v];
    }
  }
}

// Groups of 8 weight rows per workgroup up to 16 rows of x: the fewest rows (weights and x) that a CU has to stage.  A CU
// keeps some 64 cache lines in flight whatever the number of its waves, so the time is that of the CU with the most rows:
// ceil(workgroups / 256) (RG + XG).  Where a weight row is a multiple of 4 KiB the lines of 32 and, more so, 64 rows that walk
// K in step fall on few memory channels: their rows count 1.24 and 1.6 times.  us, M = 1 / 16, 16-row tiles (32 from 256 tiles
// on) -> this: 1024 x 3072 4.8 / 6.1 -> 4.4 / 5.3, 2048 x 2048 4.5 / 5.1 -> 4.1 / 4.6, 2048 x 8192 10.5 / 12.0 -> 8.3 / 9.5,
// 5120 x 2560 8.0 / 8.2 -> 7.0 / 7.5, 6144 x 4096 13.0 / 13.8 -> 10.3 / 10.1; GLU 8192 x 2048 9.0 / 9.3 -> 8.0 / 9.3, 10240 x
// 2560 11.7 / 12.7 -> 10.9 / 11.3, 16384 x 4096 28.3 / 28.1 -> 23.6 / 25.6, 22016 x 4096 39.9 / 39.6 -> 30.0 / 29.7.
static int stream_rows(int ncols, int K, bool glu, int xg) {
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

// glu 0: y [M, N] = x w^T (+ bias);  1 / 2 / 3: y [M, N / 2], SiLU / clipped / gelu GLU of w = [gate; up] (+ bias).
// nt: nontemporal weight loads.
void gemm_stream(uintptr_t y, uintptr_t x, uintptr_t w, uintptr_t bias, int M, int N, int K, int glu, int nt, float limit,
                 uintptr_t stream) {
  DLLM_HOST_CHECK(M >= 1 && M <= 64, "1 <= M <= 64");
  DLLM_HOST_CHECK(K >= SK && K % SK == 0, "K must be a positive multiple of 64");
  DLLM_HOST_CHECK(glu >= 0 && glu <= 3, "glu 0..3");
  DLLM_HOST_CHECK(N >= 1 && (glu == 0 || N % 2 == 0), "N");
  DLLM_HOST_CHECK(x % 16 == 0 && w % 16 == 0 && y % 8 == 0, "operand alignment");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int ncols = glu ? N / 2 : N;
  const bool one = M <= 16;
  const int xg = M <= 8 ? 1 : M <= 16 ? 2 : M <= 32 ? 4 : 8;
  int rg;
  if (one) {
    rg = stream_rows(ncols, K, glu != 0, xg);
  } else {
    // twice the weight rows per workgroup (half the x staging) once that still leaves a workgroup for most CUs
    const bool two = (ncols + 15) / 16 > 256;
    rg = (glu ? 4 : 2) * (two ? 2 : 1);
  }
  const int per = glu ? rg * 4 : rg * 8;
  const dim3 grid((ncols + per - 1) / per);
  // 8 waves where up to three groups of plain rows have a CU each: their K loop is over in one or two rounds; else 4
  // (several workgroups per CU)
  const bool wide = glu == 0 && (one ? rg <= 3 && grid.x <= 256 : rg == 2 && xg == 4);
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
#undef DLLM_ST_P
#undef DLLM_ST_GO
  DLLM_HIP_CHECK(hipGetLastError());
}

}  // namespace dllm
