// The body of the weight-streaming GEMM (gemm_stream.hip; with the close of a sublayer in front of it gemm_close.hip).
#pragma once
#include "common.h"

namespace dllm {

namespace {
typedef __attribute__((address_space(3))) void* lds_vptr_s;
typedef __attribute__((address_space(1))) void* glb_vptr_s;
constexpr int SK = 64;                    // K-tile
constexpr int D = 2;                      // slots of a wave's ring

__device__ __forceinline__ int sswz(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }

// What the close of a sublayer reads and writes (gemm_close.hip): one row
struct CloseArgs {
  const float* x;                         // float32 stream [K]
  const bf16* o;                          // the sublayer's output [K]
  const bf16 *ob, *wp, *bp, *wn, *bn;     // its bias (or null), the norm of the output, the norm behind the sum
  float* xo;                              // the new stream [K]
  float eps, mult, offset;
};
enum { kNoClose = 0, kRmsClose = 1, kLayerClose = 2 };
constexpr int CV = 4;                     // waves of a close

// The row of a close in CV waves, PV pieces of 4 elements per lane (places past K repeat the last ones).  Everything is loaded
// in its stored form before the first use.  `wv`: among the close's waves.  These take no part in the product: a wave that had
// weights under way as well would wait for those with its row (hipcc counts no further than to zero behind LDS-DMA).
template <int CLOSE, int PV>
struct CloseRow {
  static constexpr bool kLayer = CLOSE == kLayerClose;
  static constexpr int kBarriers = kLayer ? 4 : 2;             // of finish()
  f32x4 rx[PV];
  bf16x4 ro[PV], wp[PV], ob[PV], wn[PV], bp[kLayer ? PV : 1], bn[kLayer ? PV : 1];

  static __device__ __forceinline__ int place(int k, int wv, int lane) { return ((k * CV + wv) * 64 + lane) * 4; }

  __device__ __forceinline__ void load(const CloseArgs& c, int K, int wv, int lane) {
    const bf16* bias = c.ob ? c.ob : c.wp;                     // (off a place that is there; not used without a bias)
#pragma unroll
    for (int k = 0; k < PV; ++k) {
      const int at = min(place(k, wv, lane), K - 4);
      const auto vec = [&](const bf16* p) { return *reinterpret_cast<const bf16x4*>(p + at); };
      rx[k] = *reinterpret_cast<const f32x4*>(c.x + at);
      ro[k] = vec(c.o), wp[k] = vec(c.wp), ob[k] = vec(bias), wn[k] = vec(c.wn);
      if constexpr (kLayer) bp[k] = vec(c.bp), bn[k] = vec(c.bn);
    }
  }

  // Sum (SQ: centred sum of squares) of the row, places past K left out, in the order of the launch of its own (seqmix.hip:
  // the same four waves, the same places, wave 0 first); `red`: CV floats of LDS, other ones every time.
  template <bool SQ>
  static __device__ __forceinline__ float sum(const float (&v)[PV][4], float mean, int K, int wv, int lane, float* red) {
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < PV; ++k) {
      if (place(k, wv, lane) < K) {
#pragma unroll
        for (int j = 0; j < 4; ++j) s += SQ ? (v[k][j] - mean) * (v[k][j] - mean) : v[k][j];
      }
    }
    s = wave_sum(s);
    if (lane == 0) red[wv] = s;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");                             // (the barrier by itself keeps no load behind it)
    const f32x4 r = *reinterpret_cast<const f32x4*>(red);
    return ((r[0] + r[1]) + r[2]) + r[3];
  }

  // The normed row into `h`; the new stream to memory from one workgroup.  `red`: 4 CV floats.
  __device__ __forceinline__ void finish(const CloseArgs& c, bf16* h, float* red, int K, int wv, int lane) {
    float v[PV][4];
#pragma unroll
    for (int k = 0; k < PV; ++k)
#pragma unroll
      for (int j = 0; j < 4; ++j) v[k][j] = bf2f(ro[k][j]) + (c.ob ? bf2f(ob[k][j]) : 0.f);
    float mean = kLayer ? sum<false>(v, 0.f, K, wv, lane, red) / (float)K : 0.f;
    float inv = 1.0f / sqrtf(sum<true>(v, mean, K, wv, lane, red + CV) / (float)K + c.eps);
#pragma unroll
    for (int k = 0; k < PV; ++k) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float w = bf2f(wp[k][j]);
        if constexpr (kLayer) v[k][j] = rx[k][j] + ((v[k][j] - mean) * inv * w + bf2f(bp[k][j]));
        else v[k][j] = rx[k][j] + c.mult * (v[k][j] * inv * (c.offset + w));
      }
      if (blockIdx.x == 0 && place(k, wv, lane) < K)
        *reinterpret_cast<f32x4*>(c.xo + place(k, wv, lane)) = f32x4{v[k][0], v[k][1], v[k][2], v[k][3]};
    }
    mean = kLayer ? sum<false>(v, 0.f, K, wv, lane, red + 2 * CV) / (float)K : 0.f;
    inv = 1.0f / sqrtf(sum<true>(v, mean, K, wv, lane, red + 3 * CV) / (float)K + c.eps);
#pragma unroll
    for (int k = 0; k < PV; ++k) {
      const int at = place(k, wv, lane);
      bf16x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float w = bf2f(wn[k][j]);
        if constexpr (kLayer) o[j] = f2bf((v[k][j] - mean) * inv * w + bf2f(bn[k][j]));
        else o[j] = f2bf(v[k][j] * inv * (c.offset + w));
      }
      if (at < K) *reinterpret_cast<bf16x4*>(h + at) = o;
    }
  }
};
}  // namespace

// GLU 0: y [M, N] (+ bias [N]);  1 / 2 / 3: SiLU / clipped (`limit`) / gelu GLU, w = [gate; up], y [M, N / 2], bias
// gate | up;  4: y [M, N] in float32, soft-capped by `limit` where that is positive (logits).  A workgroup's RG groups of
// 8 weight rows are its output columns, under a GLU CW gate rows and then the same columns' up rows; XG groups of 8 rows of
// x.  An odd last group fills half an MFMA tile, its other half repeats it.
// CLOSE (M == 1): x is not read but made (CloseRow, K <= KMAX) by CV further waves, and stays in LDS.
template <int RG, int XG, int GLU, bool NT, int WAVES, int CLOSE, int KMAX>
__device__ __forceinline__ void gemm_stream_body(bf16* __restrict__ Y, const bf16* __restrict__ X, const bf16* __restrict__ W,
                                                 const bf16* __restrict__ bias, int M, int N, int K, float limit,
                                                 const CloseArgs& close) {
  constexpr bool PAIR = GLU >= 1 && GLU <= 3, CAPPED = GLU == 4;
  static_assert(!PAIR || RG % 2 == 0 || RG == 3, "a GLU's CW is a multiple of 4");
  constexpr int RT = (RG + 1) / 2, MT = (XG + 1) / 2;
  constexpr int G = CLOSE ? RG : RG + XG;                       // loads per K-tile
  constexpr int SLOT = G * 8 * SK;                              // bf16 elements of one ring slot: weights, then x
  constexpr int RING = WAVES * D * SLOT * 2, RED = WAVES * RT * MT * 1024;
  constexpr int TH = (WAVES + (CLOSE ? CV : 0)) * 64;
  static_assert(G <= 63, "vmcnt");
  __shared__ __attribute__((aligned(16))) char smem[RING > RED ? RING : RED];
  __shared__ __attribute__((aligned(16))) float close_red[CLOSE ? 4 * CV : 4];
  __shared__ __attribute__((aligned(16))) bf16 made[CLOSE ? KMAX : 8];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fq = lane >> 4;
  const int half = N / 2, ncols = PAIR ? half : N;
  constexpr int CW = PAIR ? RG * 4 : RG * 8;                    // output columns
  const int c0 = blockIdx.x * CW;
  bf16* ring = reinterpret_cast<bf16*>(smem) + wv * (D * SLOT);

  // weight row of row r of the workgroup; rows past the matrix repeat its last row
  auto wrow = [&](int r) {
    const bool up = PAIR && r >= CW;
    return (up ? half : 0) + min(c0 + (up ? r - CW : r), ncols - 1);
  };
  typedef CloseRow<CLOSE, CLOSE ? (KMAX + 256 * CV - 1) / (256 * CV) : 1> Row;
  Row row_;
  if (CLOSE != kNoClose && wv >= WAVES) row_.load(close, K, wv - WAVES, lane);
  // The bias of the epilogue: of the GLU that has one in its models, loaded here, so that no round trip is left for the end, off
  // a place that is there and in its stored form, since a load behind a branch or next to its conversion is waited for at
  // once.  (The others load theirs behind one branch: loads that nobody needs cost 0.1 us.)  us, behind a `bias ?` of its own
  // for each of a thread's eight loads -> this, M = 1 / 16: 6144 x 1024 + clipped GLU 5.18 / 5.55 -> 4.79 / 5.18, 15360 x 2560
  // 16.5 / 15.9 -> 16.2 / 15.6; 2560 x 2560 plain 4.96 / 6.15 -> 4.80 / 5.92.
  constexpr int EL = CW / 4 * MT * 16, NE = (EL + TH - 1) / TH;
  bf16 eb[NE][PAIR ? 8 : 4] = {};
  auto load_bias = [&](const bf16* bs, int n) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int cc = min(c0 + 4 * (((tid + n * TH) >> 4) % (CW / 4)) + v, ncols - 1);
      eb[n][v] = bs[bias ? cc : 0];
      if constexpr (PAIR) eb[n][4 + v] = bs[bias ? half + cc : 0];
    }
  };
  if constexpr (GLU == 2) {
#pragma unroll
    for (int n = 0; n < NE; ++n) load_bias(bias ? bias : CLOSE ? W : X, n);
    __builtin_amdgcn_sched_barrier(0);
  }
  const bf16* src[G];
#pragma unroll
  for (int q = 0; q < G; ++q) {
    const int r = 8 * (q < RG ? q : q - RG) + (lane >> 3);
    const bf16* row = q < RG ? W + (size_t)wrow(r) * K : X + (size_t)min(r, M - 1) * K;
    src[q] = row + wv * SK + sswz(r, lane & 7) * 8;
  }
  // this wave's K-tiles (0 for a short K)
  const int nk = K / SK, cnt = CLOSE != kNoClose && wv >= WAVES ? 0 : (nk - wv + WAVES - 1) / WAVES;
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
  if constexpr (CLOSE != kNoClose) {
    // The weights' requests behind the row's: a CU has some 256 lines under way, in their order, so that without this barrier the row came
    // behind the first weights (gemm_close.hip has the figures).  It waits for nothing but that the loads are issued.
    issue_barrier();
  }
#pragma unroll
  for (int u = 0; u < D; ++u)
    if (u < cnt) load(u, u);
  if constexpr (CLOSE != kNoClose) {
    if (wv >= WAVES) {
      row_.finish(close, made, close_red, K, wv - WAVES, lane);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    } else {
#pragma unroll
      for (int b = 0; b < Row::kBarriers; ++b) __builtin_amdgcn_s_barrier();
    }
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
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
            if constexpr (CLOSE != kNoClose) {
              xa[m][s] = *reinterpret_cast<const bf16x8*>(made + (i * WAVES + wv) * SK + (4 * s + fq) * 8);
            } else {
              xa[m][s] = *reinterpret_cast<const bf16x8*>(b + RG * 512 + m * 1024 + r * SK + sswz(r, 4 * s + fq) * 8);
            }
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
  if (CLOSE == kNoClose || wv < WAVES) {
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) red[(wv * RT * MT + t * MT + m) * 64 + lane] = acc[t][m];
  }
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
    if constexpr (PAIR) {
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
      if constexpr (PAIR) {
        const float up = b[v] + (bias ? bf2f(eb[n][4 + v]) : 0.f);
        // (a projection, a bias and a gate kernel until they met here: the gate kernels' arithmetic)
        z = GLU == 1 ? silu_f(z) * up : GLU == 2 ? clipped_glu_exact_f(z, up, limit, kGluAlpha) : gelu_glu_exact_f(z, up);
      }
      o[v] = f2bf(z);
    }
    if constexpr (CAPPED) {                          // logits: of the product's bf16, as a launch of their own made them
      f32x4 l;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float z = bf2f(o[v]);
        l[v] = limit > 0.f ? limit * tanhf(z / limit) : z;
      }
      float* dst = reinterpret_cast<float*>(Y) + (size_t)row * ncols + c;
      if (c + 4 <= ncols && ncols % 4 == 0) {
        *reinterpret_cast<f32x4*>(dst) = l;
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (c + v < ncols) dst[v] = l[v];
      }
      continue;
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

}  // namespace dllm
