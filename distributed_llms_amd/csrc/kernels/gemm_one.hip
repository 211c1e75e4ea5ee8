// One decode row's products off large weights: C[1, N] = x . B[N, K]^T, bf16 in, f32 accumulate, with the add and RMS norm in front of
// them where x is a normed sum.  N a multiple of 128, K of 64; a K split leaves slabs (common.h), as gemm_wide does.
//
// What bounds it: the weights (6.1-6.6 TB/s of 235 MiB, 5 of 48 MiB), and for a decode layer, a chain of launches of 4 to 40 us, that
// every launch pays 2-3 us to start, to get its first weights and to drain.  So
//  * the norm has no launch of its own: every workgroup makes the row it multiplies (K times slabs + 2 values, 72 KiB for 4096 in 8
//    slabs, out of its XCD's L2) in four waves of its own while eight others have the first weights under way.  (Loads return in
//    order: a wave that has both under way would wait for its weights with its row.)  The weights wait until the row's loads are issued (a
//    barrier): a CU has some 256 lines under way, in their order.  us, add + norm and product / in one launch, weights at once / as it is:
//    6144 x 4096 12.8 / 10.4 / 10.0, 28672 x 4096 with its SwiGLU 42.4 / 38.3 / 36.5, 10240 x 8192 34.0 / 33.0 / 32.6, 57344 x 8192 152 / 150 / 149, 3072 x
//    2048 9.0 / 6.6 / 6.0;
//  * the row is whole in LDS and each wave streams 16 weight rows through a ring of its own: no staging of x, no barriers.  us,
//    gemm_wide / this: 4096 x 14336 20.0 / 19.2, 4096 x 4096 7.6 / 7.1, 8192 x 8192 31.3 / 27.2, 128256 x 4096 160 / 155;
//  * the ring: D K-tiles of 64.  3 are enough for slices under 32 K-tiles (4096 x 14336 in 8 of 28: 19.2, with 5 19.6); longer ones
//    gain by 5 (8192 x 8192 in 4 of 32 29.0 -> 27.2, 128256 x 4096 164 -> 155);
//  * BAR, a GLU's gate and up rows: a barrier per K-tile.  Waves that drift apart land on a part of the memory channels (28672 x 4096:
//    38.5 with 3 K-tiles and 43-44 with 4 or 5 without it, 36.5 with it; 57344 x 8192 147 / 148).
// The sums have gemm_wide's order (a K-tile's halves one after the other, unsplit ones from a K-tile that hangs on the XCD) and the
// norm that of splitk_add_rms_norm / rms_norm: equal bits.
#include "gemm_pp_common.h"
#include "launchers.h"

namespace dllm {

namespace {
constexpr int OF = 4, OW = 8;             // waves: of the row, of the product (16 weight rows each)
constexpr int OFT = OF * 64;
constexpr int kOneSlabs = 8;              // most slabs of what is added
enum { kRowAsIs = 0, kRowNorm = 1, kRowAddNorm = 2, kRowSlabsNorm = 3 };

struct OneRow {
  const bf16* x;                          // kRowAsIs: the row;  kRowAddNorm: what is added to the stream
  const bf16* res;                        // the stream
  const float* part;                      // kRowSlabsNorm: `slabs` slabs of what is added
  const bf16* w;                          // norm weights
  bf16* res_out;                          // the new stream
  int slabs;
  float eps;
};

__device__ __forceinline__ void one_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
}  // namespace

// The row (kRowAsIs: nt K-tiles of it) to LDS, in OF waves of MAXV pieces of 8 elements per lane.  `first`: of the workgroups, the
// one that writes the new stream.  Past the last place the last one again, dropped.  Two barriers (kRowAsIs: one).
template <int IN, int MAXV>
__device__ __forceinline__ void one_row(const OneRow& in, int K, int ks0, int nt, bool first, char* rows, float* red, int wv, int lane) {
  const int nvec = IN == kRowAsIs ? nt * (PBK / 8) : K >> 3;
  auto place = [&](int i) { return (int)threadIdx.x + i * OFT; };
  if constexpr (IN == kRowAsIs) {
    bf16x8 v[MAXV];
#pragma unroll
    for (int i = 0; i < MAXV; ++i) v[i] = reinterpret_cast<const bf16x8*>(in.x + ks0 * PBK)[min(place(i), nvec - 1)];
#pragma unroll
    for (int i = 0; i < MAXV; ++i)
      if (place(i) < nvec) *reinterpret_cast<bf16x8*>(rows + place(i) * 16) = v[i];
    one_barrier();
    return;
  } else {
    typedef part_elem raw __attribute__((ext_vector_type(8)));
    constexpr int CH = IN == kRowSlabsNorm ? 2 : MAXV;   // pieces whose loads are under way together
    bf16x8 g[MAXV], r[MAXV];
    float ss = 0.f;
#pragma unroll
    for (int c0 = 0; c0 < MAXV; c0 += CH) {
      raw l[IN == kRowSlabsNorm ? CH : 1][kOneSlabs];
      bf16x8 h[IN == kRowAddNorm ? CH : 1];
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const int at = min(place(c0 + i), nvec - 1);
        if constexpr (IN == kRowSlabsNorm) {
#pragma unroll
          for (int s = 0; s < kOneSlabs; ++s)            // (past the last slab: that again)
            l[i][s] = *reinterpret_cast<const raw*>(reinterpret_cast<const part_elem*>(in.part) + (size_t)min(s, in.slabs - 1) * K + at * 8);
        }
        if constexpr (IN == kRowAddNorm) h[i] = reinterpret_cast<const bf16x8*>(in.x)[at];
        r[c0 + i] = reinterpret_cast<const bf16x8*>(in.res)[at];
      }
      if (c0 == 0) {
#pragma unroll
        for (int i = 0; i < MAXV; ++i) g[i] = reinterpret_cast<const bf16x8*>(in.w)[min(place(i), nvec - 1)];
      }
      __builtin_amdgcn_sched_barrier(0);
      if (c0 == 0) __builtin_amdgcn_s_barrier();         // the row's requests are out: now the weights'
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        bf16x8& v = r[c0 + i];
        if constexpr (IN != kRowNorm) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            float a = 0.f;
            if constexpr (IN == kRowSlabsNorm) {
#pragma unroll
              for (int s = 0; s < kOneSlabs; ++s) a = s < in.slabs ? a + part_value(l[i][s][j]) : a;
              a = bf2f(f2bf(a));
            } else {
              a = bf2f(h[i][j]);
            }
            v[j] = f2bf(a + bf2f(v[j]));
          }
        }
        if (place(c0 + i) < nvec) {
          if (IN != kRowNorm && first) reinterpret_cast<bf16x8*>(in.res_out)[place(c0 + i)] = v;
#pragma unroll
          for (int j = 0; j < 8; ++j) ss += bf2f(v[j]) * bf2f(v[j]);
        }
      }
    }
    ss = wave_sum(ss);
    if (lane == 0) red[wv] = ss;
    one_barrier();
    ss = 0.f;
#pragma unroll
    for (int i = 0; i < OF; ++i) ss += red[i];
    const float inv = rsqrtf(ss / (float)K + in.eps);
#pragma unroll
    for (int i = 0; i < MAXV; ++i) {
      bf16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = f2bf(bf2f(r[i][j]) * inv * bf2f(g[i][j]));
      if (place(i) < nvec) *reinterpret_cast<bf16x8*>(rows + place(i) * 16) = o;
    }
    one_barrier();
  }
}

// MODE 0: C bf16 [N];  1: slab of P [S, N];  2: SwiGLU C [N / 2], B = [gate; up].  A GLU's 16 rows of a wave are 8 gate and 8 up rows in
// pairs, so that a lane's four sums (rows 4 q .. 4 q + 3) are two columns' gates and ups.
template <int MODE, int IN, int MAXV, int D, bool NT>
__global__ void __launch_bounds__((OF + OW) * 64, 1) gemm_one_kernel(const bf16* __restrict__ B, OneRow in, int N, int K, int kts,
                                                                     int nsplit, bf16* __restrict__ C, float* __restrict__ P) {
  constexpr bool GLU = MODE == 2, BAR = GLU;
  __shared__ __attribute__((aligned(16))) char smem[OW * D * 2048 + MAXV * OFT * 16];
  __shared__ float red[OF];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int b = blockIdx.x;
  {   // consecutive slices and column tiles on one XCD (gemm_wide's order)
    const int q = gridDim.x >> 3, r = gridDim.x & 7, x = b & 7;
    b = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + (b >> 3);
  }
  const int split = b % nsplit, n_t = b / nsplit;
  const int ks0 = split * kts, nt = min(K / PBK, ks0 + kts) - ks0;       // >= 1 (host)
  const int rot = nsplit == 1 && nt >= 16 ? ((int)(blockIdx.x & 7) * nt) >> 3 : 0;
  char* rows = smem + OW * D * 2048;
  if (wv < OF) {
    one_row<IN, MAXV>(in, K, ks0, nt, b == 0, rows, red, wv, lane);
    if constexpr (BAR) {
      for (int t = 0; t < nt; ++t) __builtin_amdgcn_s_barrier();
    }
    return;
  }
  const int pw = wv - OF;
  char* ring = smem + pw * (D * 2048);
  uint32_t offB[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int i = 8 * j + (lane >> 3);                   // of the wave's 16
    const int row = GLU ? ((i >> 1) & 1 ? N / 2 : 0) + n_t * 64 + pw * 8 + 2 * (i >> 2) + (i & 1) : n_t * 128 + pw * 16 + i;
    offB[j] = (uint32_t)row * (uint32_t)(K * 2) + (uint32_t)(pswz(i, lane & 7) * 16);
  }
  const auto rb = __builtin_amdgcn_make_buffer_rsrc((void*)(reinterpret_cast<const char*>(B) + (size_t)ks0 * 128), (short)0,
                                                    (int)(unsigned)((long)N * K * 2 - (long)ks0 * 128), 0x00020000);
  auto k_of = [&](int t) { return t + rot >= nt ? t + rot - nt : t + rot; };
  auto stage = [&](int slot, int t) {                    // (past the last K-tile: that again)
    const int k = k_of(min(t, nt - 1));
#pragma unroll
    for (int j = 0; j < 2; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_vptr_p)(ring + slot * 2048 + j * 1024), 16, (int)offB[j], k * 128, 0, NT ? 2 : 0);
  };
  if constexpr (IN != kRowAsIs) __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < D; ++j) stage(j, j);
  const uint32_t lds0 = (uint32_t)(size_t)(lds_vptr_p)smem;
  const int fr = lane & 15, fq = lane >> 4;
  const uint32_t at_b = lds0 + pw * (D * 2048) + fr * 128, at_a = lds0 + OW * D * 2048 + (IN == kRowAsIs ? 0 : ks0 * 128) + fq * 16;
  const uint32_t bo0 = pswz(fr, fq) * 16, bo1 = pswz(fr, 4 + fq) * 16;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  if constexpr (IN != kRowAsIs) __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  int slot = 0;
  for (int t = 0; t < nt; ++t) {
    // the younger K-tiles in flight: D - 1, as long as there are that many
    if (t + D <= nt) pp_vm<2 * (D - 1)>();
    else pp_vm<0>();
    if constexpr (BAR) __builtin_amdgcn_s_barrier();
    bf16x8 b0, b1, a0, a1;
    const uint32_t pb = at_b + slot * 2048, pa = at_a + k_of(t) * 128;   // (a: the same for all 16 rows of an operand)
    asm volatile("ds_read_b128 %0, %1" : "=v"(b0) : "v"(pb + bo0));
    asm volatile("ds_read_b128 %0, %1" : "=v"(b1) : "v"(pb + bo1));
    asm volatile("ds_read_b128 %0, %1" : "=v"(a0) : "v"(pa));
    asm volatile("ds_read_b128 %0, %1 offset:64" : "=v"(a1) : "v"(pa));
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(b0), "+v"(b1), "+v"(a0), "+v"(a1)::"memory");
    if (t + D < nt) stage(slot, t + D);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b0, a0, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b1, a1, acc, 0, 0, 0);
    slot = slot == D - 1 ? 0 : slot + 1;
  }
  pp_vm<0>();                                            // (slices under D K-tiles: pieces that nobody waited for)
  if (fr == 0) {
    if constexpr (GLU) {
      const bf16x2 h = {f2bf(silu_f(acc[0]) * acc[2]), f2bf(silu_f(acc[1]) * acc[3])};
      *reinterpret_cast<bf16x2*>(C + n_t * 64 + pw * 8 + 2 * fq) = h;
    } else if constexpr (MODE == 0) {
      bf16x4 h;
#pragma unroll
      for (int v = 0; v < 4; ++v) h[v] = f2bf(acc[v]);
      *reinterpret_cast<bf16x4*>(C + n_t * 128 + pw * 16 + 4 * fq) = h;
    } else {
      part_store4(P, (size_t)split * N + n_t * 128 + pw * 16 + 4 * fq, acc);
    }
  }
}

// mode 0: c [n] = x b^T;  1: SwiGLU c [n / 2], b = [gate; up];  2: slabs [S, n] of `splits` K slices (S > 1, or 1: c), x a row (w = 0) or the norm of weights w
// of stream res [k] + what is added to it: nothing, x, or `nslabs` slabs at part.  res_out: the sum (not res itself: others still read it).
// Returns the number of slices S.
int gemm_one(uintptr_t c, uintptr_t slabs, uintptr_t b, int n, int k, int splits, int mode, int nt, uintptr_t x, uintptr_t res,
             uintptr_t part, int nslabs, uintptr_t w, uintptr_t res_out, float eps, uintptr_t stream) {
  DLLM_HOST_CHECK(n > 0 && n % 128 == 0 && k > 0 && k % PBK == 0 && (long)n * k * 2 < (1L << 32), "N a multiple of 128, K of 64, under 4 GiB");
  DLLM_HOST_CHECK(mode >= 0 && mode <= 2 && splits >= 1 && (mode == 2 || splits == 1), "a K split leaves slabs");
  const int kind = w == 0 ? kRowAsIs : part ? kRowSlabsNorm : x ? kRowAddNorm : kRowNorm;
  const int kts = (k / PBK + splits - 1) / splits, S = (k / PBK + kts - 1) / kts;
  if (mode == 2 && S == 1) mode = 0;
  DLLM_HOST_CHECK(mode == 2 ? slabs != 0 : c != 0, "output");
  DLLM_HOST_CHECK(kind != kRowAsIs || x, "a row");
  DLLM_HOST_CHECK(kind == kRowAsIs || res, "a stream");
  DLLM_HOST_CHECK(kind < kRowAddNorm || (res_out && res_out != res), "the new stream apart from the old one");
  DLLM_HOST_CHECK(kind != kRowSlabsNorm || (nslabs >= 1 && nslabs <= kOneSlabs), "up to 8 slabs");
  DLLM_HOST_CHECK((x | res | part | w | res_out | b) % 16 == 0 && (c | slabs) % 8 == 0, "alignment");
  const int width = kind == kRowAsIs ? kts * PBK : k;
  DLLM_HOST_CHECK(width <= 4 * OFT * 8, "rows of up to 8192");
  DLLM_HOST_CHECK(mode != 0 || kind == kRowAsIs, "a norm in front of slabs or a GLU");
  const long grid = (long)(n / 128) * S;
  DLLM_HOST_CHECK(grid < (1L << 31), "grid");
  const OneRow in{(const bf16*)x, (const bf16*)res, (const float*)part, (const bf16*)w, (bf16*)res_out, nslabs, eps};
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3((OF + OW) * 64), 0, reinterpret_cast<hipStream_t>(stream), (const bf16*)b, in,
                       n, k, kts, S, (bf16*)c, (float*)slabs);
  };
#define DLLM_ONE_V(MODE_, IN_, D_, NT_)                                          \
  do {                                                                           \
    if (width <= 2 * OFT * 8) go(gemm_one_kernel<MODE_, IN_, 2, D_, NT_>);       \
    else go(gemm_one_kernel<MODE_, IN_, 4, D_, NT_>);                            \
  } while (0)
#define DLLM_ONE_SLABS(IN_)                                                      \
  do {                                                                           \
    if (!nt) DLLM_ONE_V(1, IN_, 3, false);                                       \
    else if (kts < 32) DLLM_ONE_V(1, IN_, 3, true);                              \
    else DLLM_ONE_V(1, IN_, 5, true);                                            \
  } while (0)
  if (mode == 0) {
    if (nt) DLLM_ONE_V(0, kRowAsIs, 5, true);
    else DLLM_ONE_V(0, kRowAsIs, 5, false);
  } else if (mode == 1) {
    if (kind == kRowAsIs) DLLM_ONE_V(2, kRowAsIs, 3, true);
    else if (kind == kRowNorm) DLLM_ONE_V(2, kRowNorm, 3, true);
    else if (kind == kRowAddNorm) DLLM_ONE_V(2, kRowAddNorm, 3, true);
    else DLLM_ONE_V(2, kRowSlabsNorm, 3, true);
  } else {
    if (kind == kRowAsIs) DLLM_ONE_SLABS(kRowAsIs);
    else if (kind == kRowNorm) DLLM_ONE_SLABS(kRowNorm);
    else if (kind == kRowAddNorm) DLLM_ONE_SLABS(kRowAddNorm);
    else DLLM_ONE_SLABS(kRowSlabsNorm);
  }
#undef DLLM_ONE_SLABS
#undef DLLM_ONE_V
  DLLM_HIP_CHECK(hipGetLastError());
  return S;
}

}  // namespace dllm
