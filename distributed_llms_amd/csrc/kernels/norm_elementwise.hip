// Memory-bound per-token kernels (K1, K2, K4/K5, SwiGLU activation, argmax).
//
// All of these move bf16 through 16-byte (bf16x8) vectors: hipcc does not
// vectorize bf16 scalar loads (CDNA guide Guideline 13) and scalar bf16 costs
// ~2x on HBM-bound kernels.
#include "common.h"
#include "launchers.h"

namespace dllm {

// ---------------------------------------------------------------------------
// K2: RMSNorm, optionally fused with the residual add.
//   residual == nullptr : y = rmsnorm(x) * w
//   residual != nullptr : r = x + residual; residual <- r; y = rmsnorm(r) * w
// One 256-thread workgroup per row; the row stays in registers between the
// sum-of-squares pass and the scale pass (MAXV vectors of 8 per thread).
// ---------------------------------------------------------------------------
template <int MAXV>
__global__ void __launch_bounds__(256) rms_norm_kernel(bf16* __restrict__ y, const bf16* __restrict__ x,
                                                       bf16* __restrict__ residual,
                                                       const bf16* __restrict__ w, int hidden,
                                                       float eps, uint8_t* __restrict__ q8, float* __restrict__ qs) {
  __shared__ float red[16];
  const int row = blockIdx.x;
  const int nvec = hidden >> 3;
  const bf16x8* xr = reinterpret_cast<const bf16x8*>(x + (size_t)row * hidden);
  bf16x8* rr = residual ? reinterpret_cast<bf16x8*>(residual + (size_t)row * hidden) : nullptr;
  const bf16x8* wv = reinterpret_cast<const bf16x8*>(w);
  float v[MAXV][8];
  bf16x8 a[MAXV], b[MAXV], g[MAXV];
  float ss = 0.f;
  // every load off a clamped place and before the first use (behind the guards hipcc waited for each vector in turn, and
  // for the weight behind the block's sum)
  const bf16x8* rb = rr ? rr : xr;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int idx = min((int)threadIdx.x + i * 256, nvec - 1);
    a[i] = xr[idx];
    b[i] = rb[idx];
    g[i] = wv[idx];
  }
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int idx = threadIdx.x + i * 256;
    if (rr) {
#pragma unroll
      for (int j = 0; j < 8; ++j) a[i][j] = f2bf(bf2f(a[i][j]) + bf2f(b[i][j]));
    }
    if (idx < nvec) {
      if (rr) rr[idx] = a[i];   // normalise the bf16-rounded residual, as the reference does
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[i][j] = bf2f(a[i][j]);
        ss += v[i][j] * v[i][j];
      }
    }
  }
  ss = block_sum<256>(ss, red);
  const float inv = rsqrtf(ss / (float)hidden + eps);
  if (q8) {   // FP8 consumer (W8A8 GEMM): per-token e4m3 of the bf16-rounded output, y optional
    norm_out_fp8<MAXV, 256>(v, inv, g, nvec, y ? y + (size_t)row * hidden : nullptr, q8 + (size_t)row * hidden,
                            qs + row, red);
    return;
  }
  bf16x8* yr = reinterpret_cast<bf16x8*>(y + (size_t)row * hidden);
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int idx = threadIdx.x + i * 256;
    if (idx < nvec) {
      bf16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = f2bf(v[i][j] * inv * bf2f(g[i][j]));
      yr[idx] = o;
    }
  }
}

void rms_norm(uintptr_t y, uintptr_t x, uintptr_t residual, uintptr_t w, int rows, int hidden,
              float eps, uintptr_t stream) {
  rms_norm_q8(y, x, residual, w, rows, hidden, eps, 0, 0, stream);
}

// q8 != 0: also (y == 0: only) the per-token e4m3 quantization of the output, scales in qs
void rms_norm_q8(uintptr_t y, uintptr_t x, uintptr_t residual, uintptr_t w, int rows, int hidden, float eps,
                 uintptr_t q8, uintptr_t qs, uintptr_t stream) {
  DLLM_HOST_CHECK(hidden % 8 == 0 && hidden <= 8 * 256 * 8, "hidden must be a multiple of 8 and <= 16384");
  DLLM_HOST_CHECK(rows >= 0, "rows >= 0");
  DLLM_HOST_CHECK(y != 0 || q8 != 0, "rms_norm needs an output");
  DLLM_HOST_CHECK((q8 == 0) == (qs == 0), "q8 and its scales go together");
  if (rows == 0) return;
  const int nvec = hidden / 8;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  auto args = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(rows), dim3(256), 0, s, (bf16*)y, (const bf16*)x, (bf16*)residual,
                       (const bf16*)w, hidden, eps, (uint8_t*)q8, (float*)qs);
  };
  if (nvec <= 256) args(rms_norm_kernel<1>);
  else if (nvec <= 512) args(rms_norm_kernel<2>);
  else if (nvec <= 1024) args(rms_norm_kernel<4>);
  else args(rms_norm_kernel<8>);
  DLLM_HIP_CHECK(hipGetLastError());
}

// ---------------------------------------------------------------------------
// K1: embedding gather. One workgroup per token, 16 B per lane.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) embedding_kernel(bf16* __restrict__ out, const int32_t* __restrict__ ids,
                                                        const bf16* __restrict__ table, int hidden, int vocab) {
  const int t = blockIdx.x;
  int id = ids[t];
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);  // clamp: never read outside the table
  const bf16x8* src = reinterpret_cast<const bf16x8*>(table + (size_t)id * hidden);
  bf16x8* dst = reinterpret_cast<bf16x8*>(out + (size_t)t * hidden);
  for (int i = threadIdx.x; i < (hidden >> 3); i += 256) dst[i] = src[i];
}

void embedding(uintptr_t out, uintptr_t ids, uintptr_t table, int tokens, int hidden, int vocab,
               uintptr_t stream) {
  DLLM_HOST_CHECK(hidden % 8 == 0, "hidden % 8");
  if (tokens == 0) return;
  hipLaunchKernelGGL(embedding_kernel, dim3(tokens), dim3(256), 0, reinterpret_cast<hipStream_t>(stream),
                     (bf16*)out, (const int32_t*)ids, (const bf16*)table, hidden, vocab);
  DLLM_HIP_CHECK(hipGetLastError());
}

// ---------------------------------------------------------------------------
// K4 + K5: RoPE on q/k (rotate-half) fused with the paged KV-cache append.
// qkv [T, (Hq + 2 Hkv) * D] -> q_out [T, Hq, D] (rotated)
// k_cache [NB, Hkv, BS, D]; v_cache [NB, Hkv, D, BS] (transposed V).
// cos_sin [max_pos, D] f32 (first half cos, second half sin); nullptr = no RoPE (GPT-2).
// One workgroup per token; a thread owns 4 rotation pairs (8-byte vectors).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) rope_cache_kernel(bf16* __restrict__ q_out, const bf16* __restrict__ qkv,
                                                         const int32_t* __restrict__ positions,
                                                         const float* __restrict__ cos_sin,
                                                         bf16* __restrict__ k_cache, bf16* __restrict__ v_cache,
                                                         const int32_t* __restrict__ slots, int hq, int hkv,
                                                         int d, int bs) {
  const int t = blockIdx.x;
  const int half = d >> 1;
  const int qpr = half >> 2;  // threads per head (4 pairs each)
  const int pos = positions[t];
  const int slot = slots[t];
  const int blk = slot / bs, off = slot % bs;
  const bf16* row = qkv + (size_t)t * (hq + 2 * hkv) * d;
  const float* cs = cos_sin ? cos_sin + (size_t)pos * d : nullptr;
  // q and k: rotate (q_out null: the attention kernel rotates q itself -- K / V only here)
  const int h0 = q_out ? 0 : hq;
  for (int i = threadIdx.x + h0 * qpr; i < (hq + hkv) * qpr; i += blockDim.x) {
    const int h = i / qpr, p = (i % qpr) * 4;
    const bf16* src = row + h * d;
    bf16x4 x1 = *reinterpret_cast<const bf16x4*>(src + p);
    bf16x4 x2 = *reinterpret_cast<const bf16x4*>(src + half + p);
    bf16x4 o1, o2;
    if (cs) {
      f32x4 c = *reinterpret_cast<const f32x4*>(cs + p);
      f32x4 s = *reinterpret_cast<const f32x4*>(cs + half + p);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float a = bf2f(x1[j]), b = bf2f(x2[j]);
        o1[j] = f2bf(a * c[j] - b * s[j]);
        o2[j] = f2bf(b * c[j] + a * s[j]);
      }
    } else {
      o1 = x1;
      o2 = x2;
    }
    bf16* dst;
    if (h < hq) {
      dst = q_out + ((size_t)t * hq + h) * d;
    } else {
      dst = k_cache + (((size_t)blk * hkv + (h - hq)) * bs + krow(off, bs)) * d;
    }
    *reinterpret_cast<bf16x4*>(dst + p) = o1;
    *reinterpret_cast<bf16x4*>(dst + half + p) = o2;
  }
  // v: transposed store into [blk][h][d][bs]
  const bf16* vsrc = row + (hq + hkv) * d;
  for (int i = threadIdx.x; i < hkv * d; i += blockDim.x) {
    const int h = i / d, e = i % d;
    v_cache[((size_t)blk * hkv + h) * d * bs + vofs(off, e, d, bs)] = vsrc[i];
  }
}

// The same for batches of eight tokens and more, and for a projection still in split-K slabs (any batch): eight tokens and
// up to 1024 columns of q, k or v per workgroup, all of a thread's loads under way before the first use.
//
// V: the transposed layouts keep a key's 8-aligned group of 8 contiguous per (head, e) -- vofs(off0 + j) = vofs(off0) + j
// when off0 % 8 == 0 and bs % 8 == 0 -- so when the group's slots are consecutive and 8-aligned (a prompt's tokens:
// consecutive slots from a block start) a thread writes one 16-byte vector, through an LDS tile, where the per-token
// path scatters eight 2-byte stores (whole 64-byte lines instead of partial ones).  Any other group (a prompt boundary
// inside it, a sequence resuming mid-group, the batch tail) takes the scatter.
//
// Slabs (SC > 0: their number) are summed in slab order and rounded to bf16, as splitk_reduce sums
// them, on the way: a prompt of 128 tokens of 32 / 8 heads took a launch for the sum (3.7 us), one for K (3.3) and one for V
// (4.1); 2 / 3 / 4 / 5 / 8 slabs, sum and append 9.4 / 9.7 / 10.0 / 10.2 / 10.8 us -> 8.4 / 8.8 / 9.3 / 9.5 / 10.1.
// Only the compiled numbers of slabs (rope_cache_append below): a workgroup's eight tokens are one CU's loads, so a
// loop over more of them is slower than the sum's own launch, which spreads over the chip (128 tokens of 32 / 4 heads, 6 / 13 /
// 17 slabs, sum and append 8.9 / 11.8 / 13.1 us; summed here one by one 23.6 / 47 / 61, eight at a time 11.3 / 20 / 25).
// q_out: the rotated q, or (rotate_q 0, slabs only: the attention rotates it) the summed one.
constexpr int kAppendCols = 1024;

template <int SC>
__global__ void __launch_bounds__(256) qkv_append_kernel(bf16* __restrict__ q_out, int rotate_q,
                                                         const bf16* __restrict__ qkv, const float* __restrict__ part,
                                                         long slab, const int32_t* __restrict__ positions,
                                                         const float* __restrict__ cos_sin, bf16* __restrict__ k_cache,
                                                         bf16* __restrict__ v_cache, const int32_t* __restrict__ slots,
                                                         int tokens, int hq, int hkv, int d, int bs, int by_row) {
  __shared__ __attribute__((aligned(16))) bf16 tile[8][kAppendCols + 8];
  __shared__ int sl[8];
  constexpr int R = 4;                                 // four elements or pairs of four per item, R items in flight
  constexpr int NS = SC > 0 ? SC : 1;
  const int width = (hq + 2 * hkv) * d, half = d >> 1;
  const int hpc = max(1, kAppendCols / d);             // heads per workgroup
  const int nkv = (hkv + hpc - 1) / hpc;
  int t0 = blockIdx.x * 8, y = blockIdx.y;
  if (by_row) {
    t0 = blockIdx.y * 8;
    y = (blockIdx.x + (blockIdx.y >> 3)) % gridDim.x;
  }
  const int n = min(8, tokens - t0), tid = threadIdx.x;
  const int what = y < nkv ? 2 : y < 2 * nkv ? 1 : 0;          // v, k, q
  const int h0 = (what == 2 ? y : what == 1 ? y - nkv : y - 2 * nkv) * hpc;
  const int heads = min(hpc, (what == 0 ? hq : hkv) - h0);
  const int col0 = ((what == 0 ? 0 : what == 1 ? hq : hq + hkv) + h0) * d;      // first column in a row of qkv
  // four consecutive values from element p on: in their stored form, and summed
  typedef part_elem raw4 __attribute__((ext_vector_type(4)));
  auto load = [&](raw4 (&l)[NS], bf16x4& v, size_t p) {
    if constexpr (SC == 0) v = *reinterpret_cast<const bf16x4*>(qkv + p);
    if constexpr (SC > 0) {
#pragma unroll
      for (int s = 0; s < NS; ++s)
        l[s] = __builtin_nontemporal_load(reinterpret_cast<const raw4*>(reinterpret_cast<const part_elem*>(part) + p + s * slab));
    }
  };
  auto finish = [&](const raw4 (&l)[NS]) {
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NS; ++s) a += f32x4{part_value(l[s][0]), part_value(l[s][1]), part_value(l[s][2]), part_value(l[s][3])};
    return bf16x4{f2bf(a[0]), f2bf(a[1]), f2bf(a[2]), f2bf(a[3])};
  };
  if (what == 2) {
    const int per = heads * d / 4, total = 8 * per;    // items of a token, of the workgroup
    if (tid < 8) sl[tid] = tid < n ? slots[t0 + tid] : -1;
    for (int i0 = tid; i0 < total; i0 += 256 * R) {
      raw4 l[R][NS];
      bf16x4 v[R];
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const int i = min(i0 + u * 256, total - 1), j = min(i / per, n - 1);
        load(l[u], v[u], (size_t)(t0 + j) * width + col0 + (i % per) * 4);
      }
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const int i = i0 + u * 256;
        if (i >= total) break;
        const int j = i / per;
        if constexpr (SC != 0) v[u] = finish(l[u]);
        *reinterpret_cast<bf16x4*>(&tile[j][(i % per) * 4]) = v[u];
      }
    }
    __syncthreads();
    bool full = n == 8 && bs % 8 == 0 && sl[0] >= 0 && sl[0] % 8 == 0;
#pragma unroll
    for (int j = 1; j < 8; ++j) full = full && sl[j] == sl[0] + j;
    if (full) {
      const int blk = sl[0] / bs, off0 = sl[0] % bs;
      for (int i = tid; i < heads * d; i += 256) {
        const int h = h0 + i / d, e = i % d;
        bf16x8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = tile[j][i];
        *reinterpret_cast<bf16x8*>(v_cache + ((size_t)blk * hkv + h) * d * bs + vofs(off0, e, d, bs)) = o;
      }
      return;
    }
    for (int j = 0; j < n; ++j) {
      const int blk = sl[j] / bs, off = sl[j] % bs;
      for (int i = tid; i < heads * d; i += 256)
        v_cache[((size_t)blk * hkv + h0 + i / d) * d * bs + vofs(off, i % d, d, bs)] = tile[j][i];
    }
    return;
  }
  // q and k: pairs (e, e + d / 2), four of them per item
  const bool rot = cos_sin != nullptr && (what == 1 || rotate_q);
  const int qpr = half >> 2, per = heads * qpr, total = n * per;
  constexpr int RP = 2;
  for (int i0 = tid; i0 < total; i0 += 256 * RP) {
    raw4 l1[RP][NS], l2[RP][NS];
    f32x4 c[RP], s[RP];
    bf16x4 x1[RP], x2[RP];
    int pos[RP], slot[RP];
#pragma unroll
    for (int u = 0; u < RP; ++u) {
      const int i = min(i0 + u * 256, total - 1), t = t0 + i / per;
      pos[u] = positions[t];
      slot[u] = slots[t];
      const size_t p = (size_t)t * width + col0 + (i % per) / qpr * d + (i % qpr) * 4;
      load(l1[u], x1[u], p);
      load(l2[u], x2[u], p + half);
    }
    const float* table = rot ? cos_sin : nullptr;
    if (table) {
#pragma unroll
      for (int u = 0; u < RP; ++u) {
        const float* cs = table + (size_t)pos[u] * d + (min(i0 + u * 256, total - 1) % qpr) * 4;
        c[u] = *reinterpret_cast<const f32x4*>(cs);
        s[u] = *reinterpret_cast<const f32x4*>(cs + half);
      }
    }
#pragma unroll
    for (int u = 0; u < RP; ++u) {
      const int i = i0 + u * 256;
      if (i >= total) break;
      const int t = t0 + i / per, h = h0 + (i % per) / qpr, e = (i % qpr) * 4;
      if constexpr (SC != 0) {
        x1[u] = finish(l1[u]);
        x2[u] = finish(l2[u]);
      }
      bf16x4 o1 = x1[u], o2 = x2[u];
      if (rot) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float a = bf2f(x1[u][j]), b = bf2f(x2[u][j]);
          o1[j] = f2bf(a * c[u][j] - b * s[u][j]);
          o2[j] = f2bf(b * c[u][j] + a * s[u][j]);
        }
      }
      bf16* dst = what == 0 ? q_out + ((size_t)t * hq + h) * d
                            : k_cache + (((size_t)(slot[u] / bs) * hkv + h) * bs + krow(slot[u] % bs, bs)) * d;
      *reinterpret_cast<bf16x4*>(dst + e) = o1;
      *reinterpret_cast<bf16x4*>(dst + half + e) = o2;
    }
  }
}

// part != 0: qkv as nparts split-K slabs, `slab` elements apart (qkv unused); q_out: the rotated q, or the summed one of slabs
// where rotate_q is 0; 0: neither
void rope_cache_append(uintptr_t q_out, int rotate_q, uintptr_t qkv, uintptr_t part, int nparts, long slab,
                       uintptr_t positions, uintptr_t cos_sin, uintptr_t k_cache, uintptr_t v_cache, uintptr_t slots,
                       int tokens, int hq, int hkv, int d, int bs, int v_groups, uintptr_t stream) {
  DLLM_HOST_CHECK(d % 8 == 0 && d <= 256, "head_dim must be a multiple of 8, <= 256");
  DLLM_HOST_CHECK(hq % hkv == 0, "Hq % Hkv");
  DLLM_HOST_CHECK(part == 0 || (nparts >= 1 && slab >= (long)tokens * (hq + 2 * hkv) * d), "qkv partial slabs");
  DLLM_HOST_CHECK(part != 0 || rotate_q || q_out == 0, "an unrotated q is read from qkv itself");
  if (tokens == 0) return;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (part == 0 && !(v_groups && bs % 8 == 0 && tokens >= 8)) {
    hipLaunchKernelGGL(rope_cache_kernel, dim3(tokens), dim3(256), 0, st, (bf16*)q_out, (const bf16*)qkv,
                       (const int32_t*)positions, (const float*)cos_sin, (bf16*)k_cache, (bf16*)v_cache,
                       (const int32_t*)slots, hq, hkv, d, bs);
    DLLM_HIP_CHECK(hipGetLastError());
    return;
  }
  const int hpc = d > kAppendCols ? 1 : kAppendCols / d;
  const int groups = (tokens + 7) / 8, pieces = 2 * ((hkv + hpc - 1) / hpc) + (q_out ? (hq + hpc - 1) / hpc : 0);
  // Up to what the caches hold the grid takes all groups of v, then of k, then of q, which have different lengths; past that a
  // group's pieces are neighbours, so that its rows are read as one stretch of memory, the first piece moving on with the groups
  // so that every XCD gets every kind.  us, by kind -> by row, q written: 32 / 8 heads of 128, 12000 / 16000 / 32000 tokens (147 /
  // 197 / 393 MB) 64 / 92 / 182 -> 57 / 79 / 150, 32 / 32 at 4096 / 16000 48 / 178 -> 42 / 151, 16 / 16 of 96 at 12000 / 32000 52.8 / 138
  // -> 51.2 / 131; but 64 / 8 of 128 at 4096 (84 MB) 31.4 -> 33.6, 32 / 8 of 64 at 4096 (25 MB) 14.6 -> 15.7
  const int by_row = (long)tokens * (2 * hkv + (q_out ? hq : 0)) * d * 2 >= 100000000 && groups < 65536;
  const dim3 grid(by_row ? pieces : groups, by_row ? groups : pieces);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, (bf16*)q_out, rotate_q, (const bf16*)qkv, (const float*)part, slab,
                       (const int32_t*)positions, (const float*)cos_sin, (bf16*)k_cache, (bf16*)v_cache,
                       (const int32_t*)slots, tokens, hq, hkv, d, bs, by_row);
  };
  switch (part ? nparts : 0) {
    case 0: go(qkv_append_kernel<0>); break;
    case 2: go(qkv_append_kernel<2>); break;
    case 3: go(qkv_append_kernel<3>); break;
    case 4: go(qkv_append_kernel<4>); break;
    case 5: go(qkv_append_kernel<5>); break;
    case 8: go(qkv_append_kernel<8>); break;
    default: DLLM_HOST_CHECK(false, "2, 3, 4, 5 or 8 slabs (ops.APPEND_SLABS)");
  }
  DLLM_HIP_CHECK(hipGetLastError());
}

// ---------------------------------------------------------------------------
// SwiGLU activation: gu [T, 2I] = [gate | up] -> out [T, I] = silu(gate) * up.
// Grid-stride over bf16x8 vectors.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) silu_mul_kernel(bf16* __restrict__ out, const bf16* __restrict__ gu,
                                                       int inter, long total_vec) {
  const int vpr = inter >> 3;
  for (long v = (long)blockIdx.x * 256 + threadIdx.x; v < total_vec; v += (long)gridDim.x * 256) {
    const long t = v / vpr;
    const int c = (int)(v % vpr) * 8;
    bf16x8 g = *reinterpret_cast<const bf16x8*>(gu + t * 2 * inter + c);
    bf16x8 u = *reinterpret_cast<const bf16x8*>(gu + t * 2 * inter + inter + c);
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = f2bf(silu_f(bf2f(g[j])) * bf2f(u[j]));
    *reinterpret_cast<bf16x8*>(out + t * inter + c) = o;
  }
}

void silu_mul(uintptr_t out, uintptr_t gu, int tokens, int inter, uintptr_t stream) {
  DLLM_HOST_CHECK(inter % 8 == 0, "intermediate % 8");
  const long total = (long)tokens * (inter / 8);
  if (total == 0) return;
  long blocks = (total + 255) / 256;
  if (blocks > 256 * 8) blocks = 256 * 8;
  hipLaunchKernelGGL(silu_mul_kernel, dim3((unsigned)blocks), dim3(256), 0, reinterpret_cast<hipStream_t>(stream),
                     (bf16*)out, (const bf16*)gu, inter, total);
  DLLM_HIP_CHECK(hipGetLastError());
}

// ---------------------------------------------------------------------------
// a <- a + b (bf16, 16-byte vectors): closes the residual stream at a stage boundary.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) add_inplace_kernel(bf16* __restrict__ a, const bf16* __restrict__ b,
                                                          long nvec) {
  for (long v = (long)blockIdx.x * 256 + threadIdx.x; v < nvec; v += (long)gridDim.x * 256) {
    bf16x8 x = reinterpret_cast<bf16x8*>(a)[v];
    const bf16x8 y = reinterpret_cast<const bf16x8*>(b)[v];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = f2bf(bf2f(x[j]) + bf2f(y[j]));
    reinterpret_cast<bf16x8*>(a)[v] = x;
  }
}

void add_inplace(uintptr_t a, uintptr_t b, long n, uintptr_t stream) {
  DLLM_HOST_CHECK(n % 8 == 0, "numel % 8");
  const long nvec = n / 8;
  if (nvec == 0) return;
  long blocks = (nvec + 255) / 256;
  if (blocks > 2048) blocks = 2048;
  hipLaunchKernelGGL(add_inplace_kernel, dim3((unsigned)blocks), dim3(256), 0, reinterpret_cast<hipStream_t>(stream),
                     (bf16*)a, (const bf16*)b, nvec);
  DLLM_HIP_CHECK(hipGetLastError());
}

// ---------------------------------------------------------------------------
// K10 tail: greedy argmax over the vocabulary. One 1024-thread workgroup per row.
// Ties resolve to the smallest index (matches torch.argmax on the fp32 values).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void argmax_merge(float& bv, int& bi, float v, int i) {
  if (v > bv || (v == bv && i < bi) || (bv != bv)) { bv = v; bi = i; }
}

__global__ void __launch_bounds__(1024) argmax_kernel(int32_t* __restrict__ out, const bf16* __restrict__ logits,
                                                      int vocab, long row_stride) {
  __shared__ float sv[16];
  __shared__ int si[16];
  const bf16* row = logits + (size_t)blockIdx.x * row_stride;
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  const int nvec = ((((uintptr_t)row) & 15) == 0) ? vocab >> 3 : 0;
  const bf16x8* rv = reinterpret_cast<const bf16x8*>(row);
  // four 16-byte loads in flight per thread before the first compare (one per iteration left the
  // 250 KB row at ~3.5 TB/s).  A thread visits its indices in increasing order, so inside its scan
  // a strict > keeps the smallest index among equal values (one compare and two selects, not the
  // cross-thread merge's tie and NaN rules)
  for (int v0 = threadIdx.x; v0 < nvec; v0 += 4 * 1024) {
    bf16x8 x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int v = v0 + u * 1024;
      if (v < nvec) x[u] = rv[v];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int v = v0 + u * 1024;
      if (v < nvec) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float xv = bf2f(x[u][j]);
          const bool take = xv > bv;
          bv = take ? xv : bv;
          bi = take ? v * 8 + j : bi;
        }
      }
    }
  }
  for (int i = nvec * 8 + threadIdx.x; i < vocab; i += 1024) argmax_merge(bv, bi, bf2f(row[i]), i);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    float ov = __shfl_xor(bv, o, 64);
    int oi = __shfl_xor(bi, o, 64);
    argmax_merge(bv, bi, ov, oi);
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) { sv[wid] = bv; si[wid] = bi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; ++w) argmax_merge(bv, bi, sv[w], si[w]);
    out[blockIdx.x] = bi;
  }
}

void argmax(uintptr_t out, uintptr_t logits, int rows, int vocab, long row_stride, uintptr_t stream) {
  if (rows == 0) return;
  hipLaunchKernelGGL(argmax_kernel, dim3(rows), dim3(1024), 0, reinterpret_cast<hipStream_t>(stream),
                     (int32_t*)out, (const bf16*)logits, vocab, row_stride);
  DLLM_HIP_CHECK(hipGetLastError());
}

}  // namespace dllm
