// Kernels of layer-list models with per-sequence state (ops/seqmix.py): a float32 residual stream
// with RMS norms before and after every sublayer, short causal convolutions whose tail lives in a
// state slot, the real-gated linear recurrent unit (gates, then a chunked linear scan), the
// attention input stages (convolution + per-head norm + interleaved rotation + paged append; whole-
// projection norm + half-split rotation + paged append; per-head norm before or after a paired rotation, with query
// factors, + paged append), embedding (+ learned positions) + norm, the close of
// pre-norm sublayers (one or two outputs, each normed apart), a token shift whose previous row lives in a state
// slot, the entry of a looped span, sublayers between two layer norms, the averaged keys / values of blocks of
// positions, clipped and gelu GLUs and the logit soft cap.  The attention input stages take projection biases and
// values shared between layers.
//
// Every kernel is a template over the activation type T (bf16 or float): the float32 build is the
// exact path (true 32-bit everywhere), the bf16 build keeps in float32 what feeds a norm, a
// rotation, a gate of the recurrence or the state.  Sizes are runtime values with bounds checks,
// no divisibility assumed: widths, head sizes, taps and block counts come from the model's config.
#include <math.h>

#include "common.h"
#include "launchers.h"
#include "stream_common.h"

namespace dllm {

// --------------------------------------------------------------------------- embedding -> f32
// V elements per lane, a row in as many workgroups as it takes (a loop of 2-byte loads waited for each: 16 rows of 2560
// 2.9 us from cached rows, 2.1 now; cold 7.9 us before)
template <typename T, int V>
__global__ void __launch_bounds__(256) sm_embed_kernel(float* __restrict__ out, const int32_t* __restrict__ ids,
                                                       const void* __restrict__ table_, int width, int vocab,
                                                       float scale) {
  int id = ids[blockIdx.x];
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
  for (long i = (blockIdx.y * 256L + threadIdx.x) * V; i < width; i += gridDim.y * 256L * V) {
    float v[V];
    ldv<V>((const T*)table_ + (size_t)id * width + i, v);
#pragma unroll
    for (int j = 0; j < V; ++j) v[j] *= scale;
    stv<V>(out + (size_t)blockIdx.x * width + i, v);
  }
}

void sm_embed_f32(uintptr_t out, uintptr_t ids, uintptr_t table, int tokens, int width, int vocab, float scale, int f32,
                  uintptr_t stream) {
  if (tokens <= 0) return;
  DLLM_HOST_CHECK(width > 0 && vocab > 0, "embed sizes");
  const bool vec = width % 8 == 0 && table % 32 == 0 && out % 32 == 0;
  const dim3 grid(tokens, std::min(65535, (width - 1) / (vec ? 2048 : 256) + 1));
  SM_DISPATCH_V(f32, vec, sm_embed_kernel, grid, dim3(256), 0, stream, (float*)out, (const int32_t*)ids,
                (const void*)table, width, vocab, scale);
}

// --------------------------------------------------------------------------- embedding + RMS norm -> f32 stream
// x = e / sqrt(mean(e^2) + eps) * (offset + w) for e = table[id] * scale (+ pos_table[position], a learned
// vector per position, when given), as the float32 stream and -- when h is given -- also in the activation
// type (the input of a first sublayer that reads the stream unnormed).
template <typename T>
__global__ void __launch_bounds__(256) sm_embed_norm_kernel(float* __restrict__ x, void* __restrict__ h_,
                                                            const int32_t* __restrict__ ids,
                                                            const void* __restrict__ table_, const void* __restrict__ w_,
                                                            int width, int vocab, float eps, float offset, float scale,
                                                            const void* __restrict__ pos_table_,
                                                            const int32_t* __restrict__ positions, int max_pos) {
  __shared__ float red[16];
  const T* table = (const T*)table_;
  const T* w = (const T*)w_;
  int id = ids[blockIdx.x];
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
  const T* src = table + (size_t)id * width;
  const T* prow = nullptr;
  if (pos_table_) {
    int p = positions[blockIdx.x];
    p = p < 0 ? 0 : (p >= max_pos ? max_pos - 1 : p);
    prow = (const T*)pos_table_ + (size_t)p * width;
  }
  float ss = 0.f;
  for (int i = threadIdx.x; i < width; i += 256) {
    const float v = ldf(src + i) * scale + (prow ? ldf(prow + i) : 0.f);
    ss += v * v;
  }
  ss = block_sum(ss, red);
  const float inv = 1.0f / sqrtf(ss / (float)width + eps);
  float* dst = x + (size_t)blockIdx.x * width;
  T* h = h_ ? (T*)h_ + (size_t)blockIdx.x * width : nullptr;
  for (int i = threadIdx.x; i < width; i += 256) {
    const float e = ldf(src + i) * scale + (prow ? ldf(prow + i) : 0.f);
    const float v = e * inv * (offset + ldf(w + i));
    dst[i] = v;
    if (h) stf(h + i, v);
  }
}

void sm_embed_norm(uintptr_t x, uintptr_t h, uintptr_t ids, uintptr_t table, uintptr_t w, int tokens, int width,
                   int vocab, float eps, float offset, float scale, uintptr_t pos_table, uintptr_t positions,
                   int max_pos, int f32, uintptr_t stream) {
  if (tokens <= 0) return;
  DLLM_HOST_CHECK(width > 0 && vocab > 0 && x && w && (!pos_table || (positions && max_pos > 0)),
                  "embed_norm arguments");
  SM_DISPATCH(f32, sm_embed_norm_kernel, dim3(tokens), dim3(256), 0, stream, (float*)x, (void*)h, (const int32_t*)ids,
              (const void*)table, (const void*)w, width, vocab, eps, offset, scale, (const void*)pos_table,
              (const int32_t*)positions, max_pos);
}

// --------------------------------------------------------------------------- RMS norm of an f32 row
// y = x * rsqrt(mean(x^2) + eps) * (offset + w); one workgroup per row, V elements per lane and step.
template <typename T, int V>
__global__ void __launch_bounds__(256) sm_rms_norm_kernel(void* __restrict__ y_, const float* __restrict__ x,
                                                          const void* __restrict__ w_, int width, float eps,
                                                          float offset) {
  __shared__ float red[16];
  T* y = (T*)y_ + (size_t)blockIdx.x * width;
  const T* w = (const T*)w_;
  const float* xr = x + (size_t)blockIdx.x * width;
  float ss = 0.f;
  for (int i = threadIdx.x * V; i < width; i += 256 * V) {
    float v[V];
    ldv<V>(xr + i, v);
#pragma unroll
    for (int j = 0; j < V; ++j) ss += v[j] * v[j];
  }
  ss = block_sum(ss, red);
  const float inv = 1.0f / sqrtf(ss / (float)width + eps);
  for (int i = threadIdx.x * V; i < width; i += 256 * V) {
    float v[V], g[V];
    ldv<V>(xr + i, v);
    ldv<V>(w + i, g);
#pragma unroll
    for (int j = 0; j < V; ++j) v[j] = v[j] * inv * (offset + g[j]);
    stv<V>(y + i, v);
  }
}

// The same for a row that fits the registers (NV pieces of 8 elements per lane, the same lane for the same elements): x
// and w loaded once, before the first use, off clamped places.
template <typename T, int NV>
__global__ void __launch_bounds__(256) sm_rms_norm_row_kernel(void* __restrict__ y_, const float* __restrict__ x,
                                                              const void* __restrict__ w_, int width, float eps,
                                                              float offset) {
  __shared__ float red[16];
  T* y = (T*)y_ + (size_t)blockIdx.x * width;
  const float* xr = x + (size_t)blockIdx.x * width;
  float v[NV][8], g[NV][8];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int i = min((k * 256 + (int)threadIdx.x) * 8, width - 8);
    ldv<8>(xr + i, v[k]);
    ldv<8>((const T*)w_ + i, g[k]);
  }
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < NV; ++k)
    if ((k * 256 + (int)threadIdx.x) * 8 < width) {
#pragma unroll
      for (int j = 0; j < 8; ++j) ss += v[k][j] * v[k][j];
    }
  ss = block_sum<256>(ss, red);
  const float inv = 1.0f / sqrtf(ss / (float)width + eps);
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int i = (k * 256 + threadIdx.x) * 8;
    if (i < width) {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[k][j] = v[k][j] * inv * (offset + g[k][j]);
      stv<8>(y + i, v[k]);
    }
  }
}

void sm_rms_norm(uintptr_t y, uintptr_t x, uintptr_t w, int rows, int width, float eps, float offset, int f32,
                 uintptr_t stream) {
  if (rows <= 0) return;
  DLLM_HOST_CHECK(width > 0, "norm width");
  if (width % 8 == 0 && width <= 8192) {
    const auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(rows), dim3(256), 0, (hipStream_t)stream, (void*)y, (const float*)x, (const void*)w,
                         width, eps, offset);
    };
#define SM_RMS_ROW(T)                                                \
  do {                                                               \
    if (width <= 2048) go(sm_rms_norm_row_kernel<T, 1>);             \
    else if (width <= 4096) go(sm_rms_norm_row_kernel<T, 2>);        \
    else go(sm_rms_norm_row_kernel<T, 4>);                           \
  } while (0)
    if (f32) SM_RMS_ROW(float);
    else SM_RMS_ROW(bf16);
#undef SM_RMS_ROW
    DLLM_HIP_CHECK(hipGetLastError());
    return;
  }
  SM_DISPATCH_V(f32, width % 8 == 0, sm_rms_norm_kernel, dim3(rows), dim3(256), 0, stream, (void*)y, (const float*)x,
                (const void*)w, width, eps, offset);
}

// --------------------------------------------------------------------------- close of a sublayer (rows past 16384)
// x += mult * rms_norm(v) * (offset + w_post) with v = o + bias, or v = s1 o + s2 o2 when a second input is
// given (two mixers side by side);  h = rms_norm(x) * (offset + w_next) when w_next, else, when h is
// given, the new stream itself in the activation type (a following sublayer that reads x unnormed)
// (offset 1: weights stored around zero; 0: plain weights).
template <typename T, int V>
__global__ void __launch_bounds__(256) sm_post_norm_add_kernel(float* __restrict__ x, const void* __restrict__ o_,
                                                               const void* __restrict__ bias_,
                                                               const void* __restrict__ wp_,
                                                               const void* __restrict__ wn_, void* __restrict__ h_,
                                                               int width, float eps, float mult, float offset,
                                                               const void* __restrict__ o2_, float s1, float s2) {
  __shared__ float red[16];
  const T* o = (const T*)o_ + (size_t)blockIdx.x * width;
  const T* o2 = o2_ ? (const T*)o2_ + (size_t)blockIdx.x * width : nullptr;
  const T* bias = (const T*)bias_;
  const T* wp = (const T*)wp_;
  const T* wn = (const T*)wn_;
  float* xr = x + (size_t)blockIdx.x * width;
  float ss = 0.f;
  for (int i = threadIdx.x * V; i < width; i += 256 * V) {
    float v[V], bb[V];
    ldv<V>(o + i, v);
    if (o2) {
      ldv<V>(o2 + i, bb);
#pragma unroll
      for (int j = 0; j < V; ++j) v[j] = s1 * v[j] + s2 * bb[j];
    }
    if (bias) {
      ldv<V>(bias + i, bb);
#pragma unroll
      for (int j = 0; j < V; ++j) v[j] += bb[j];
    }
#pragma unroll
    for (int j = 0; j < V; ++j) ss += v[j] * v[j];
  }
  ss = block_sum(ss, red);
  const float inv = 1.0f / sqrtf(ss / (float)width + eps);
  float sq = 0.f;
  for (int i = threadIdx.x * V; i < width; i += 256 * V) {
    float v[V], bb[V], g[V], xv[V];
    ldv<V>(o + i, v);
    if (o2) {
      ldv<V>(o2 + i, bb);
#pragma unroll
      for (int j = 0; j < V; ++j) v[j] = s1 * v[j] + s2 * bb[j];
    }
    if (bias) {
      ldv<V>(bias + i, bb);
#pragma unroll
      for (int j = 0; j < V; ++j) v[j] += bb[j];
    }
    ldv<V>(wp + i, g);
    ldv<V>(xr + i, xv);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      xv[j] = xv[j] + mult * (v[j] * inv * (offset + g[j]));
      sq += xv[j] * xv[j];
    }
    stv<V>(xr + i, xv);
    if (!wn && h_) stv<V>((T*)h_ + (size_t)blockIdx.x * width + i, xv);
  }
  if (!wn) return;
  sq = block_sum(sq, red);
  const float inv2 = 1.0f / sqrtf(sq / (float)width + eps);
  T* h = (T*)h_ + (size_t)blockIdx.x * width;
  for (int i = threadIdx.x * V; i < width; i += 256 * V) {      // each lane re-reads what it wrote itself
    float xv[V], g[V];
    ldv<V>(xr + i, xv);
    ldv<V>(wn + i, g);
#pragma unroll
    for (int j = 0; j < V; ++j) xv[j] = xv[j] * inv2 * (offset + g[j]);
    stv<V>(h + i, xv);
  }
}

// --------------------------------------------------------------------------- layer norms on the float32 stream
// One workgroup per row, the row in registers (NV pieces of V consecutive elements per lane): the mean first, then the
// mean of the squared deviations from it.
template <int V, int NV>
__device__ __forceinline__ void ln_stats(const float (&v)[NV][V], int width, float eps, float* red, float& mean, float& inv) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < NV; ++k)
#pragma unroll
    for (int j = 0; j < V; ++j) s += v[k][j];                          // places beyond the row hold 0
  s = wave_sum(s);
  if (lane == 0) red[wid] = s;
  __syncthreads();
  mean = (red[0] + red[1] + red[2] + red[3]) / (float)width;
  float q = 0.f;
#pragma unroll
  for (int k = 0; k < NV; ++k)
    if ((k * 256 + (int)threadIdx.x) * V < width) {
#pragma unroll
      for (int j = 0; j < V; ++j) q += (v[k][j] - mean) * (v[k][j] - mean);
    }
  q = wave_sum(q);
  if (lane == 0) red[4 + wid] = q;
  __syncthreads();
  inv = 1.0f / sqrtf((red[4] + red[5] + red[6] + red[7]) / (float)width + eps);
}

template <typename T, int V, int NV>
__global__ void __launch_bounds__(256) sm_layer_norm_kernel(void* __restrict__ y_, const float* __restrict__ x,
                                                            const void* __restrict__ w_, const void* __restrict__ b_,
                                                            int width, float eps) {
  __shared__ float red[8];
  const float* xr = x + (size_t)blockIdx.x * width;
  float v[NV][V], w[NV][V], b[NV][V];
#pragma unroll
  for (int k = 0; k < NV; ++k) {                  // off clamped places: no load waits behind another's guard
    const int i = min((k * 256 + (int)threadIdx.x) * V, width - V);
    ldv<V>(xr + i, v[k]);
    ldv<V>((const T*)w_ + i, w[k]);
    ldv<V>((const T*)b_ + i, b[k]);
  }
#pragma unroll
  for (int k = 0; k < NV; ++k)
    if ((k * 256 + (int)threadIdx.x) * V >= width) {
#pragma unroll
      for (int j = 0; j < V; ++j) v[k][j] = 0.f;
    }
  float mean, inv;
  ln_stats<V, NV>(v, width, eps, red, mean, inv);
  T* y = (T*)y_ + (size_t)blockIdx.x * width;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int i = (k * 256 + threadIdx.x) * V;
    if (i < width) {
#pragma unroll
      for (int j = 0; j < V; ++j) v[k][j] = (v[k][j] - mean) * inv * w[k][j] + b[k][j];
      stv<V>(y + i, v[k]);
    }
  }
}

// One row of a product that is still in `parts` split-K slabs (V = 4; common.h part_elem): their sum, rounded to bf16 as the
// reduction of a split product rounds it.  CH slabs a round, off clamped places, all of a round's loads before its first
// use (with the adds behind `slab < parts` hipcc moved each load into its branch: ten round trips for 12 slabs).
template <int CH, int NV, int V>
__device__ __forceinline__ void ln_slab_rounds(const float* __restrict__ P, int parts, size_t row, int width, float (&v)[NV][V]) {
  typedef part_elem raw __attribute__((ext_vector_type(4)));
  const size_t slab = (size_t)gridDim.x * width;
  float a[NV][4];
#pragma unroll
  for (int k = 0; k < NV; ++k)
#pragma unroll
    for (int j = 0; j < 4; ++j) a[k][j] = 0.f;
  for (int s0 = 0; s0 < parts; s0 += CH) {
    raw l[CH][NV];
#pragma unroll
    for (int u = 0; u < CH; ++u)
#pragma unroll
      for (int k = 0; k < NV; ++k)
        l[u][k] = *reinterpret_cast<const raw*>(reinterpret_cast<const part_elem*>(P) + min(s0 + u, parts - 1) * slab + row +
                                                min((k * 256 + (int)threadIdx.x) * V, width - V));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < CH; ++u)
#pragma unroll
      for (int k = 0; k < NV; ++k)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float t = a[k][j] + part_value(l[u][k][j]);
          a[k][j] = s0 + u < parts ? t : a[k][j];
        }
  }
#pragma unroll
  for (int k = 0; k < NV; ++k)
#pragma unroll
    for (int j = 0; j < V; ++j) v[k][j] = bf2f(f2bf(a[k][j & 3]));
}
template <int NV, int V>
__device__ __forceinline__ void ln_slabs(const float* __restrict__ P, int parts, size_t row, int width, float (&v)[NV][V]) {
  if constexpr (NV <= 4) {
    if (parts <= 4) ln_slab_rounds<4, NV, V>(P, parts, row, width, v);        // uniform
    else if (parts <= 8) ln_slab_rounds<8, NV, V>(P, parts, row, width, v);
    else ln_slab_rounds<12, NV, V>(P, parts, row, width, v);
  } else {
    ln_slab_rounds<2, NV, V>(P, parts, row, width, v);
  }
}

// The close of a sublayer between two layer norms: x += layer_norm(o + bias) (weight wp, bias bp; `bias` null: none), and
// with wn: h = layer_norm(x) (wn, bn), the next sublayer's input.  parts > 0: o is the sum of that many split-K slabs
// [rows, width] (common.h part_load; bf16 results, rounded as the reduction of a split product rounds them).
// Two kernels of one body: the slabs in flight would cost the other form its occupancy (6376 rows: 37 us as one, 30.5 apart).
template <typename T, int V, int NV, bool SLABS>
__device__ __forceinline__ void post_layer_norm_row(
    float* red, float* __restrict__ x, const void* __restrict__ o_, int parts, const void* __restrict__ bias_,
    const void* __restrict__ wp_, const void* __restrict__ bp_, const void* __restrict__ wn_, const void* __restrict__ bn_,
    void* __restrict__ h_, int width, float eps) {
  const size_t row = (size_t)blockIdx.x * width;
  float* xr = x + row;
  typedef T vec __attribute__((ext_vector_type(V)));
  typedef float fvec __attribute__((ext_vector_type(V)));
  // up to 16 elements per lane are held with all that goes with them; a wider row's stream and weights come in rounds of 16
  // elements (all at once they took 512 registers and scratch: 4096 rows of 16383, f32, 664 us, of 4097 241)
  constexpr bool kEarly = NV * V <= 16;
  constexpr int CH = kEarly ? NV : 16 / V;
  float v[NV][V], xv[NV][V];
  fvec rx[NV];
  vec rw[NV], rb[NV], rwn[NV], rbn[NV], rc[NV];
  // every load off a clamped place, in its stored form and before the first use: no load waits behind
  // another's guard or conversion, and the next norm's weights do not wait for this one's sums (16 rows of 2560: with 12
  // slabs 8.6 us before, 5.4 now, without 4.7 and 3.6; 6376 rows 34.2 and 30.5)
  auto at = [&](int k) { return min((k * 256 + (int)threadIdx.x) * V, width - V); };
  auto load = [&](vec (&r)[NV], const void* from, int k0, int n) {
#pragma unroll
    for (int k = k0; k < k0 + n; ++k) r[k] = *reinterpret_cast<const vec*>((const T*)from + at(k));
  };
  auto load_x = [&](int k0, int n) {
#pragma unroll
    for (int k = k0; k < k0 + n; ++k) rx[k] = *reinterpret_cast<const fvec*>(xr + at(k));
  };
  vec ro[NV];
  if (kEarly) load_x(0, NV);
  if (!SLABS) load(ro, (const T*)o_ + row, 0, NV);
  if (kEarly) load(rw, wp_, 0, NV), load(rb, bp_, 0, NV);
  if (kEarly && bias_) load(rc, bias_, 0, NV);
  if (kEarly && wn_) load(rwn, wn_, 0, NV), load(rbn, bn_, 0, NV);
  if constexpr (SLABS) {
    ln_slabs<NV>((const float*)o_, parts, row, width, v);
  } else {
#pragma unroll
    for (int k = 0; k < NV; ++k)
#pragma unroll
      for (int j = 0; j < V; ++j) v[k][j] = (float)ro[k][j];
  }
#pragma unroll
  for (int k0 = 0; k0 < NV; k0 += CH) {
    if (!kEarly && bias_) load(rc, bias_, k0, CH);
#pragma unroll
    for (int k = k0; k < k0 + CH; ++k) {
      const bool in = (k * 256 + (int)threadIdx.x) * V < width;
#pragma unroll
      for (int j = 0; j < V; ++j) {
        if (bias_) v[k][j] += (float)rc[k][j];
        v[k][j] = in ? v[k][j] : 0.f;
      }
    }
  }
  float mean, inv;
  ln_stats<V, NV>(v, width, eps, red, mean, inv);
#pragma unroll
  for (int k0 = 0; k0 < NV; k0 += CH) {
    if (!kEarly) load_x(k0, CH), load(rw, wp_, k0, CH), load(rb, bp_, k0, CH);
#pragma unroll
    for (int k = k0; k < k0 + CH; ++k) {
      const int i = (k * 256 + threadIdx.x) * V;
#pragma unroll
      for (int j = 0; j < V; ++j) xv[k][j] = i < width ? rx[k][j] : 0.f;
      if (i < width) {
#pragma unroll
        for (int j = 0; j < V; ++j) xv[k][j] += (v[k][j] - mean) * inv * (float)rw[k][j] + (float)rb[k][j];
        stv<V>(xr + i, xv[k]);
      }
    }
    if (!kEarly) __builtin_amdgcn_sched_barrier(0);
  }
  if (!wn_) return;
  ln_stats<V, NV>(xv, width, eps, red + 8, mean, inv);
  T* h = (T*)h_ + row;
#pragma unroll
  for (int k0 = 0; k0 < NV; k0 += CH) {
    if (!kEarly) load(rwn, wn_, k0, CH), load(rbn, bn_, k0, CH);
#pragma unroll
    for (int k = k0; k < k0 + CH; ++k) {
      const int i = (k * 256 + threadIdx.x) * V;
      if (i < width) {
#pragma unroll
        for (int j = 0; j < V; ++j) xv[k][j] = (xv[k][j] - mean) * inv * (float)rwn[k][j] + (float)rbn[k][j];
        stv<V>(h + i, xv[k]);
      }
    }
    if (!kEarly) __builtin_amdgcn_sched_barrier(0);
  }
}

template <typename T, int V, int NV>
__global__ void __launch_bounds__(256) sm_post_layer_norm_kernel(
    float* __restrict__ x, const void* __restrict__ o, const void* __restrict__ bias, const void* __restrict__ wp,
    const void* __restrict__ bp, const void* __restrict__ wn, const void* __restrict__ bn, void* __restrict__ h, int width,
    float eps) {
  __shared__ float red[16];
  post_layer_norm_row<T, V, NV, false>(red, x, o, 0, bias, wp, bp, wn, bn, h, width, eps);
}
template <typename T, int V, int NV>
__global__ void __launch_bounds__(256) sm_post_layer_norm_slabs_kernel(
    float* __restrict__ x, const void* __restrict__ o, int parts, int width, const void* __restrict__ bias,
    const void* __restrict__ wp, const void* __restrict__ bp, const void* __restrict__ wn, const void* __restrict__ bn,
    void* __restrict__ h, float eps) {              // (sizes among the first 14 words: those come with the wave)
  __shared__ float red[16];
  post_layer_norm_row<T, V, NV, true>(red, x, o, parts, bias, wp, bp, wn, bn, h, width, eps);
}

// V = 4 elements per lane and piece (width a multiple of 4), else one; the fewest pieces that hold the row
#define SM_LN_DISPATCH(f32, width, KERNEL, grid, stream, ...)                                                        \
  do {                                                                                                             \
    DLLM_HOST_CHECK((width) > 0 && (width) <= 16384, "layer norm width");                                          \
    const int np_ = ((width) + ((width) % 4 ? 255 : 1023)) / ((width) % 4 ? 256 : 1024);                           \
    if ((width) % 4 == 0) {                                                                                        \
      if (np_ <= 1) SM_LN_GO(f32, KERNEL, 4, 1, grid, stream, __VA_ARGS__);                                        \
      else if (np_ <= 2) SM_LN_GO(f32, KERNEL, 4, 2, grid, stream, __VA_ARGS__);                                   \
      else if (np_ <= 3) SM_LN_GO(f32, KERNEL, 4, 3, grid, stream, __VA_ARGS__);                                   \
      else if (np_ <= 4) SM_LN_GO(f32, KERNEL, 4, 4, grid, stream, __VA_ARGS__);                                   \
      else if (np_ <= 8) SM_LN_GO(f32, KERNEL, 4, 8, grid, stream, __VA_ARGS__);                                   \
      else if (np_ <= 12) SM_LN_GO(f32, KERNEL, 4, 12, grid, stream, __VA_ARGS__);                                 \
      else SM_LN_GO(f32, KERNEL, 4, 16, grid, stream, __VA_ARGS__);                                                \
    } else if (np_ <= 4) SM_LN_GO(f32, KERNEL, 1, 4, grid, stream, __VA_ARGS__);                                   \
    else if (np_ <= 16) SM_LN_GO(f32, KERNEL, 1, 16, grid, stream, __VA_ARGS__);                                   \
    else if (np_ <= 32) SM_LN_GO(f32, KERNEL, 1, 32, grid, stream, __VA_ARGS__);                                   \
    else SM_LN_GO(f32, KERNEL, 1, 64, grid, stream, __VA_ARGS__);                                                  \
    DLLM_HIP_CHECK(hipGetLastError());                                                                             \
  } while (0)
// ... of a product in slabs (bf16, width a multiple of 4)
#define SM_LN_SLABS(width, KERNEL, grid, stream, ...)                                                                \
  do {                                                                                                             \
    DLLM_HOST_CHECK((width) > 0 && (width) <= 16384 && (width) % 4 == 0, "layer norm width");                      \
    const auto go_ = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(256), 0, (hipStream_t)(stream), __VA_ARGS__); }; \
    const int np_ = ((width) + 1023) / 1024;                                                                       \
    if (np_ <= 1) go_(KERNEL<bf16, 4, 1>);                                                                         \
    else if (np_ <= 2) go_(KERNEL<bf16, 4, 2>);                                                                    \
    else if (np_ <= 3) go_(KERNEL<bf16, 4, 3>);                                                                    \
    else if (np_ <= 4) go_(KERNEL<bf16, 4, 4>);                                                                    \
    else if (np_ <= 8) go_(KERNEL<bf16, 4, 8>);                                                                    \
    else go_(KERNEL<bf16, 4, 16>);                                                                                 \
    DLLM_HIP_CHECK(hipGetLastError());                                                                             \
  } while (0)
#define SM_LN_GO(f32, KERNEL, V, NV, grid, stream, ...)                                                              \
  do {                                                                                                             \
    if (f32) hipLaunchKernelGGL(HIP_KERNEL_NAME(KERNEL<float, V, NV>), grid, dim3(256), 0, (hipStream_t)(stream), __VA_ARGS__); \
    else hipLaunchKernelGGL(HIP_KERNEL_NAME(KERNEL<bf16, V, NV>), grid, dim3(256), 0, (hipStream_t)(stream), __VA_ARGS__);      \
  } while (0)

void sm_layer_norm(uintptr_t y, uintptr_t x, uintptr_t w, uintptr_t b, int rows, int width, float eps, int f32,
                   uintptr_t stream) {
  if (rows <= 0) return;
  DLLM_HOST_CHECK(y && x && w && b, "layer norm arguments");
  SM_LN_DISPATCH(f32, width, sm_layer_norm_kernel, dim3(rows), stream, (void*)y, (const float*)x, (const void*)w,
                 (const void*)b, width, eps);
}

// The embedding as the float32 stream and the first sublayer's normed input of it in one launch (sm_embed_kernel's row and, in
// the same lanes and order, sm_rms_norm_row_kernel's or sm_layer_norm_kernel's norm of it): a decode step is a chain of launches
// whose round trips bound it, and a prompt reads its stream once less.  us in two -> one, RMS: one row of 1024 3.9 -> 2.4, 16 / 6376 of
// 2560 4.4 / 31 -> 2.9 / 22; layer norm: 32 / 7021 of 2560 4.5 / 34 -> 3.2 / 23.
template <typename T, int V, int NV, bool LAYER>
__global__ void __launch_bounds__(256) sm_embed_first_norm_kernel(
    const int32_t* __restrict__ ids, const void* __restrict__ table_, int width, int vocab, float scale, float eps, float offset,
    const void* __restrict__ w_, const void* __restrict__ b_, float* __restrict__ x_, void* __restrict__ y_) {
  __shared__ float red[16];
  float v[NV][V], w[NV][V], b[NV][V];
#pragma unroll
  for (int k = 0; k < NV; ++k) {                  // off clamped places: no load waits behind another's guard
    const int i = min((k * 256 + (int)threadIdx.x) * V, width - V);
    ldv<V>((const T*)w_ + i, w[k]);
    if constexpr (LAYER) ldv<V>((const T*)b_ + i, b[k]);
  }
  int id = ids[blockIdx.x];
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
  const T* src = (const T*)table_ + (size_t)id * width;
#pragma unroll
  for (int k = 0; k < NV; ++k) ldv<V>(src + min((k * 256 + (int)threadIdx.x) * V, width - V), v[k]);
  float* x = x_ + (size_t)blockIdx.x * width;
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int i = (k * 256 + threadIdx.x) * V;
#pragma unroll
    for (int j = 0; j < V; ++j) v[k][j] *= scale;
    if (i < width) {
      stv<V>(x + i, v[k]);
#pragma unroll
      for (int j = 0; j < V; ++j) ss += v[k][j] * v[k][j];
    } else {
#pragma unroll
      for (int j = 0; j < V; ++j) v[k][j] = 0.f;
    }
  }
  float mean = 0.f, inv;
  if constexpr (LAYER) ln_stats<V, NV>(v, width, eps, red, mean, inv);
  else inv = 1.0f / sqrtf(block_sum<256>(ss, red) / (float)width + eps);
  T* y = (T*)y_ + (size_t)blockIdx.x * width;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int i = (k * 256 + threadIdx.x) * V;
    if (i < width) {
#pragma unroll
      for (int j = 0; j < V; ++j)
        v[k][j] = LAYER ? (v[k][j] - mean) * inv * w[k][j] + b[k][j] : v[k][j] * inv * (offset + w[k][j]);
      stv<V>(y + i, v[k]);
    }
  }
}

// b: the bias of a layer norm, 0: an RMS norm with weights (offset + w).  Widths: sm_embed_first_norm_fits
bool sm_embed_first_norm_fits(int width, bool layer) { return layer ? width % 4 == 0 && width <= 4096 : width % 8 == 0 && width <= 8192; }

void sm_embed_first_norm(uintptr_t x, uintptr_t y, uintptr_t ids, uintptr_t table, uintptr_t w, uintptr_t b, int tokens, int width,
                         int vocab, float scale, float eps, float offset, int f32, uintptr_t stream) {
  if (tokens <= 0) return;
  DLLM_HOST_CHECK(width > 0 && vocab > 0 && x && y && ids && table && w && sm_embed_first_norm_fits(width, b != 0), "embedding and norm sizes");
  DLLM_HOST_CHECK((x | y | table | w | b) % 32 == 0, "embedding and norm alignment");
  const auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(tokens), dim3(256), 0, (hipStream_t)stream, (const int32_t*)ids, (const void*)table, width, vocab,
                       scale, eps, offset, (const void*)w, (const void*)b, (float*)x, (void*)y);
  };
#define SM_EFN(T)                                                                  \
  do {                                                                             \
    if (b) {                                                                       \
      if (width <= 1024) go(sm_embed_first_norm_kernel<T, 4, 1, true>);            \
      else if (width <= 2048) go(sm_embed_first_norm_kernel<T, 4, 2, true>);       \
      else if (width <= 3072) go(sm_embed_first_norm_kernel<T, 4, 3, true>);       \
      else go(sm_embed_first_norm_kernel<T, 4, 4, true>);                          \
    } else if (width <= 2048) go(sm_embed_first_norm_kernel<T, 8, 1, false>);      \
    else if (width <= 4096) go(sm_embed_first_norm_kernel<T, 8, 2, false>);        \
    else go(sm_embed_first_norm_kernel<T, 8, 4, false>);                           \
  } while (0)
  if (f32) SM_EFN(float);
  else SM_EFN(bf16);
#undef SM_EFN
  DLLM_HIP_CHECK(hipGetLastError());
}

void sm_post_layer_norm_add(uintptr_t x, uintptr_t o, int parts, uintptr_t bias, uintptr_t w_post, uintptr_t b_post,
                            uintptr_t w_next, uintptr_t b_next, uintptr_t h, int rows, int width, float eps, int f32,
                            uintptr_t stream) {
  if (rows <= 0) return;
  DLLM_HOST_CHECK(x && o && w_post && b_post && (!w_next || (b_next && h)), "post_layer_norm_add arguments");
  DLLM_HOST_CHECK(parts >= 0 && (parts == 0 || (!f32 && width % 4 == 0)), "post_layer_norm_add slabs");
  if (parts > 0)
    SM_LN_SLABS(width, sm_post_layer_norm_slabs_kernel, dim3(rows), stream, (float*)x, (const void*)o, parts,
                width, (const void*)bias, (const void*)w_post, (const void*)b_post, (const void*)w_next, (const void*)b_next,
                (void*)h, eps);
  else
    SM_LN_DISPATCH(f32, width, sm_post_layer_norm_kernel, dim3(rows), stream, (float*)x, (const void*)o,
                   (const void*)bias, (const void*)w_post, (const void*)b_post, (const void*)w_next, (const void*)b_next,
                   (void*)h, width, eps);
}

// The close of a sublayer around RMS norms, the row in registers (NV pieces of V elements per lane): every load -- o or its
// slabs, the second input, bias, stream and both weights -- goes out before the first use, and nothing is read twice (the
// three-pass form above re-read o, x and the new x, with each pass's loads behind a block reduction).
// parts > 0: o is the sum of that many split-K slabs [rows, width], rounded as the reduction of a split product rounds it.
// 2560 wide, bf16: 16 rows 4.3 -> 3.2 us (bound by the launch and two reductions), 6376 rows 44 -> 35 us (5.6 TB/s).
// LAST: h is the norm of the whole stack's output, which else is a launch of sm_rms_norm: the row passes through LDS (`row_s`,
// width floats) into that kernel's lanes, so that its sum has the same order and h the same bits (a step of the small layer list takes
// as long as with the close's own order).
template <typename T, int V, int NV, bool SLABS, bool LAST = false>
__device__ __forceinline__ void post_norm_row(float* red, float* __restrict__ x, const void* __restrict__ o_, int parts,
                                              const void* __restrict__ bias_, const void* __restrict__ wp_,
                                              const void* __restrict__ wn_, void* __restrict__ h_, int width, float eps,
                                              float mult, float offset, const void* __restrict__ o2_, float s1, float s2,
                                              float* row_s = nullptr) {
  const size_t row = (size_t)blockIdx.x * width;
  float* xr = x + row;
  typedef T vec __attribute__((ext_vector_type(V)));
  typedef float fvec __attribute__((ext_vector_type(V)));
  float v[NV][V], xv[NV][V];
  fvec rx[NV];
  vec rwp[NV], rwn[NV], r2[NV], rc[NV];
  // in their stored form: no load behind a conversion (hipcc would wait there)
  auto at = [&](int k) { return min((k * 256 + (int)threadIdx.x) * V, width - V); };
  auto load = [&](vec (&r)[NV], const void* from) {
#pragma unroll
    for (int k = 0; k < NV; ++k) r[k] = *reinterpret_cast<const vec*>((const T*)from + at(k));
  };
#pragma unroll
  for (int k = 0; k < NV; ++k) rx[k] = *reinterpret_cast<const fvec*>(xr + at(k));
  vec ro[NV];
  if (!SLABS) load(ro, (const T*)o_ + row);
  load(rwp, wp_);
  typedef T vec8 __attribute__((ext_vector_type(8)));
  constexpr int N8 = LAST ? (NV * V + 7) / 8 : 1;
  vec8 rw8[N8];
  auto at8 = [&](int k) { return min((k * 256 + (int)threadIdx.x) * 8, width - 8); };
  if constexpr (LAST) {
#pragma unroll
    for (int k = 0; k < N8; ++k) rw8[k] = *reinterpret_cast<const vec8*>((const T*)wn_ + at8(k));
  } else {
    if (wn_) load(rwn, wn_);
  }
  if (o2_) load(r2, (const T*)o2_ + row);
  if (bias_) load(rc, bias_);
  if constexpr (SLABS) {
    ln_slabs<NV>((const float*)o_, parts, row, width, v);
  } else {
#pragma unroll
    for (int k = 0; k < NV; ++k)
#pragma unroll
      for (int j = 0; j < V; ++j) v[k][j] = (float)ro[k][j];
  }
#pragma unroll
  for (int k = 0; k < NV; ++k)
#pragma unroll
    for (int j = 0; j < V; ++j) {
      xv[k][j] = rx[k][j];
      if (o2_) v[k][j] = s1 * v[k][j] + s2 * (float)r2[k][j];
      if (bias_) v[k][j] += (float)rc[k][j];
    }
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < NV; ++k)
    if ((k * 256 + (int)threadIdx.x) * V < width) {
#pragma unroll
      for (int j = 0; j < V; ++j) ss += v[k][j] * v[k][j];
    }
  ss = block_sum<256>(ss, red);
  const float inv = 1.0f / sqrtf(ss / (float)width + eps);
  float sq = 0.f;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int i = (k * 256 + threadIdx.x) * V;
    if (i < width) {
#pragma unroll
      for (int j = 0; j < V; ++j) {
        xv[k][j] = xv[k][j] + mult * (v[k][j] * inv * (offset + (float)rwp[k][j]));
        sq += xv[k][j] * xv[k][j];
      }
      stv<V>(xr + i, xv[k]);
      if constexpr (LAST) stv<V>(row_s + i, xv[k]);
      else if (!wn_ && h_) stv<V>((T*)h_ + row + i, xv[k]);
    }
  }
  if constexpr (LAST) {
    __syncthreads();
    float y[N8][8];
    float s8 = 0.f;
#pragma unroll
    for (int k = 0; k < N8; ++k) {
      ldv<8>(row_s + at8(k), y[k]);
      if ((k * 256 + (int)threadIdx.x) * 8 < width) {
#pragma unroll
        for (int j = 0; j < 8; ++j) s8 += y[k][j] * y[k][j];
      }
    }
    s8 = block_sum<256>(s8, red);
    const float inv8 = 1.0f / sqrtf(s8 / (float)width + eps);
#pragma unroll
    for (int k = 0; k < N8; ++k) {
      const int i = (k * 256 + threadIdx.x) * 8;
      if (i < width) {
#pragma unroll
        for (int j = 0; j < 8; ++j) y[k][j] = y[k][j] * inv8 * (offset + (float)rw8[k][j]);
        stv<8>((T*)h_ + row + i, y[k]);
      }
    }
    return;
  }
  if (!wn_) return;
  sq = block_sum<256>(sq, red);
  const float inv2 = 1.0f / sqrtf(sq / (float)width + eps);
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int i = (k * 256 + threadIdx.x) * V;
    if (i < width) {
#pragma unroll
      for (int j = 0; j < V; ++j) xv[k][j] = xv[k][j] * inv2 * (offset + (float)rwn[k][j]);
      stv<V>((T*)h_ + row + i, xv[k]);
    }
  }
}

template <typename T, int V, int NV>
__global__ void __launch_bounds__(256) sm_post_norm_row_kernel(float* __restrict__ x, const void* __restrict__ o,
                                                               const void* __restrict__ bias, const void* __restrict__ wp,
                                                               const void* __restrict__ wn, void* __restrict__ h, int width,
                                                               float eps, float mult, float offset,
                                                               const void* __restrict__ o2, float s1, float s2) {
  __shared__ float red[16];
  post_norm_row<T, V, NV, false>(red, x, o, 0, bias, wp, wn, h, width, eps, mult, offset, o2, s1, s2);
}
template <typename T, int V, int NV>
__global__ void __launch_bounds__(256) sm_post_norm_slabs_kernel(float* __restrict__ x, const void* __restrict__ o,
                                                                 int parts, const void* __restrict__ bias,
                                                                 const void* __restrict__ wp, const void* __restrict__ wn,
                                                                 void* __restrict__ h, int width, float eps, float mult,
                                                                 float offset, const void* __restrict__ o2, float s1,
                                                                 float s2) {
  __shared__ float red[16];
  post_norm_row<T, V, NV, true>(red, x, o, parts, bias, wp, wn, h, width, eps, mult, offset, o2, s1, s2);
}

template <typename T, int NV, bool SLABS>
__global__ void __launch_bounds__(256) sm_post_norm_last_kernel(float* __restrict__ x, const void* __restrict__ o, int parts,
                                                                int width, const void* __restrict__ bias,
                                                                const void* __restrict__ wp, const void* __restrict__ wn,
                                                                void* __restrict__ h, float eps, float mult, float offset) {
  __shared__ float red[16];
  __shared__ __attribute__((aligned(16))) float row_s[NV * 1024];
  post_norm_row<T, 4, NV, SLABS, true>(red, x, o, parts, bias, wp, wn, h, width, eps, mult, offset, nullptr, 0.f, 0.f, row_s);
}

// The close of the last sublayer with the norm behind it, h in the bits of sm_rms_norm (widths of its row kernel).
bool sm_post_norm_last_fits(int width) { return width % 8 == 0 && width <= 8192; }

void sm_post_norm_last(uintptr_t x, uintptr_t o, int parts, uintptr_t bias, uintptr_t w_post, uintptr_t w_next, uintptr_t h, int rows,
                       int width, float eps, float mult, float offset, int f32, uintptr_t stream) {
  if (rows <= 0) return;
  DLLM_HOST_CHECK(x && o && w_post && w_next && h && width > 0 && sm_post_norm_last_fits(width), "post_norm_last arguments");
  DLLM_HOST_CHECK(parts >= 0 && (parts == 0 || !f32), "post_norm_last slabs");
  const auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(rows), dim3(256), 0, (hipStream_t)stream, (float*)x, (const void*)o, parts, width,
                       (const void*)bias, (const void*)w_post, (const void*)w_next, (void*)h, eps, mult, offset);
  };
#define SM_LAST(T, SLABS_)                                                    \
  do {                                                                        \
    if (width <= 1024) go(sm_post_norm_last_kernel<T, 1, SLABS_>);            \
    else if (width <= 2048) go(sm_post_norm_last_kernel<T, 2, SLABS_>);       \
    else if (width <= 3072) go(sm_post_norm_last_kernel<T, 3, SLABS_>);       \
    else if (width <= 4096) go(sm_post_norm_last_kernel<T, 4, SLABS_>);       \
    else go(sm_post_norm_last_kernel<T, 8, SLABS_>);                          \
  } while (0)
  if (f32) SM_LAST(float, false);
  else if (parts > 0) SM_LAST(bf16, true);
  else SM_LAST(bf16, false);
#undef SM_LAST
  DLLM_HIP_CHECK(hipGetLastError());
}

void sm_post_norm_add(uintptr_t x, uintptr_t o, int parts, uintptr_t bias, uintptr_t w_post, uintptr_t w_next, uintptr_t h,
                      int rows, int width, float eps, float mult, float offset, uintptr_t o2, float s1, float s2,
                      int f32, uintptr_t stream) {
  if (rows <= 0) return;
  DLLM_HOST_CHECK(width > 0 && (!w_next || h), "post_norm_add arguments");
  DLLM_HOST_CHECK(parts >= 0 && (parts == 0 || (!f32 && width % 4 == 0 && width <= 16384)), "post_norm_add slabs");
  if (width <= 16384) {
    if (parts > 0)
      SM_LN_SLABS(width, sm_post_norm_slabs_kernel, dim3(rows), stream, (float*)x, (const void*)o, parts,
                  (const void*)bias, (const void*)w_post, (const void*)w_next, (void*)h, width, eps, mult, offset,
                  (const void*)o2, s1, s2);
    else
      SM_LN_DISPATCH(f32, width, sm_post_norm_row_kernel, dim3(rows), stream, (float*)x, (const void*)o,
                     (const void*)bias, (const void*)w_post, (const void*)w_next, (void*)h, width, eps, mult, offset,
                     (const void*)o2, s1, s2);
    return;
  }
  SM_DISPATCH_V(f32, width % 8 == 0, sm_post_norm_add_kernel, dim3(rows), dim3(256), 0, stream, (float*)x,
                (const void*)o, (const void*)bias, (const void*)w_post, (const void*)w_next, (void*)h, width, eps, mult,
                offset, (const void*)o2, s1, s2);
}

// --------------------------------------------------------------------------- entry of a looped span
// x += x0 (a second float32 stream, when given) + vec (one row [width] of the activation type for every
// token, when given), in place.
template <typename T>
__global__ void __launch_bounds__(256) sm_stream_enter_kernel(float* __restrict__ x, const float* __restrict__ x0,
                                                              const void* __restrict__ vec_, long n, int width) {
  const T* vec = (const T*)vec_;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
    float v = x[i];
    if (x0) v += x0[i];
    if (vec) v += ldf(vec + (int)(i % width));
    x[i] = v;
  }
}

void sm_stream_enter(uintptr_t x, uintptr_t x0, uintptr_t vec, int rows, int width, int f32, uintptr_t stream) {
  if (rows <= 0) return;
  DLLM_HOST_CHECK(width > 0 && x, "stream_enter arguments");
  const long n = (long)rows * width;
  const unsigned grid = (unsigned)std::min<long>((n + 255) / 256, 65535);
  SM_DISPATCH(f32, sm_stream_enter_kernel, dim3(grid), dim3(256), 0, stream, (float*)x, (const float*)x0,
              (const void*)vec, n, width);
}

// --------------------------------------------------------------------------- close of a pre-norm sublayer
// x += coef * (f(o, w1) + f(o2, w2)) with f(o, w) = o / sqrt(mean(o^2) + eps) * w when w is given and o itself
// otherwise (o2 null: one term): two mixer outputs are normed apart, each with its own plain weight, before
// they are summed.  With wn: h = x / sqrt(mean(x^2) + eps) * wn, the next sublayer's input.
template <typename T, int V>
__global__ void __launch_bounds__(256) sm_mix_add_kernel(float* __restrict__ x, const void* __restrict__ o_,
                                                         const void* __restrict__ w1_, const void* __restrict__ o2_,
                                                         const void* __restrict__ w2_, const void* __restrict__ wn_,
                                                         void* __restrict__ h_, int width, float eps, float coef) {
  __shared__ float red[16];
  const T* o = (const T*)o_ + (size_t)blockIdx.x * width;
  const T* o2 = o2_ ? (const T*)o2_ + (size_t)blockIdx.x * width : nullptr;
  const T* w1 = (const T*)w1_;
  const T* w2 = (const T*)w2_;
  const T* wn = (const T*)wn_;
  float* xr = x + (size_t)blockIdx.x * width;
  float inv1 = 1.f, inv2 = 1.f;
  if (w1 || (o2 && w2)) {
    float s1 = 0.f, s2 = 0.f;
    for (int i = threadIdx.x * V; i < width; i += 256 * V) {
      float v[V];
      if (w1) {
        ldv<V>(o + i, v);
#pragma unroll
        for (int j = 0; j < V; ++j) s1 += v[j] * v[j];
      }
      if (o2 && w2) {
        ldv<V>(o2 + i, v);
#pragma unroll
        for (int j = 0; j < V; ++j) s2 += v[j] * v[j];
      }
    }
    if (w1) inv1 = 1.0f / sqrtf(block_sum(s1, red) / (float)width + eps);
    if (o2 && w2) inv2 = 1.0f / sqrtf(block_sum(s2, red) / (float)width + eps);
  }
  float sq = 0.f;
  for (int i = threadIdx.x * V; i < width; i += 256 * V) {
    float v[V], g[V], xv[V], y[V];
    ldv<V>(o + i, v);
    if (w1) {
      ldv<V>(w1 + i, g);
#pragma unroll
      for (int j = 0; j < V; ++j) v[j] = v[j] * inv1 * g[j];
    }
#pragma unroll
    for (int j = 0; j < V; ++j) y[j] = v[j];
    if (o2) {
      ldv<V>(o2 + i, v);
      if (w2) {
        ldv<V>(w2 + i, g);
#pragma unroll
        for (int j = 0; j < V; ++j) v[j] = v[j] * inv2 * g[j];
      }
#pragma unroll
      for (int j = 0; j < V; ++j) y[j] += v[j];
    }
    ldv<V>(xr + i, xv);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      xv[j] = xv[j] + coef * y[j];
      sq += xv[j] * xv[j];
    }
    stv<V>(xr + i, xv);
  }
  if (!wn) return;
  sq = block_sum(sq, red);
  const float invn = 1.0f / sqrtf(sq / (float)width + eps);
  T* h = (T*)h_ + (size_t)blockIdx.x * width;
  for (int i = threadIdx.x * V; i < width; i += 256 * V) {      // each lane re-reads what it wrote itself
    float xv[V], g[V];
    ldv<V>(xr + i, xv);
    ldv<V>(wn + i, g);
#pragma unroll
    for (int j = 0; j < V; ++j) xv[j] = xv[j] * invn * g[j];
    stv<V>(h + i, xv);
  }
}

void sm_mix_add(uintptr_t x, uintptr_t o, uintptr_t w1, uintptr_t o2, uintptr_t w2, uintptr_t w_next, uintptr_t h,
                int rows, int width, float eps, float coef, int f32, uintptr_t stream) {
  if (rows <= 0) return;
  DLLM_HOST_CHECK(width > 0 && x && o && (!w_next || h) && (!w2 || o2), "mix_add arguments");
  SM_DISPATCH_V(f32, width % 8 == 0, sm_mix_add_kernel, dim3(rows), dim3(256), 0, stream, (float*)x, (const void*)o,
                (const void*)w1, (const void*)o2, (const void*)w2, (const void*)w_next, (void*)h, width, eps, coef);
}

// --------------------------------------------------------------------------- token shift
// y_t = h_t + (h_(t-1) - h_t) * w per channel, h_(t-1) the UNBLENDED previous row of the same sequence: the
// batch row before it, for a chunk's first token the row the state slot keeps (zeros at position 0).  One
// workgroup per token; the workgroup of a chunk's FIRST token also brings the slot up to date -- it writes
// the chunk's last row there after it has read the old one, and nobody else touches that slot in the launch.
template <typename T, int V>
__global__ void __launch_bounds__(256) sm_token_shift_kernel(void* __restrict__ y_, const void* __restrict__ h_,
                                                             const void* __restrict__ w_, void* __restrict__ state_,
                                                             const int32_t* __restrict__ cu,
                                                             const int32_t* __restrict__ positions,
                                                             const int32_t* __restrict__ tok_seq,
                                                             const int32_t* __restrict__ slots, int width) {
  const int t = blockIdx.x, b = tok_seq[t];
  const int lo = cu[b], hi = cu[b + 1];
  const T* h = (const T*)h_ + (size_t)t * width;
  const T* w = (const T*)w_;
  T* y = (T*)y_ + (size_t)t * width;
  const bool first = t == lo;
  T* st = (T*)state_ + (size_t)slots[b] * width;
  const T* prev = first ? st : h - width;
  const bool zero = first && positions[t] == 0;
  const T* last = (const T*)h_ + (size_t)(hi - 1) * width;
  for (int i = threadIdx.x * V; i < width; i += 256 * V) {
    float c[V], p[V], g[V];
    ldv<V>(h + i, c);
    ldv<V>(w + i, g);
    if (zero) {
#pragma unroll
      for (int j = 0; j < V; ++j) p[j] = 0.f;
    } else {
      ldv<V>(prev + i, p);
    }
#pragma unroll
    for (int j = 0; j < V; ++j) c[j] = c[j] + (p[j] - c[j]) * g[j];
    stv<V>(y + i, c);
    if (first) {                                // same thread read st[i ..] just above
      ldv<V>(last + i, p);
      stv<V>(st + i, p);
    }
  }
}

void sm_token_shift(uintptr_t y, uintptr_t h, uintptr_t w, uintptr_t state, uintptr_t cu, uintptr_t positions,
                    uintptr_t tok_seq, uintptr_t slots, int tokens, int width, int f32, uintptr_t stream) {
  if (tokens <= 0) return;
  DLLM_HOST_CHECK(width > 0 && y && h && w && state && cu && positions && tok_seq && slots && y != h,
                  "token_shift arguments");
  const int esz = f32 ? 4 : 2;
  const bool vec = width % 8 == 0 && y % (8 * esz) == 0 && h % (8 * esz) == 0 && w % (8 * esz) == 0 && state % (8 * esz) == 0;
  SM_DISPATCH_V(f32, vec, sm_token_shift_kernel, dim3(tokens), dim3(256), 0, stream, (void*)y, (const void*)h,
                (const void*)w, (void*)state, (const int32_t*)cu, (const int32_t*)positions, (const int32_t*)tok_seq,
                (const int32_t*)slots, width);
}

// --------------------------------------------------------------------------- causal convolution with state
// (conv_input / conv_input_v, the reads of a token's earlier inputs, are in stream_common.h)
template <typename T, typename OT, int V, int TAPS>
__global__ void __launch_bounds__(256) sm_causal_conv_kernel(void* __restrict__ y_, const void* __restrict__ u_,
                                                             long stride, const void* __restrict__ w_,
                                                             const void* __restrict__ bias_,
                                                             const void* __restrict__ in_bias_,
                                                             const void* __restrict__ state_,
                                                             const int32_t* __restrict__ cu,
                                                             const int32_t* __restrict__ positions,
                                                             const int32_t* __restrict__ tok_seq,
                                                             const int32_t* __restrict__ slots, int C, int taps_,
                                                             int act) {
  const int taps = TAPS > 0 ? TAPS : taps_;
  const int t = blockIdx.x;
  const int b = tok_seq[t];
  const int tl = t - cu[b], pos = positions[t];
  const T* u = (const T*)u_;
  const T* w = (const T*)w_;
  const T* st = (const T*)state_ + (size_t)slots[b] * (taps - 1) * C;
  const T* bias = (const T*)bias_;
  const T* in_bias = (const T*)in_bias_;
  OT* y = (OT*)y_ + (size_t)t * C;
  for (int c = (blockIdx.y * 256 + threadIdx.x) * V; c < C; c += gridDim.y * 256 * V) {
    float acc[V], ib[V], xv[V], wv[V];
#pragma unroll
    for (int j = 0; j < V; ++j) acc[j] = 0.f, ib[j] = 0.f;
    if (bias) ldv<V>(bias + c, acc);
    if (in_bias) ldv<V>(in_bias + c, ib);
    if constexpr (TAPS > 0) {                        // every load at once, off a place that is always there
      float xs[TAPS][V], ws[TAPS][V];
#pragma unroll
      for (int j = 0; j < TAPS; ++j) {
        ldv<V>(conv_row(u, stride, st, t, tl, TAPS - 1 - j, TAPS, C) + c, xs[j]);
        ldv<V>(w + (size_t)j * C + c, ws[j]);
      }
#pragma unroll
      for (int j = 0; j < TAPS; ++j)
        if (TAPS - 1 - j <= pos) {                   // (uniform)
#pragma unroll
          for (int e = 0; e < V; ++e) acc[e] += ws[j][e] * (xs[j][e] + ib[e]);
        }
    } else {
      for (int j = 0; j < taps; ++j) {
        if (!conv_input_v<T, V>(u, stride, st, t, tl, pos, taps - 1 - j, taps, c, C, xv)) continue;
        ldv<V>(w + (size_t)j * C + c, wv);
#pragma unroll
        for (int e = 0; e < V; ++e) acc[e] += wv[e] * (xv[e] + ib[e]);
      }
    }
    if (act == 1) {                                  // silu, in float32 with the exact exponential
#pragma unroll
      for (int e = 0; e < V; ++e) acc[e] = acc[e] / (1.0f + expf(-acc[e]));
    }
    stv<V>(y + c, acc);
  }
}

// The same over many tokens, 3 or 4 taps: a thread takes 8 channels of kConvRun tokens, whose rows overlap (7 rows and one read of the
// weights for 4 tokens, 16 and 4 by themselves), all of them in one round trip where the run lies inside a sequence.
// us with the state's launch, bf16 to float32: rows one by one behind branches / all at once (above) / runs.  4 taps: 8000 tokens x 2560
// 46 / 41 / 31, 1000 x 5120 17.5 / 15.8 / 13.8, 4000 x 1024 15.6 / 13.9 / 12.8, but 1000 x 2560 11.4 / 10.6 / 10.2 (to bf16 9.9 / 9.1 /
// 10.2), 500 x 5120 10.5 / 9.9 / 10.2 (9.6 / 9.2 / 10.2), 2000 x 1024 8.8 / 8.5 / 9.0: runs from some 100000 threads on, three
// workgroups for two CUs.  3 taps 8000 x 5120 67 / 64 / 52.  2 taps share too little: 55 / 51 / 53, 1000 x 5120 to bf16 11.0 / 11.1 / 11.8.
constexpr int kConvRun = 4;
constexpr long kConvRunThreads = 256 * 384;

template <typename T, typename OT, int TAPS>
__global__ void __launch_bounds__(256) sm_causal_conv_run_kernel(
    void* __restrict__ y_, const void* __restrict__ u_, long stride, const void* __restrict__ w_, const void* __restrict__ bias_,
    const void* __restrict__ in_bias_, const void* __restrict__ state_, const int32_t* __restrict__ cu,
    const int32_t* __restrict__ positions, const int32_t* __restrict__ tok_seq, const int32_t* __restrict__ slots, int C, int act,
    int tokens) {
  const long id = (long)blockIdx.x * 256 + threadIdx.x;
  const int t0 = (int)(id / (C / 8)) * kConvRun, c = (int)(id % (C / 8)) * 8;
  if (t0 >= tokens) return;
  const T* u = (const T*)u_ + c;
  const T* w = (const T*)w_ + c;
  const int t1 = min(t0 + kConvRun, tokens) - 1, b0 = tok_seq[t0], b1 = tok_seq[t1], tl0 = t0 - cu[b0];
  float bias[8], ib[8], wv[TAPS][8];
#pragma unroll
  for (int e = 0; e < 8; ++e) bias[e] = ib[e] = 0.f;
  if (bias_) ldv<8>((const T*)bias_ + c, bias);
  if (in_bias_) ldv<8>((const T*)in_bias_ + c, ib);
#pragma unroll
  for (int j = 0; j < TAPS; ++j) ldv<8>(w + (size_t)j * C, wv[j]);
  auto finish = [&](int t, float (&acc)[8]) {
    if (act == 1) {                                  // silu, in float32 with the exact exponential
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = acc[e] / (1.0f + expf(-acc[e]));
    }
    stv<8>((OT*)y_ + (size_t)t * C + c, acc);
  };
  if (b0 == b1 && tl0 >= TAPS - 1) {
    float x[kConvRun + TAPS - 1][8];                 // row i: token t0 - (TAPS - 1) + i
#pragma unroll
    for (int i = 0; i < kConvRun + TAPS - 1; ++i) ldv<8>(u + (size_t)min(t0 - (TAPS - 1) + i, t1) * stride, x[i]);
#pragma unroll
    for (int q = 0; q < kConvRun; ++q) {
      if (t0 + q > t1) break;
      float acc[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = bias[e];
#pragma unroll
      for (int j = 0; j < TAPS; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += wv[j][e] * (x[q + j][e] + ib[e]);
      finish(t0 + q, acc);
    }
    return;
  }
  for (int t = t0; t <= t1; ++t) {
    const int b = tok_seq[t], tl = t - cu[b], pos = positions[t];
    const T* st = (const T*)state_ + (size_t)slots[b] * (TAPS - 1) * C + c;
    float acc[8], xs[TAPS][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = bias[e];
#pragma unroll
    for (int j = 0; j < TAPS; ++j) ldv<8>(conv_row(u, stride, st, t, tl, TAPS - 1 - j, TAPS, C), xs[j]);
#pragma unroll
    for (int j = 0; j < TAPS; ++j)
      if (TAPS - 1 - j <= pos) {
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += wv[j][e] * (xs[j][e] + ib[e]);
      }
    finish(t, acc);
  }
}

// New tail of every sequence: row j of the state becomes the input at position end - (taps - 1) + j
// (end = the chunk's last position + 1).  One thread per (sequence, V channels) walks j upwards: row j
// of the old tail is read (as row j + n, n the chunk's length) only before it is overwritten.
template <typename T, int V>
__global__ void __launch_bounds__(256) sm_conv_state_kernel(void* __restrict__ state_, const void* __restrict__ u_,
                                                            long stride, const int32_t* __restrict__ cu,
                                                            const int32_t* __restrict__ positions,
                                                            const int32_t* __restrict__ slots, int C, int taps) {
  const int b = blockIdx.x;
  const int lo = cu[b], n = cu[b + 1] - lo;
  if (n <= 0) return;
  const int start = positions[lo];
  T* st = (T*)state_ + (size_t)slots[b] * (taps - 1) * C;
  const T* u = (const T*)u_;
  for (int c = (blockIdx.y * 256 + threadIdx.x) * V; c < C; c += gridDim.y * 256 * V) {
    for (int j = 0; j < taps - 1; ++j) {
      const int tl = n - (taps - 1) + j;              // local index of the row that lands in tail row j
      float v[V];
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] = 0.f;
      if (tl >= 0) ldv<V>(u + (size_t)(lo + tl) * stride + c, v);
      else if (start + tl >= 0) ldv<V>(st + (size_t)(j + n) * C + c, v);
      stv<V>(st + (size_t)j * C + c, v);
    }
  }
}

static void launch_conv_state(uintptr_t state, uintptr_t u, long stride, uintptr_t cu, uintptr_t positions,
                              uintptr_t slots, int seqs, int C, int taps, int f32, int vec, uintptr_t stream) {
  const int per = 256 * (vec ? 8 : 1);
  SM_DISPATCH_V(f32, vec, sm_conv_state_kernel, dim3(seqs, std::min(8, (C + per - 1) / per)), dim3(256), 0, stream,
                (void*)state, (const void*)u, stride, (const int32_t*)cu, (const int32_t*)positions,
                (const int32_t*)slots, C, taps);
}

// The tail update alone (a caller that ran the convolution in a kernel of its own).
void sm_conv_tail(uintptr_t state, uintptr_t u, long stride, uintptr_t cu, uintptr_t positions, uintptr_t slots, int seqs,
                  int C, int taps, int f32, uintptr_t stream) {
  if (seqs <= 0 || taps <= 1) return;
  DLLM_HOST_CHECK(C > 0 && stride >= C, "conv sizes");
  const int esz = f32 ? 4 : 2;
  launch_conv_state(state, u, stride, cu, positions, slots, seqs, C, taps, f32,
                    C % 8 == 0 && stride % 8 == 0 && (u % (8 * esz)) == 0, stream);
}

void sm_causal_conv(uintptr_t y, uintptr_t u, long stride, uintptr_t w, uintptr_t bias, uintptr_t in_bias,
                    uintptr_t state, uintptr_t cu, uintptr_t positions, uintptr_t tok_seq, uintptr_t slots,
                    int tokens, int seqs, int C, int taps, int f32, int out_f32, int act, uintptr_t stream) {
  if (tokens <= 0 || seqs <= 0) return;
  DLLM_HOST_CHECK(C > 0 && taps >= 1 && stride >= C && (act == 0 || act == 1), "conv sizes");
  const int esz = f32 ? 4 : 2;
  const int vec = C % 8 == 0 && stride % 8 == 0 && (u % (8 * esz)) == 0;
  const int per = 256 * (vec ? 8 : 1);
  const dim3 grid(tokens, std::min(8, (C + per - 1) / per));
  hipStream_t s = (hipStream_t)stream;
#define SM_CONV_N(T, OT, V, N)                                                                                         \
  hipLaunchKernelGGL(HIP_KERNEL_NAME(sm_causal_conv_kernel<T, OT, V, N>), grid, dim3(256), 0, s, (void*)y, (const void*)u, \
                     stride, (const void*)w, (const void*)bias, (const void*)in_bias, (const void*)state,     \
                     (const int32_t*)cu, (const int32_t*)positions, (const int32_t*)tok_seq, (const int32_t*)slots, C, taps, act)
#define SM_CONV_RUN(T, OT, N)                                                                                        \
  hipLaunchKernelGGL(HIP_KERNEL_NAME(sm_causal_conv_run_kernel<T, OT, N>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, \
                     (void*)y, (const void*)u, stride, (const void*)w, (const void*)bias, (const void*)in_bias,              \
                     (const void*)state, (const int32_t*)cu, (const int32_t*)positions, (const int32_t*)tok_seq,             \
                     (const int32_t*)slots, C, act, tokens)
#define SM_CONV_T(T, OT, N)                                                                                            \
  do {                                                                                                                 \
    if (N > 2 && runs) SM_CONV_RUN(T, OT, (N > 2 ? N : 3));                                                            \
    else if (vec) SM_CONV_N(T, OT, 8, N);                                                                              \
    else SM_CONV_N(T, OT, 1, N);                                                                                       \
  } while (0)
#define SM_CONV(T, OT)                                                                                                 \
  do {                                                                                                                 \
    if (taps == 2) SM_CONV_T(T, OT, 2);                                                                                \
    else if (taps == 3) SM_CONV_T(T, OT, 3);                                                                           \
    else if (taps == 4) SM_CONV_T(T, OT, 4);                                                                           \
    else if (vec) SM_CONV_N(T, OT, 8, 0);                                                                              \
    else SM_CONV_N(T, OT, 1, 0);                                                                                       \
  } while (0)
  const long threads = (long)((tokens + kConvRun - 1) / kConvRun) * (C / 8);
  const bool runs = vec && threads >= kConvRunThreads;
  if (f32) SM_CONV(float, float);
  else if (out_f32) SM_CONV(bf16, float);
  else SM_CONV(bf16, bf16);
#undef SM_CONV_RUN
#undef SM_CONV_N
#undef SM_CONV_T
#undef SM_CONV
  DLLM_HIP_CHECK(hipGetLastError());
  if (taps > 1) launch_conv_state(state, u, stride, cu, positions, slots, seqs, C, taps, f32, vec, stream);
}

// --------------------------------------------------------------------------- RG-LRU gates
// a = exp(-scale * sigmoid(Ra_b u_b + ra_b) * softplus(lam)),  g = sqrt(1 - a^2) * sigmoid(Ri_b u_b + ri_b) * u,
// with the transposed gate matrices [nb, in, out] (consecutive lanes on consecutive outputs).
__device__ __forceinline__ float sigmoid_f(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float softplus_f(float x) { return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x))); }

// Few tokens (decode): GT tokens x one block of bw channels per workgroup on the vector ALUs; the
// token tile's u_b sits in LDS, every weight is read once per workgroup.
constexpr int GT = 4;

template <typename T>
__global__ void __launch_bounds__(256) sm_rglru_gates_small_kernel(float* __restrict__ a_out, float* __restrict__ g_out,
                                                                   const float* __restrict__ u,
                                                                   const void* __restrict__ ra_t_,
                                                                   const void* __restrict__ ra_b_,
                                                                   const void* __restrict__ ri_t_,
                                                                   const void* __restrict__ ri_b_,
                                                                   const void* __restrict__ lam_, int tokens, int nb,
                                                                   int bw, float scale) {
  extern __shared__ float ubs[];                      // [GT][bw]
  const int t0 = blockIdx.x * GT, b = blockIdx.y, C = nb * bw;
  const int nt = min(GT, tokens - t0);
  for (int i = threadIdx.x; i < GT * bw; i += 256) {
    const int k = i / bw, c = i - k * bw;
    ubs[i] = k < nt ? u[(size_t)(t0 + k) * C + b * bw + c] : 0.f;
  }
  __syncthreads();
  const T* ra = (const T*)ra_t_ + (size_t)b * bw * bw;
  const T* ri = (const T*)ri_t_ + (size_t)b * bw * bw;
  for (int o = threadIdx.x; o < bw; o += 256) {
    float ar[GT], ai[GT];
    const float br = ldf((const T*)ra_b_ + b * bw + o), bi = ldf((const T*)ri_b_ + b * bw + o);
#pragma unroll
    for (int k = 0; k < GT; ++k) ar[k] = br, ai[k] = bi;
    int i = 0;
    for (; i + 8 <= bw; i += 8) {                      // 16 weight loads in flight, then their FMAs
      float wr[8], wi[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) wr[j] = ldf(ra + (size_t)(i + j) * bw + o), wi[j] = ldf(ri + (size_t)(i + j) * bw + o);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
#pragma unroll
        for (int k = 0; k < GT; ++k) {
          const float x = ubs[k * bw + i + j];
          ar[k] = fmaf(wr[j], x, ar[k]);
          ai[k] = fmaf(wi[j], x, ai[k]);
        }
      }
    }
    for (; i < bw; ++i) {
      const float wr = ldf(ra + (size_t)i * bw + o), wi = ldf(ri + (size_t)i * bw + o);
#pragma unroll
      for (int k = 0; k < GT; ++k) {
        const float x = ubs[k * bw + i];
        ar[k] = fmaf(wr, x, ar[k]);
        ai[k] = fmaf(wi, x, ai[k]);
      }
    }
    const float sp = softplus_f(ldf((const T*)lam_ + b * bw + o));
#pragma unroll
    for (int k = 0; k < GT; ++k) {
      if (k < nt) {
        const float av = expf(-scale * sigmoid_f(ar[k]) * sp);
        const size_t idx = (size_t)(t0 + k) * C + b * bw + o;
        a_out[idx] = av;
        g_out[idx] = sqrtf(1.0f - av * av) * sigmoid_f(ai[k]) * ubs[k * bw + o];
      }
    }
  }
}

// The same for blocks whose width is a multiple of 8: a lane loads 8 consecutive outputs of one input
// row (16 bytes of bf16) and the workgroup's 8 lane groups take every 8th input row; their partial
// sums meet in LDS.  256 outputs of block b per workgroup.
template <typename T>
__global__ void __launch_bounds__(256) sm_rglru_gates_small_vec_kernel(
    float* __restrict__ a_out, float* __restrict__ g_out, const float* __restrict__ u, const void* __restrict__ ra_t_,
    const void* __restrict__ ra_b_, const void* __restrict__ ri_t_, const void* __restrict__ ri_b_,
    const void* __restrict__ lam_, int tokens, int nb, int bw, float scale) {
  extern __shared__ float smem[];
  float* ubs = smem;                                  // [GT][bw]
  float* red = smem + GT * bw;                        // [8 groups][GT][256]
  const int t0 = blockIdx.x * GT, b = blockIdx.y, C = nb * bw, o0 = blockIdx.z * 256;
  const int nt = min(GT, tokens - t0);
  const int tid = threadIdx.x, og = tid & 31, kg = tid >> 5;
  for (int i = tid; i < GT * bw; i += 256) {
    const int k = i / bw, c = i - k * bw;
    ubs[i] = k < nt ? u[(size_t)(t0 + k) * C + b * bw + c] : 0.f;
  }
  __syncthreads();
  const T* ra = (const T*)ra_t_ + (size_t)b * bw * bw;
  const T* ri = (const T*)ri_t_ + (size_t)b * bw * bw;
  const int ob = o0 + 8 * og;                         // this lane's 8 outputs
  float ar[GT][8], ai[GT][8];
#pragma unroll
  for (int k = 0; k < GT; ++k)
#pragma unroll
    for (int j = 0; j < 8; ++j) ar[k][j] = 0.f, ai[k][j] = 0.f;
  if (ob < bw) {
    for (int i = kg; i < bw; i += 8) {
      float wr[8], wi[8];
      ldv<8>(ra + (size_t)i * bw + ob, wr);
      ldv<8>(ri + (size_t)i * bw + ob, wi);
#pragma unroll
      for (int k = 0; k < GT; ++k) {
        const float x = ubs[k * bw + i];
#pragma unroll
        for (int j = 0; j < 8; ++j) ar[k][j] = fmaf(wr[j], x, ar[k][j]), ai[k][j] = fmaf(wi[j], x, ai[k][j]);
      }
    }
  }
  // the 8 lane groups' partial sums meet in LDS, one gate after the other (the same 32 KiB)
  float sr[GT], si[GT];
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    __syncthreads();
#pragma unroll
    for (int k = 0; k < GT; ++k)
#pragma unroll
      for (int j = 0; j < 8; ++j) red[(kg * GT + k) * 256 + 8 * og + j] = pass ? ai[k][j] : ar[k][j];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < GT; ++k) {                    // this thread finishes (token k, output o0 + tid)
      float sum = 0.f;
#pragma unroll
      for (int g8 = 0; g8 < 8; ++g8) sum += red[(g8 * GT + k) * 256 + tid];
      if (pass) si[k] = sum; else sr[k] = sum;
    }
  }
  const int o = o0 + tid;
  if (o >= bw) return;
  const int ch = b * bw + o;
  const float sp = softplus_f(ldf((const T*)lam_ + ch));
  const float rb = ldf((const T*)ra_b_ + ch), ib = ldf((const T*)ri_b_ + ch);
#pragma unroll
  for (int k = 0; k < GT; ++k) {
    if (k < nt) {
      const float av = expf(-scale * sigmoid_f(sr[k] + rb) * sp);
      const size_t at = (size_t)(t0 + k) * C + ch;
      a_out[at] = av;
      g_out[at] = sqrtf(1.0f - av * av) * sigmoid_f(si[k] + ib) * ubs[k * bw + o];
    }
  }
}

// Many tokens (prompts), float32: the two block-diagonal products on the float32 matrix cores
// (v_mfma_f32_32x32x2_f32: true 32-bit operands and sums, which the gates of the recurrence require).
// One workgroup per (64 tokens, block b, 128 outputs of the block): each wave owns 32 outputs and, for
// both gates, two 32 x 32 accumulators (token rows 0-31 and 32-63).  The token tile's u_b passes through
// LDS in K chunks of kGK (A operand: lane l = row l % 32, k l / 32); the gate matrices are the B operand
// from global memory, kGU k-steps of loads issued ahead of the MFMAs that use them.
constexpr int kGT = 64;       // tokens per workgroup
constexpr int kGK = 128;      // K chunk in LDS
constexpr int kGU = 8;        // k-steps (of 2) per group of loads

__global__ void __launch_bounds__(256) sm_rglru_gates_kernel(float* __restrict__ a_out, float* __restrict__ g_out,
                                                             const float* __restrict__ u,
                                                             const float* __restrict__ ra_t,
                                                             const float* __restrict__ ra_b,
                                                             const float* __restrict__ ri_t,
                                                             const float* __restrict__ ri_b,
                                                             const float* __restrict__ lam, int tokens, int nb, int bw,
                                                             float scale) {
  __shared__ float ub[kGT][kGK + 1];
  const int t0 = blockIdx.x * kGT, b = blockIdx.y, C = nb * bw;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = lane & 31, half = lane >> 5;
  const int o = blockIdx.z * 128 + wave * 32 + n;            // this lane's output channel inside block b
  const int oc = min(o, bw - 1);
  const float* ra = ra_t + (size_t)b * bw * bw;
  const float* ri = ri_t + (size_t)b * bw * bw;
  f32x16 cr0, ci0, cr1, ci1;
#pragma unroll
  for (int i = 0; i < 16; ++i) cr0[i] = ci0[i] = cr1[i] = ci1[i] = 0.f;
  for (int kc = 0; kc < bw; kc += kGK) {
    const int kn = min(kGK, bw - kc);
    __syncthreads();
    for (int i = tid; i < kGT * kGK; i += 256) {
      const int r = i / kGK, k = i - r * kGK;
      ub[r][k] = (t0 + r < tokens && k < kn) ? u[(size_t)(t0 + r) * C + b * bw + kc + k] : 0.f;
    }
    __syncthreads();
    // groups of kGU k-steps: the next group's weights and u values are loaded before the current
    // group's 4 kGU MFMAs issue, so their latency hides behind 64-cycle matrix instructions
    float br[2][kGU], bi[2][kGU], a0[2][kGU], a1[2][kGU];
    auto load_group = [&](int ks0, int buf) {
#pragma unroll
      for (int j = 0; j < kGU; ++j) {
        const int k = 2 * (ks0 + j) + half;                  // inside the chunk
        const bool ok = k < kn && o < bw;
        const size_t at = (size_t)(kc + min(k, kn - 1)) * bw + oc;
        const float wr = ra[at], wi = ri[at];
        br[buf][j] = ok ? wr : 0.f;
        bi[buf][j] = ok ? wi : 0.f;
        const int kk = min(k, kGK - 1);
        a0[buf][j] = k < kn ? ub[n][kk] : 0.f;
        a1[buf][j] = k < kn ? ub[32 + n][kk] : 0.f;
      }
    };
    auto mma_group = [&](int buf) {
#pragma unroll
      for (int j = 0; j < kGU; ++j) {
        cr0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[buf][j], br[buf][j], cr0, 0, 0, 0);
        ci0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[buf][j], bi[buf][j], ci0, 0, 0, 0);
        cr1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[buf][j], br[buf][j], cr1, 0, 0, 0);
        ci1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[buf][j], bi[buf][j], ci1, 0, 0, 0);
      }
    };
    load_group(0, 0);
    for (int ks0 = 0; 2 * ks0 < kn; ks0 += 2 * kGU) {
      const bool more1 = 2 * (ks0 + kGU) < kn, more2 = 2 * (ks0 + 2 * kGU) < kn;
      if (more1) load_group(ks0 + kGU, 1);
      mma_group(0);
      if (more1) {
        if (more2) load_group(ks0 + 2 * kGU, 0);
        mma_group(1);
      }
    }
  }
  if (o >= bw) return;
  const int ch = b * bw + o;
  const float rb = ra_b[ch], ib = ri_b[ch];
  const float sp = softplus_f(lam[ch]);
#pragma unroll
  for (int hh = 0; hh < 2; ++hh) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = 32 * hh + 8 * (i >> 2) + 4 * half + (i & 3);    // accumulator register i of this lane
      const int t = t0 + row;
      if (t < tokens) {
        const float av = expf(-scale * sigmoid_f((hh ? cr1[i] : cr0[i]) + rb) * sp);
        const size_t idx = (size_t)t * C + ch;
        a_out[idx] = av;
        g_out[idx] = sqrtf(1.0f - av * av) * sigmoid_f((hh ? ci1[i] : ci0[i]) + ib) * u[idx];
      }
    }
  }
}

// The same products for bf16 gate matrices on the bf16 matrix cores, as exact as on the float32 ones: u = h + m + l in three
// bf16 pieces (8 significant bits each, 24 in all: nothing of u is lost), each times the bf16 weight an exact product, the
// sums in float32.  Three products at 16 times the rate: 20 us of them, beside which the vector work (taking u apart, putting
// the weights' columns together, the gates' functions) bounds it.  One workgroup per (64 tokens, block b, 256 outputs): two waves by
// tokens, two by outputs, and of a wave's 128 outputs lane n owns 4 n .. 4 n + 3, one in each of four products: u is taken apart once
// per block, the weights come in 8-byte loads a k-step of 16 ahead (8 rows of them make four fragments in 16 v_perm), u, a and g
// in 16-byte ones.  The pieces of u pass through LDS in K chunks of kSK, two of them (rows kSP apart: the 16 byte reads of 8
// rows fall on banks of their own); two workgroups share a CU, one's vector work under the other's products.
// The gates' functions are those of the other kernels (sigmoid_f, sqrtf): a and g have the same bits whichever kernel the alignment
// and the rule below choose.  (Quotient and root off the hardware's approximations and a Newton step each: 83 us for 94, but 1 % of
// a and 2 % of g another last bit.  With a second step and the remainder all bits were there, in 93 us.)
// us, 10 blocks of 256, 6376 / 3000 / 300 tokens: 126 / 64 / 40 with an output per lane (weights two bytes at a time) and u taken apart
// for 128 outputs, 94 / 50 / 27 here (275 on the float32 matrix cores at 6376); 4 blocks, 2000 / 168: 42 / 39 -> 28 / 26.  Largest
// error of a and g against 64 bits there 5.4e-7 and 8.1e-6, means 1.8e-8 and 2.8e-8, as before.
// Blocks a multiple of 4 wide, 16-byte aligned.
constexpr int kST = 64;       // tokens per workgroup
constexpr int kSO = 256;      // outputs
constexpr int kSK = 64;       // K chunk in LDS
constexpr int kSP = kSK + 8;
constexpr float kBfMax = 0x1.fep+127f;

__global__ void __launch_bounds__(256, 2) sm_rglru_gates_split_kernel(
    float* __restrict__ a_out, float* __restrict__ g_out, const float* __restrict__ u, const bf16* __restrict__ ra_t,
    const bf16* __restrict__ ra_b, const bf16* __restrict__ ri_t, const bf16* __restrict__ ri_b,
    const bf16* __restrict__ lam, int tokens, int nb, int bw, float scale) {
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  __shared__ __attribute__((aligned(16))) bf16 us[2][3][kST][kSP];
  const int t0 = blockIdx.x * kST, b = blockIdx.y, C = nb * bw;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = lane & 31, half = lane >> 5;
  const int wm = wave >> 1, wn = wave & 1;
  const int o = blockIdx.z * kSO + wn * 128 + 4 * n;         // this lane's four output channels inside block b
  const size_t blk = (size_t)b * bw * bw;
  // rows of u, a and g through buffers of this workgroup's tokens: nothing is read or written past the last one
  const size_t row0 = (size_t)t0 * C;
  const int bytes = min(kST, tokens - t0) * C * 4;
  const auto ru = __builtin_amdgcn_make_buffer_rsrc((void*)(u + row0), (short)0, bytes, 0x00020000);
  const auto rsa = __builtin_amdgcn_make_buffer_rsrc((void*)(a_out + row0), (short)0, bytes, 0x00020000);
  const auto rsg = __builtin_amdgcn_make_buffer_rsrc((void*)(g_out + row0), (short)0, bytes, 0x00020000);
  auto row4 = [&](int r, int k) -> f32x4 {                   // channels k .. k + 3 of the block in the workgroup's row r
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ru, (r * C + b * bw + k) * 4, 0, 0));
  };

  // a chunk's values of this thread: four of row (tid >> 4) + 16 q each, zero past the block
  f32x4 x[4];
  auto load_u = [&](int kc) {
    const int k = kc + 4 * (tid & 15);
#pragma unroll
    for (int q = 0; q < 4; ++q) x[q] = row4((tid >> 4) + 16 * q, k);
    if (kc + kSK > bw) {                                     // uniform
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[q][e] = k + e < bw ? x[q][e] : 0.f;
    }
  };
  auto store_u = [&](int buf) {
    uint32_t top = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = x[q][e];                             // (the cast of a vector's element takes its first)
        top = max(top, __builtin_bit_cast(uint32_t, v) & 0x7fffffffu);
      }
    const bool plain = top <= __builtin_bit_cast(uint32_t, kBfMax);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      bf16x4 h, m, l;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = x[q][e];
        h[e] = f2bf(v);
        const float vm = v - bf2f(h[e]);
        m[e] = f2bf(vm);
        l[e] = f2bf(vm - bf2f(m[e]));
      }
      if (!plain) {      // (a finite value above the largest bf16 keeps a finite first piece; an infinite or NaN one has no others)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = x[q][e];
          const bool fin = __builtin_isfinite(v);
          h[e] = f2bf(fin ? fminf(fmaxf(v, -kBfMax), kBfMax) : v);
          const float vm = fin ? v - bf2f(h[e]) : 0.f;
          m[e] = f2bf(vm);
          l[e] = f2bf(vm - bf2f(m[e]));
        }
      }
      const int r = (tid >> 4) + 16 * q, k = 4 * (tid & 15);
      *reinterpret_cast<bf16x4*>(&us[buf][0][r][k]) = h;
      *reinterpret_cast<bf16x4*>(&us[buf][1][r][k]) = m;
      *reinterpret_cast<bf16x4*>(&us[buf][2][r][k]) = l;
    }
  };
  // rows k0 + 8 half .. of this lane's columns of a gate matrix (zero past the block), and the four fragments they make
  const auto rr = __builtin_amdgcn_make_buffer_rsrc((void*)(ra_t + blk), (short)0, bw * bw * 2, 0x00020000);
  const auto ri = __builtin_amdgcn_make_buffer_rsrc((void*)(ri_t + blk), (short)0, bw * bw * 2, 0x00020000);
  const int lane_w = (8 * half * bw + o) * 2;
  auto load_w = [&](u32x2 (&w)[8], const __amdgpu_buffer_rsrc_t& g, int k0) {
#pragma unroll
    for (int q = 0; q < 8; ++q)
      w[q] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(g, lane_w + (k0 + q) * bw * 2, 0, 0));
  };
  auto fragments = [&](bf16x8 (&f)[4], const u32x2 (&w)[8]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      u32x4 v;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        v[q] = __builtin_amdgcn_perm(w[2 * q + 1][j >> 1], w[2 * q][j >> 1], j & 1 ? 0x07060302u : 0x05040100u);
      f[j] = __builtin_bit_cast(bf16x8, v);
    }
  };

  f32x16 cr[4], ci[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i) cr[j][i] = ci[j][i] = 0.f;
  u32x2 wr[8], wi[8];
  load_u(0);
  load_w(wr, rr, 0);
  load_w(wi, ri, 0);
  store_u(0);
  int buf = 0;
  for (int kc = 0; kc < bw; kc += kSK, buf ^= 1) {
    __syncthreads();                                         // chunk kc is there; the other buffer's readers are through
    const bool more = kc + kSK < bw;                         // uniform
    if (more) load_u(kc + kSK);
#pragma unroll
    for (int s = 0; s < kSK / 16; ++s) {
      const int k0 = kc + 16 * s;
      if (k0 < bw) {                                         // uniform
        bf16x8 a[3], f[4];
#pragma unroll
        for (int p = 0; p < 3; ++p) a[p] = *reinterpret_cast<const bf16x8*>(&us[buf][p][32 * wm + n][16 * s + 8 * half]);
        fragments(f, wr);
        load_w(wr, rr, k0 + 16);                             // (past the last step: zeros, not used)
        __builtin_amdgcn_sched_barrier(0);                   // (hipcc moves these loads behind the products)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int p = 2; p >= 0; --p)                       // the small pieces first
            cr[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[p], f[j], cr[j], 0, 0, 0);
        fragments(f, wi);
        load_w(wi, ri, k0 + 16);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int p = 2; p >= 0; --p) ci[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[p], f[j], ci[j], 0, 0, 0);
      }
    }
    if (more) store_u(buf ^ 1);
  }
  if (o >= bw) return;
  f32x4 ux[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) ux[i] = row4(32 * wm + 4 * half + i, o);
  float rb[4], ib[4], sp[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int ch = b * bw + min(o + j, bw - 1);
    rb[j] = bf2f(ra_b[ch]), ib[j] = bf2f(ri_b[ch]), sp[j] = softplus_f(bf2f(lam[ch]));
  }
#pragma unroll 1
  for (int i0 = 0; i0 < 16; i0 += 4) {                       // accumulator register i of this lane: row 8 (i / 4) + 4 half + i % 4
    const int r = 32 * wm + 2 * i0 + 4 * half;
    f32x4 un[4];                                             // the next four rows' u
#pragma unroll
    for (int i = 0; i < 4; ++i) un[i] = row4(min(r + 8, kST - 4) + i, o);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f32x4 av, gv;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        av[j] = expf(-scale * sigmoid_f(cr[j][i] + rb[j]) * sp[j]);
        gv[j] = sqrtf(1.0f - av[j] * av[j]) * sigmoid_f(ci[j][i] + ib[j]) * ux[i][j];
      }
      const int at = ((r + i) * C + b * bw + o) * 4;
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, av), rsa, at, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, gv), rsg, at, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      ux[j] = un[j];
#pragma unroll
      for (int i = 0; i < 12; ++i) cr[j][i] = cr[j][i + 4], ci[j][i] = ci[j][i + 4];
    }
  }
}

// The same sums with an output per lane and 32 per wave, 128 tokens by 128 outputs per workgroup, u and the weights element by
// element: any width and alignment, and no lane idle from blocks of 128 on.  Bound by its vector work and by two-byte loads.
// Which kernel, us, this / the one above: widths that are no multiple of 4 this (8 blocks of 255, 300 / 16000 tokens 40 / 257
// against 59 / 503 element by element there); 8 blocks of 64, 128, 256: 2000 tokens 27 / 20, 31 / 23, 47 / 30; 4500 tokens 34 / 38,
// 43 / 47, 94 / 66; 8000 36 / 47, 49 / 58, 115 / 86: blocks up to 128 leave half of the other's waves idle, which counts once the CUs
// hold two workgroups each; 3 blocks of 24, 300 / 16000 tokens: 23 / 34, 27 / 52.
constexpr int kCT = 128;      // tokens per workgroup

// (The arguments come in one piece, which is loaded.  Preloaded into the waves' registers as the other kernels' are, they cost it 2 % at
// few tokens, 8 blocks of 255 at 300 / 1000 / 8000 us 39.9 / 42.8 / 118 -> 40.5 / 43.3 / 118, 8 blocks of 129 at 500 33.0 -> 33.4.)
struct GateArgs {
  float *a, *g;
  const float* u;
  const bf16 *ra_t, *ra_b, *ri_t, *ri_b, *lam;
  int tokens, nb, bw;
  float scale;
};
__global__ void __launch_bounds__(256, 2) sm_rglru_gates_column_kernel(const GateArgs p) {
  float *__restrict__ a_out = p.a, *__restrict__ g_out = p.g;
  const float* __restrict__ u = p.u;
  const bf16 *__restrict__ ra_t = p.ra_t, *__restrict__ ri_t = p.ri_t;
  const bf16 *ra_b = p.ra_b, *ri_b = p.ri_b, *lam = p.lam;
  const int tokens = p.tokens, nb = p.nb, bw = p.bw;
  const float scale = p.scale;
  __shared__ __attribute__((aligned(16))) bf16 us[3][kCT][kSP];
  const int t0 = blockIdx.x * kCT, b = blockIdx.y, C = nb * bw;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = lane & 31, half = lane >> 5;
  const int o = blockIdx.z * 128 + wave * 32 + n;            // this lane's output channel inside block b
  const int oc = min(o, bw - 1);
  const bf16* ra = ra_t + (size_t)b * bw * bw + oc;
  const bf16* ri = ri_t + (size_t)b * bw * bw + oc;
  f32x16 cr[4], ci[4];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int i = 0; i < 16; ++i) cr[m][i] = ci[m][i] = 0.f;
  bf16x8 wr[2], wi[2];
  auto load_w = [&](int k0, int buf) {                       // rows k0 + 8 half .. of this lane's output column
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const size_t at = (size_t)min(k0 + 8 * half + j, bw - 1) * bw;
      wr[buf][j] = ra[at];
      wi[buf][j] = ri[at];
    }
  };
  load_w(0, 0);
  const float* ub = u + (size_t)b * bw;
  for (int kc = 0; kc < bw; kc += kSK) {
    __syncthreads();
#pragma unroll 8
    for (int i = tid; i < kCT * kSK; i += 256) {             // a wave per row of the chunk
      const int r = i / kSK, k = i - r * kSK;
      const bool ok = t0 + r < tokens && kc + k < bw;
      float x = ub[(size_t)min(t0 + r, tokens - 1) * C + min(kc + k, bw - 1)];
      x = ok ? x : 0.f;
      // (a finite x above the largest bf16 keeps a finite first piece; an infinite or NaN one has no others)
      const bool fin = __builtin_isfinite(x);
      const bf16 h = f2bf(fin ? fminf(fmaxf(x, -kBfMax), kBfMax) : x);
      const float xm = fin ? x - bf2f(h) : 0.f;
      const bf16 m = f2bf(xm);
      us[0][r][k] = h;
      us[1][r][k] = m;
      us[2][r][k] = f2bf(xm - bf2f(m));
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < kSK / 16; ++s) {
      if (kc + 16 * s < bw) {                                // uniform
        load_w(kc + 16 * (s + 1), (s + 1) & 1);              // (past the last step: the last row, not used)
        bf16x8 br = wr[s & 1], bi = wi[s & 1];
        if (kc + 16 * (s + 1) > bw) {                        // uniform: rows past the block
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (kc + 16 * s + 8 * half + j >= bw) br[j] = bi[j] = (bf16)0.f;
        }
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
          for (int p = 2; p >= 0; --p) {                     // the small pieces first
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(&us[p][32 * m + n][16 * s + 8 * half]);
            cr[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, br, cr[m], 0, 0, 0);
            ci[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, bi, ci[m], 0, 0, 0);
          }
      }
    }
  }
  if (o >= bw) return;
  const int ch = b * bw + o;
  const float rb = bf2f(ra_b[ch]), ib = bf2f(ri_b[ch]), sp = softplus_f(bf2f(lam[ch]));
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i)
      x[i] = u[(size_t)min(t0 + 32 * m + 8 * (i >> 2) + 4 * half + (i & 3), tokens - 1) * C + ch];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int t = t0 + 32 * m + 8 * (i >> 2) + 4 * half + (i & 3);    // accumulator register i of this lane
      const float av = expf(-scale * sigmoid_f(cr[m][i] + rb) * sp);
      const float gv = sqrtf(1.0f - av * av) * sigmoid_f(ci[m][i] + ib) * x[i];
      if (t < tokens) {
        a_out[(size_t)t * C + ch] = av;
        g_out[(size_t)t * C + ch] = gv;
      }
    }
  }
}

void sm_rglru_gates(uintptr_t a, uintptr_t g, uintptr_t u, uintptr_t ra_t, uintptr_t ra_b, uintptr_t ri_t,
                    uintptr_t ri_b, uintptr_t lam, int tokens, int nb, int bw, float scale, int f32,
                    uintptr_t stream) {
  if (tokens <= 0) return;
  DLLM_HOST_CHECK(nb > 0 && bw > 0 && nb <= 65535 && (bw + 127) / 128 <= 65535, "rglru gate sizes");
  const size_t lds = (size_t)GT * bw * sizeof(float);
  const size_t lds_vec = lds + (size_t)8 * GT * 256 * sizeof(float);
  if (tokens <= 64 && bw % 8 == 0 && lds_vec <= 64 * 1024) {
    SM_DISPATCH(f32, sm_rglru_gates_small_vec_kernel, dim3((tokens + GT - 1) / GT, nb, (bw + 255) / 256), dim3(256),
                lds_vec, stream, (float*)a, (float*)g, (const float*)u, (const void*)ra_t, (const void*)ra_b,
                (const void*)ri_t, (const void*)ri_b, (const void*)lam, tokens, nb, bw, scale);
    return;
  }
  if (tokens <= 64 && lds <= 48 * 1024) {
    SM_DISPATCH(f32, sm_rglru_gates_small_kernel, dim3((tokens + GT - 1) / GT, nb), dim3(256), lds, stream, (float*)a,
                (float*)g, (const float*)u, (const void*)ra_t, (const void*)ra_b, (const void*)ri_t,
                (const void*)ri_b, (const void*)lam, tokens, nb, bw, scale);
    return;
  }
  if (!f32) {
    const dim3 grid((tokens + kST - 1) / kST, nb, (bw + kSO - 1) / kSO), cols((tokens + kCT - 1) / kCT, nb, (bw + 127) / 128);
    const bool vec = bw % 4 == 0 && (u | a | g) % 16 == 0 && (ra_t | ri_t) % 8 == 0;
    const bool split = vec && bw >= 48 && (bw > 128 || (size_t)grid.x * nb <= 512);
#define SM_GATES(KERNEL_, GRID_)                                                                                           \
  hipLaunchKernelGGL(KERNEL_, GRID_, dim3(256), 0, (hipStream_t)stream, (float*)a, (float*)g, (const float*)u,               \
                     (const bf16*)ra_t, (const bf16*)ra_b, (const bf16*)ri_t, (const bf16*)ri_b, (const bf16*)lam, tokens,   \
                     nb, bw, scale)
    if (split) SM_GATES(sm_rglru_gates_split_kernel, grid);
    else
      hipLaunchKernelGGL(sm_rglru_gates_column_kernel, cols, dim3(256), 0, (hipStream_t)stream,
                         GateArgs{(float*)a, (float*)g, (const float*)u, (const bf16*)ra_t, (const bf16*)ra_b, (const bf16*)ri_t,
                                  (const bf16*)ri_b, (const bf16*)lam, tokens, nb, bw, scale});
#undef SM_GATES
    DLLM_HIP_CHECK(hipGetLastError());
    return;
  }
  hipLaunchKernelGGL(sm_rglru_gates_kernel, dim3((tokens + kGT - 1) / kGT, nb, (bw + 127) / 128), dim3(256), 0,
                     (hipStream_t)stream, (float*)a, (float*)g, (const float*)u, (const float*)ra_t, (const float*)ra_b,
                     (const float*)ri_t, (const float*)ri_b, (const float*)lam, tokens, nb, bw, scale);
  DLLM_HIP_CHECK(hipGetLastError());
}

// --------------------------------------------------------------------------- RG-LRU scan
// S_t = a_t S_(t-1) + g_t per (sequence, channel), from the slot's state (zero at position 0);
// out_t = S_t * gelu_tanh(y_raw_t + y_bias).  One thread per channel walks its sequence's chunk.
__device__ __forceinline__ float gelu_tanh_f(float z) {
  return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}

template <typename T>
__global__ void __launch_bounds__(64) sm_rglru_scan_kernel(void* __restrict__ out_, const float* __restrict__ a,
                                                           const float* __restrict__ g,
                                                           const void* __restrict__ y_raw_, long y_stride,
                                                           const void* __restrict__ y_bias_,
                                                           float* __restrict__ state, const int32_t* __restrict__ cu,
                                                           const int32_t* __restrict__ positions,
                                                           const int32_t* __restrict__ slots, int C) {
  const int b = blockIdx.y;
  const int c = blockIdx.x * 64 + threadIdx.x;
  const int lo = cu[b], hi = cu[b + 1];
  if (c >= C || hi <= lo) return;
  const T* y_raw = (const T*)y_raw_;
  T* out = (T*)out_;
  float* sp = state + (size_t)slots[b] * C + c;
  float s = positions[lo] > 0 ? *sp : 0.f;
  const float yb = ldf((const T*)y_bias_ + c);
  // the recurrence is a dependent chain, its operands are not: 8 steps' loads go out together
  int t = lo;
  for (; t + 8 <= hi; t += 8) {
    float av[8], gv[8], yv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const size_t i = (size_t)(t + j) * C + c;
      av[j] = a[i];
      gv[j] = g[i];
      yv[j] = ldf(y_raw + (size_t)(t + j) * y_stride + c);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      s = fmaf(av[j], s, gv[j]);
      stf(out + (size_t)(t + j) * C + c, s * gelu_tanh_f(yv[j] + yb));
    }
  }
  for (; t < hi; ++t) {
    const size_t i = (size_t)t * C + c;
    s = fmaf(a[i], s, g[i]);
    stf(out + i, s * gelu_tanh_f(ldf(y_raw + (size_t)t * y_stride + c) + yb));
  }
  *sp = s;
}

// Long chunks of few sequences: the recurrence S_t = a_t S_(t-1) + g_t is affine in S, so a chunk cut
// into segments of kSeg tokens is scanned in two launches.  The first reduces every segment to its
// composition (A = prod a_t, B = the segment scanned from zero); the second gives every (sequence,
// segment) its start state -- the slot's state folded through the earlier segments' (A, B) -- and scans
// the segment with outputs.  sequences x segments x channels / 64 waves instead of sequences x channels / 64.
constexpr int kSeg = 128;

__global__ void __launch_bounds__(64) sm_rglru_seg_reduce_kernel(float* __restrict__ ab, float* __restrict__ s0,
                                                                 const float* __restrict__ a,
                                                                 const float* __restrict__ g,
                                                                 const float* __restrict__ state,
                                                                 const int32_t* __restrict__ cu,
                                                                 const int32_t* __restrict__ positions,
                                                                 const int32_t* __restrict__ slots, int C, int nseg) {
  const int b = blockIdx.y, sg = blockIdx.z;
  const int c = blockIdx.x * 64 + threadIdx.x;
  const int lo = cu[b] + sg * kSeg, hi = min(cu[b + 1], lo + kSeg);
  if (c >= C || lo >= hi) return;
  // the sequence's state before this step, copied where the second launch reads it: that launch's last
  // segment overwrites the slot while other segments may not have started yet
  if (sg == 0) s0[(size_t)b * C + c] = positions[lo] > 0 ? state[(size_t)slots[b] * C + c] : 0.f;
  float A = 1.f, B = 0.f;
  int t = lo;
  for (; t + 8 <= hi; t += 8) {
    float av[8], gv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) av[j] = a[(size_t)(t + j) * C + c], gv[j] = g[(size_t)(t + j) * C + c];
#pragma unroll
    for (int j = 0; j < 8; ++j) A *= av[j], B = fmaf(av[j], B, gv[j]);
  }
  for (; t < hi; ++t) {
    const float av = a[(size_t)t * C + c];
    A *= av, B = fmaf(av, B, g[(size_t)t * C + c]);
  }
  float* o = ab + (((size_t)b * nseg + sg) * 2) * C + c;
  o[0] = A;
  o[C] = B;
}

template <typename T>
__global__ void __launch_bounds__(64) sm_rglru_seg_scan_kernel(void* __restrict__ out_, const float* __restrict__ a,
                                                               const float* __restrict__ g,
                                                               const void* __restrict__ y_raw_, long y_stride,
                                                               const void* __restrict__ y_bias_,
                                                               float* __restrict__ state, const float* __restrict__ ab,
                                                               const float* __restrict__ s0,
                                                               const int32_t* __restrict__ cu,
                                                               const int32_t* __restrict__ slots, int C, int nseg) {
  const int b = blockIdx.y, sg = blockIdx.z;
  const int c = blockIdx.x * 64 + threadIdx.x;
  const int first = cu[b], end = cu[b + 1];
  const int lo = first + sg * kSeg, hi = min(end, lo + kSeg);
  if (c >= C || lo >= hi) return;
  const T* y_raw = (const T*)y_raw_;
  T* out = (T*)out_;
  float s = s0[(size_t)b * C + c];
  for (int j = 0; j < sg; ++j) {                          // the earlier segments, composed
    const float* p = ab + (((size_t)b * nseg + j) * 2) * C + c;
    s = fmaf(p[0], s, p[C]);
  }
  const float yb = ldf((const T*)y_bias_ + c);
  int t = lo;
  for (; t + 8 <= hi; t += 8) {
    float av[8], gv[8], yv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const size_t i = (size_t)(t + j) * C + c;
      av[j] = a[i];
      gv[j] = g[i];
      yv[j] = ldf(y_raw + (size_t)(t + j) * y_stride + c);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      s = fmaf(av[j], s, gv[j]);
      stf(out + (size_t)(t + j) * C + c, s * gelu_tanh_f(yv[j] + yb));
    }
  }
  for (; t < hi; ++t) {
    const size_t i = (size_t)t * C + c;
    s = fmaf(a[i], s, g[i]);
    stf(out + i, s * gelu_tanh_f(ldf(y_raw + (size_t)t * y_stride + c) + yb));
  }
  if (hi == end) state[(size_t)slots[b] * C + c] = s;     // the sequence's last segment leaves the new state
}

// ab: workspace of seqs x (ceil(max_q_len / kSeg) x 2 + 1) x C floats (0: always the one-launch scan)
void sm_rglru_scan(uintptr_t out, uintptr_t a, uintptr_t g, uintptr_t y_raw, long y_stride, uintptr_t y_bias,
                   uintptr_t state, uintptr_t cu, uintptr_t positions, uintptr_t slots, int seqs, int C, int max_q_len,
                   uintptr_t ab, int f32, uintptr_t stream) {
  if (seqs <= 0) return;
  DLLM_HOST_CHECK(C > 0 && y_stride >= C && seqs <= 65535, "rglru scan sizes");
  const int nseg = (max_q_len + kSeg - 1) / kSeg;
  if (ab && nseg > 1 && nseg <= 65535) {
    const dim3 grid((C + 63) / 64, seqs, nseg);
    float* s0 = (float*)ab + (size_t)seqs * nseg * 2 * C;
    hipLaunchKernelGGL(sm_rglru_seg_reduce_kernel, grid, dim3(64), 0, (hipStream_t)stream, (float*)ab, s0,
                       (const float*)a, (const float*)g, (const float*)state, (const int32_t*)cu,
                       (const int32_t*)positions, (const int32_t*)slots, C, nseg);
    DLLM_HIP_CHECK(hipGetLastError());
    SM_DISPATCH(f32, sm_rglru_seg_scan_kernel, grid, dim3(64), 0, stream, (void*)out, (const float*)a, (const float*)g,
                (const void*)y_raw, y_stride, (const void*)y_bias, (float*)state, (const float*)ab, (const float*)s0,
                (const int32_t*)cu, (const int32_t*)slots, C, nseg);
    return;
  }
  SM_DISPATCH(f32, sm_rglru_scan_kernel, dim3((C + 63) / 64, seqs), dim3(64), 0, stream, (void*)out, (const float*)a,
              (const float*)g, (const void*)y_raw, y_stride, (const void*)y_bias, (float*)state, (const int32_t*)cu,
              (const int32_t*)positions, (const int32_t*)slots, C);
}

// --------------------------------------------------------------------------- RG-LRU, one token per sequence
// The whole recurrent branch of a decode step in one launch: the causal convolution of x (with its bias) and its new tail,
// both gates, the state update and the gelu(y) product -- what the conv, conv tail, gate and scan kernels above do in four.
// One workgroup per (64 outputs of a block of bw channels, GT_ sequences).  It is bound by round trips and by what one CU
// can pull in (256 outputs per workgroup: 10.2-10.8 us, of one sequence as of 16), so the outputs are cut small and the
// loads go out in as few rounds as they can: lane group og = tid % 8 owns 8 consecutive outputs and kg = tid / 8 every 32nd
// input row of both gate matrices, a block of up to 256 being one round of kRows rows per thread that is sent out before
// anything waits (the gate kernel had two weight loads in flight per thread: 19-27 us by itself), and each finishing
// thread has its state, y and biases in registers before the convolution starts.
// A gate needs all bw convolved inputs of its block, so every workgroup of a block convolves them all, and the tail may
// move only when all have read it: each counts itself in `arrived` [state slots][blocks] once its reads have returned, and
// the last of them -- nobody waits -- writes the new tail.  The count belongs to the slot whose tail it guards, so launches
// on other slots, on whatever stream or in whatever graph, never meet in it, and it wraps to zero by itself at the last
// arrival (rows that share the scratch slot leave a whole number of turns).
// What is then left is a chain in one wave (us of 4.7 behind the launch: 1.1 to send all loads out, 0.3 convolution, 1.5 products,
// 0.5 sums, 0.7 close): a whole round of rows is multiplied without a branch or select per row (1.5 -> 0.8), and the softplus and
// the gelu(y), which ask for no gate, are made under the weights' round trip (close 0.7 -> 0.4).
// 4 blocks of 256, 4 taps, bf16, in a graph: one sequence 6.1 -> 5.5 us (30 in four launches); 10 blocks: 16 sequences 9.6 -> 8.3
// (42), 64 sequences 19.4 -> 18.
constexpr int kRows = 8;       // gate matrix rows in flight per thread
constexpr int kStepTaps = 8;   // at most
constexpr int kStepOut = 64;   // outputs per workgroup
constexpr int kCountStride = 32;
template <typename T> struct Raw8 { typedef bf16x8 type; };
template <> struct Raw8<float> { typedef float type __attribute__((ext_vector_type(8))); };

template <typename T, int GT_, int TAPS_>
__global__ void __launch_bounds__(256) sm_rglru_step_kernel(
    const int32_t* __restrict__ slots, const int32_t* __restrict__ positions, const void* __restrict__ ra_t_,
    const void* __restrict__ ri_t_, int seqs, int nb, int bw, int taps, void* conv_state_,   // (14 words: they come with the wave)
    void* __restrict__ out_, const void* __restrict__ x_, const void* __restrict__ y_, long ld,
    const void* __restrict__ conv_w_, const void* __restrict__ conv_b_, const void* __restrict__ x_b_,
    const void* __restrict__ ra_b_, const void* __restrict__ ri_b_, const void* __restrict__ lam_, const void* __restrict__ y_b_,
    float* __restrict__ state, float scale, unsigned* __restrict__ arrived) {
  typedef typename Raw8<T>::type raw8;
  extern __shared__ float smem[];
  constexpr int kPitch = 2 * GT_ * kStepOut + 4;      // (+ 4: the groups of a wave write to banks of their own)
  float* red = smem;                                  // [32 groups][2 gates][GT_][64], kPitch apart
  float* red2 = red + 32 * kPitch;                    // [2 gates][GT_][64]
  float* ubs = red2 + 2 * GT_ * kStepOut;             // [GT_][bw] convolved inputs
  T* tail = (T*)(ubs + GT_ * bw);                     // [GT_][taps - 1][bw] the new tail
  __shared__ int last[GT_];
  const int nz = (bw + kStepOut - 1) / kStepOut;
  const int b = blockIdx.x / nz, o0 = (blockIdx.x % nz) * kStepOut;
  const int s0 = blockIdx.y * GT_, C = nb * bw;
  const int tid = threadIdx.x, og = tid & 7, kg = tid >> 3;
  const int ob = min(o0 + 8 * og, bw - 8);            // this lane's 8 outputs (past the block: repeated, never used)
  const T* ra = (const T*)ra_t_ + (size_t)b * bw * bw + ob;
  const T* ri = (const T*)ri_t_ + (size_t)b * bw * bw + ob;
  raw8 wr[kRows], wi[kRows];
  auto load_rows = [&](int i0) {
#pragma unroll
    for (int q = 0; q < kRows; ++q) {
      const size_t at = (size_t)min(i0 + 32 * q, bw - 1) * bw;
      wr[q] = *reinterpret_cast<const raw8*>(ra + at);
      wi[q] = *reinterpret_cast<const raw8*>(ri + at);
    }
  };
  // every load off a clamped place and none behind a branch (hipcc waits out a load inside a branch, uniform or not,
  // before the next: 15 round trips, 5 us).  A lane's first channel, what the finishing threads (output fo of sequence fk)
  // need, and the first round of weights go out together
  const int fk = __builtin_amdgcn_readfirstlane(tid >> 6), fo = o0 + (tid & 63), fq = min(s0 + min(fk, GT_ - 1), seqs - 1);
  const bool fin = fk < GT_ && s0 + fk < seqs && fo < bw;
  const int fc = b * bw + min(fo, bw - 1);
  float* fstate = state + (size_t)slots[fq] * C + fc;
  int pos[GT_], slot[GT_];
#pragma unroll
  for (int k = 0; k < GT_; ++k) {
    const int q = min(s0 + k, seqs - 1);                        // past the last sequence: repeated, never used
    pos[k] = positions[q], slot[k] = slots[q];
  }
  T w[TAPS_], v[GT_][TAPS_], xb, cb;
  auto load_taps = [&](int c) {
    xb = ((const T*)x_b_)[c], cb = ((const T*)conv_b_)[c];
#pragma unroll
    for (int j = 0; j < TAPS_; ++j) w[j] = ((const T*)conv_w_)[(size_t)min(j, taps - 1) * C + c];
#pragma unroll
    for (int k = 0; k < GT_; ++k) {
      const T* st = (const T*)conv_state_ + (size_t)slot[k] * (taps - 1) * C + c;
      const T* xr = (const T*)x_ + (size_t)min(s0 + k, seqs - 1) * ld + c;
#pragma unroll
      for (int j = 0; j < TAPS_; ++j) v[k][j] = *(j < taps - 1 ? st + (size_t)j * C : xr);
    }
  };
  load_taps(b * bw + min(tid, bw - 1));
  const float s_in = *fstate;
  const T y_in = ((const T*)y_)[(size_t)fq * ld + fc], y_b = ((const T*)y_b_)[fc], lam = ((const T*)lam_)[fc];
  const T rb = ((const T*)ra_b_)[fc], ib = ((const T*)ri_b_)[fc];
  const int fpos = positions[fq];
  load_rows(kg);

  // convolution of the block's channels, a lane per channel; the new tail (the old one a row up, then x) waits in LDS
  for (int ci = tid; ci < bw; ci += 256) {
    if (ci != tid) load_taps(b * bw + ci);
#pragma unroll
    for (int k = 0; k < GT_; ++k) {
      float acc = (float)cb;
#pragma unroll
      for (int j = 0; j < TAPS_; ++j) {
        if (j < taps) {
          const bool live = taps - 1 - j <= pos[k];             // the row lies at or after the sequence's start
          const T z = live ? v[k][j] : (T)0.f;
          if (live) acc += (float)w[j] * ((float)z + (float)xb);
          if (j > 0) tail[(size_t)(k * (taps - 1) + j - 1) * bw + ci] = z;
        }
      }
      ubs[k * bw + ci] = acc;
    }
  }
  __syncthreads();                                    // every read of the old tail in this workgroup has returned
  // (counters on lines of their own; the answer is not needed before the end)
  unsigned before = 0;
  if (tid < GT_ && s0 + tid < seqs)
    before = atomicInc(arrived + ((size_t)(tid == 0 ? slot[0] : slot[GT_ - 1]) * nb + b) * kCountStride, nz - 1);

  // what the state's close takes besides the gates, under the weights' round trip (pinned: hipcc sinks it to its use)
  float sp = 0.f, gy = 0.f;
  if (fk < GT_) {                                     // uniform
    sp = softplus_f((float)lam), gy = gelu_tanh_f((float)y_in + (float)y_b);
    asm volatile("" : "+v"(sp), "+v"(gy));
  }
  float ar[GT_][8], ai[GT_][8];
#pragma unroll
  for (int k = 0; k < GT_; ++k)
#pragma unroll
    for (int j = 0; j < 8; ++j) ar[k][j] = 0.f, ai[k][j] = 0.f;
  for (int i0 = kg; i0 < bw; i0 += 32 * kRows) {
    if (i0 > kg) load_rows(i0);
    if (i0 - kg + 32 * kRows <= bw) {                           // uniform: a whole round, without a branch or select per row
      float u[GT_][kRows];
#pragma unroll
      for (int k = 0; k < GT_; ++k)
#pragma unroll
        for (int q = 0; q < kRows; ++q) u[k][q] = ubs[k * bw + i0 + 32 * q];
#pragma unroll
      for (int q = 0; q < kRows; ++q)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float fr = (float)wr[q][j], fi = (float)wi[q][j];
#pragma unroll
          for (int k = 0; k < GT_; ++k) ar[k][j] = fmaf(fr, u[k][q], ar[k][j]), ai[k][j] = fmaf(fi, u[k][q], ai[k][j]);
        }
      continue;
    }
#pragma unroll
    for (int q = 0; q < kRows; ++q) {
      const int base = i0 - kg + 32 * q, i = base + kg;         // base: uniform
      if (base < bw) {
        float fr[8], fi[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          fr[j] = (float)wr[q][j], fi[j] = (float)wi[q][j];
          if (base + 32 > bw) fr[j] = i < bw ? fr[j] : 0.f, fi[j] = i < bw ? fi[j] : 0.f;   // a last, partial round
        }
#pragma unroll
        for (int k = 0; k < GT_; ++k) {
          const float u = i < bw ? ubs[k * bw + min(i, bw - 1)] : 0.f;
#pragma unroll
          for (int j = 0; j < 8; ++j) ar[k][j] = fmaf(fr[j], u, ar[k][j]), ai[k][j] = fmaf(fi[j], u, ai[k][j]);
        }
      }
    }
  }
#pragma unroll
  for (int k = 0; k < GT_; ++k)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float* r0 = red + kg * kPitch + k * kStepOut + 8 * og + 4 * h;
      float* r1 = red + kg * kPitch + (GT_ + k) * kStepOut + 8 * og + 4 * h;
      *reinterpret_cast<f32x4*>(r0) = f32x4{ar[k][4 * h], ar[k][4 * h + 1], ar[k][4 * h + 2], ar[k][4 * h + 3]};
      *reinterpret_cast<f32x4*>(r1) = f32x4{ai[k][4 * h], ai[k][4 * h + 1], ai[k][4 * h + 2], ai[k][4 * h + 3]};
    }
  __syncthreads();
  for (int e = tid; e < 2 * GT_ * kStepOut; e += 256) {         // (gate, sequence, output): the 32 groups in order
    float sum = 0.f;
#pragma unroll
    for (int g = 0; g < 32; ++g) sum += red[g * kPitch + e];
    red2[e] = sum;
  }
  if (tid < GT_) last[tid] = before == nz - 1;
  __syncthreads();
  if (fin) {
    const float sr = red2[fk * kStepOut + (tid & 63)], si = red2[(GT_ + fk) * kStepOut + (tid & 63)];
    const float av = expf(-scale * sigmoid_f(sr + (float)rb) * sp);
    const float gv = sqrtf(1.0f - av * av) * sigmoid_f(si + (float)ib) * ubs[fk * bw + fo];
    const float s = fmaf(av, fpos > 0 ? s_in : 0.f, gv);
    *fstate = s;
    stf((T*)out_ + (size_t)fq * C + b * bw + fo, s * gy);
  }
#pragma unroll
  for (int k = 0; k < GT_; ++k) {
    if (s0 + k < seqs && last[k]) {                   // uniform
      for (int ci = tid; ci < bw; ci += 256) {
        T* st = (T*)conv_state_ + (size_t)slot[k] * (taps - 1) * C + b * bw + ci;
        for (int j = 0; j < taps - 1; ++j) st[(size_t)j * C] = tail[(size_t)(k * (taps - 1) + j) * bw + ci];
      }
    }
  }
}

// Every sequence brings one token, token q of the batch is sequence q's.  x / y: the two halves of the projection (rows
// ld apart); out [tokens, C]; arrived: num_slots x blocks counters, 32 ints apart, zero before the first launch.
void sm_rglru_step(uintptr_t out, uintptr_t x, uintptr_t y, long ld, uintptr_t conv_w, uintptr_t conv_b, uintptr_t x_b,
                   uintptr_t conv_state, uintptr_t ra_t, uintptr_t ra_b, uintptr_t ri_t, uintptr_t ri_b, uintptr_t lam,
                   uintptr_t y_b, uintptr_t state, uintptr_t positions, uintptr_t slots, int seqs, int nb,
                   int bw, int taps, float scale, uintptr_t arrived, long arrived_len, int num_slots, int f32,
                   uintptr_t stream) {
  if (seqs <= 0) return;
  DLLM_HOST_CHECK(nb > 0 && bw >= 8 && bw % 8 == 0 && bw <= 512 && (long)nb * bw <= (1L << 24), "rglru step block sizes");
  DLLM_HOST_CHECK(taps >= 1 && taps <= kStepTaps && ld >= (long)nb * bw, "rglru step sizes");
  // sequences per workgroup: two halve the passes over the matrices, which the L2 bears while the grid is small.  us, one / two:
  // 10 blocks of 256 at 16 / 28 / 32 sequences 7.3 / 9.8 / 10.7 and 8.4 / 10.2 / 10.4, 4 blocks of 256 at 32 6.5 and 7.0, 8 blocks of
  // 64 5.0 and 6.2, 20 of 128 10.6 and 10.1; at 64 16.6, 8.2, 6.2, 16.0 and 16.8, 8.6, 6.2, 16.1; at 128 10 and 16 of 256 28.3, 41.9 and
  // 26.4, 38.7
  const int gt = seqs <= 32 ? 1 : 2;
  const int groups = (seqs + gt - 1) / gt;
  DLLM_HOST_CHECK(arrived != 0 && (long)num_slots * nb * kCountStride <= arrived_len && groups <= 65535, "rglru step counters");
  const size_t lds = ((size_t)(33 * 2 * gt * kStepOut + 32 * 4) + (size_t)gt * bw) * sizeof(float) +
                     (size_t)gt * (taps - 1) * bw * (f32 ? 4 : 2);
  // consecutive workgroups run on consecutive XCDs: the (block, output) index first, so that with 8 or more of them a
  // weight tile is read into the L2 of as few XCDs as can be
  const dim3 grid(nb * ((bw + kStepOut - 1) / kStepOut), groups);
#define SM_STEP(T, G_, N_)                                                                                                \
  do {                                                                                                               \
    if (lds > 64 * 1024)                                                                                             \
      DLLM_HIP_CHECK(hipFuncSetAttribute((const void*)sm_rglru_step_kernel<T, G_, N_>,                                    \
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));                      \
    hipLaunchKernelGGL(HIP_KERNEL_NAME(sm_rglru_step_kernel<T, G_, N_>), grid, dim3(256), lds, (hipStream_t)stream,       \
                       (const int32_t*)slots, (const int32_t*)positions, (const void*)ra_t, (const void*)ri_t, seqs, nb, bw,  \
                       taps, (void*)conv_state, (void*)out, (const void*)x, (const void*)y, ld, (const void*)conv_w,          \
                       (const void*)conv_b, (const void*)x_b, (const void*)ra_b, (const void*)ri_b, (const void*)lam,         \
                       (const void*)y_b, (float*)state, scale, (unsigned*)arrived);                                          \
  } while (0)
#define SM_STEP_T(T)                                            \
  do {                                                          \
    if (gt == 1 && taps <= 4) SM_STEP(T, 1, 4);                 \
    else if (gt == 1) SM_STEP(T, 1, kStepTaps);                 \
    else if (taps <= 4) SM_STEP(T, 2, 4);                       \
    else SM_STEP(T, 2, kStepTaps);                              \
  } while (0)
  if (f32) SM_STEP_T(float);
  else SM_STEP_T(bf16);
#undef SM_STEP_T
#undef SM_STEP
  DLLM_HIP_CHECK(hipGetLastError());
}

// --------------------------------------------------------------------------- clipped GLU
template <typename T, int V>
__global__ void __launch_bounds__(256) sm_clipped_glu_kernel(void* __restrict__ out_, const void* __restrict__ gu_,
                                                             const void* __restrict__ bias_, int F, float limit,
                                                             float alpha) {
  const T* gu = (const T*)gu_ + (size_t)blockIdx.x * 2 * F;
  const T* bias = (const T*)bias_;
  T* out = (T*)out_ + (size_t)blockIdx.x * F;
  for (int c = (blockIdx.y * 256 + threadIdx.x) * V; c < F; c += gridDim.y * 256 * V) {
    float gv[V], uv[V], b1[V], b2[V];
    ldv<V>(gu + c, gv);
    ldv<V>(gu + F + c, uv);
    if (bias) {
      ldv<V>(bias + c, b1);
      ldv<V>(bias + F + c, b2);
#pragma unroll
      for (int j = 0; j < V; ++j) gv[j] += b1[j], uv[j] += b2[j];
    }
#pragma unroll
    for (int j = 0; j < V; ++j) gv[j] = clipped_glu_exact_f(gv[j], uv[j], limit, alpha);
    stv<V>(out + c, gv);
  }
}

void sm_clipped_glu(uintptr_t out, uintptr_t gu, uintptr_t bias, int tokens, int F, float limit, float alpha, int f32,
                    uintptr_t stream) {
  if (tokens <= 0 || F <= 0) return;
  const int vec = F % 8 == 0;
  const int per = 256 * (vec ? 8 : 1);
  SM_DISPATCH_V(f32, vec, sm_clipped_glu_kernel, dim3(tokens, std::min(16, (F + per - 1) / per)), dim3(256), 0, stream,
                (void*)out, (const void*)gu, (const void*)bias, F, limit, alpha);
}

// --------------------------------------------------------------------------- gelu GLU
// out [T, F] = gelu_tanh(gate) * up of a fused gate | up projection
template <typename T, int V>
__global__ void __launch_bounds__(256) sm_gelu_glu_kernel(void* __restrict__ out_, const void* __restrict__ gu_, int F) {
  const T* gu = (const T*)gu_ + (size_t)blockIdx.x * 2 * F;
  T* out = (T*)out_ + (size_t)blockIdx.x * F;
  for (int c = (blockIdx.y * 256 + threadIdx.x) * V; c < F; c += gridDim.y * 256 * V) {
    float g[V], u[V];
    ldv<V>(gu + c, g);
    ldv<V>(gu + F + c, u);
#pragma unroll
    for (int j = 0; j < V; ++j) g[j] = gelu_glu_exact_f(g[j], u[j]);
    stv<V>(out + c, g);
  }
}

void sm_gelu_glu(uintptr_t out, uintptr_t gu, int tokens, int F, int f32, uintptr_t stream) {
  if (tokens <= 0 || F <= 0) return;
  DLLM_HOST_CHECK(out && gu, "gelu_glu arguments");
  const int vec = F % 8 == 0;
  const int per = 256 * (vec ? 8 : 1);
  SM_DISPATCH_V(f32, vec, sm_gelu_glu_kernel, dim3(tokens, std::min(16, (F + per - 1) / per)), dim3(256), 0, stream,
                (void*)out, (const void*)gu, F);
}

// --------------------------------------------------------------------------- logit soft cap
template <typename T>
__global__ void __launch_bounds__(256) sm_softcap_kernel(float* __restrict__ out, const void* __restrict__ x_, long n,
                                                         float cap, float scale) {
  const T* x = (const T*)x_;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
    const float v = ldf(x + i) * scale;
    out[i] = cap > 0.f ? cap * tanhf(v / cap) : v;
  }
}

void sm_softcap(uintptr_t out, uintptr_t x, long n, float cap, float scale, int f32, uintptr_t stream) {
  if (n <= 0) return;
  const int grid = (int)std::min<long>((n + 255) / 256, 65535);
  SM_DISPATCH(f32, sm_softcap_kernel, dim3(grid), dim3(256), 0, stream, (float*)out, (const void*)x, n, cap, scale);
}

// --------------------------------------------------------------------------- attention input stage
// One wave per (token, head) of the fused projection [q heads | k heads | v heads]: the causal
// convolution of the head's channels, then for q / k the RMS norm over the head (plain weight) and
// the rotation of pairs (2i, 2i + 1), i < nrot, by pos * freqs[i] (cos and sin scaled by mag);
// q goes to q_out [T, H, D], k / v to the paged caches [NB, G, BS, D] / [NB, G, Dv, BS] (V transposed
// inside a block).
template <typename T>
__global__ void __launch_bounds__(64) sm_attn_prep_kernel(
    void* __restrict__ q_out_, const void* __restrict__ qkv_, const void* __restrict__ conv_w_,
    const void* __restrict__ state_, const void* __restrict__ q_norm_, const void* __restrict__ k_norm_,
    const float* __restrict__ freqs, int nrot, float mag, float eps, void* __restrict__ k_cache_,
    void* __restrict__ v_cache_, const int32_t* __restrict__ slot_mapping, const int32_t* __restrict__ cu,
    const int32_t* __restrict__ positions, const int32_t* __restrict__ tok_seq, const int32_t* __restrict__ slots,
    int H, int G, int D, int Dv, int taps, int bs) {
  extern __shared__ float hv[];                      // the head's values [max(D, Dv)]
  const int t = blockIdx.x, head = blockIdx.y, lane = threadIdx.x;
  const int C = H * D + G * (D + Dv);
  const int b = tok_seq[t];
  const int tl = t - cu[b], pos = positions[t];
  const T* qkv = (const T*)qkv_;
  const T* w = (const T*)conv_w_;
  const T* st = (const T*)state_ + (size_t)slots[b] * (taps - 1) * C;
  // channel range and kind of this head
  int c0, n, kind;                                   // kind 0 q, 1 k, 2 v
  if (head < H) c0 = head * D, n = D, kind = 0;
  else if (head < H + G) c0 = H * D + (head - H) * D, n = D, kind = 1;
  else c0 = H * D + G * D + (head - H - G) * Dv, n = Dv, kind = 2;
  float ss = 0.f;
  for (int e = lane; e < n; e += 64) {
    const int c = c0 + e;
    float acc = 0.f;
    for (int j = 0; j < taps; ++j)
      acc += ldf(w + (size_t)j * C + c) * conv_input(qkv, (long)C, st, t, tl, pos, taps - 1 - j, taps, c, C);
    hv[e] = acc;
    ss += acc * acc;
  }
  T* dst;
  if (kind == 0) dst = (T*)q_out_ + ((size_t)t * H + head) * D;
  else {
    const int slot = slot_mapping[t];
    const int blk = slot / bs, off = slot - blk * bs;
    if (kind == 1) dst = (T*)k_cache_ + (((size_t)blk * G + (head - H)) * bs + off) * D;
    else dst = (T*)v_cache_ + ((size_t)blk * G + (head - H - G)) * Dv * bs + off;
  }
  if (kind == 2) {
    for (int e = lane; e < n; e += 64) stf(dst + (size_t)e * bs, hv[e]);
    return;
  }
  ss = wave_sum(ss);
  const float inv = 1.0f / sqrtf(ss / (float)n + eps);
  const T* nw = (const T*)(kind == 0 ? q_norm_ : k_norm_);
  __syncthreads();
  for (int e = lane; e < n; e += 64) hv[e] = hv[e] * inv * ldf(nw + e);
  __syncthreads();
  const float fpos = (float)pos;
  for (int i = lane; 2 * i < n; i += 64) {
    float x0 = hv[2 * i], x1 = 2 * i + 1 < n ? hv[2 * i + 1] : 0.f;
    if (i < nrot) {
      const float ang = fpos * freqs[i];
      const float cs = cosf(ang) * mag, sn = sinf(ang) * mag;
      const float r0 = x0 * cs - x1 * sn, r1 = x1 * cs + x0 * sn;
      x0 = r0, x1 = r1;
    }
    stf(dst + 2 * i, x0);
    if (2 * i + 1 < n) stf(dst + 2 * i + 1, x1);
  }
}

// The same with even head sizes: a lane owns rotation pairs (channels 2e, 2e + 1), so the convolution
// reads 2-element vectors, the rotation needs no exchange through LDS, and q / k leave as 2-element
// stores.  Heads up to 128 R wide, R <= 4.
// On prompts it was bound by round trips (a tap's rows behind a branch each) and by the cosines and sines, the same in all heads: all
// rows of a head go out at once (TAPS 2 .. 4, known to the compiler: as a number up to 4 they cost 14 registers and 3 to 28 % of
// the prompts of 100 to 1000 tokens), and in MANY a wave takes every 4 gridDim.y-th head of its token, which share the angles.
// TAPS 0: any number, one after the other.
// us with the state's launch, a tap at a time behind branches -> this, q + k + v heads x width, 100 / 500 / 2048 / 8000 tokens:
//   24 x 128, 4 taps    7.2 / 10.9 / 29 / 92  ->  7.0 / 10.8 / 23 / 61       80 x 64, 4 taps  8.7 / 21.1 / 72 / 260  ->  8.7 / 17.9 / 49 / 145
//   10 x 256, 4 taps    7.6 / 9.8 / 24 / 68   ->  6.9 / 9.1 / 20 / 50        9 x 64, 5 taps   6.9 / 7.5 / 13.3 / 43  ->  6.6 / 7.4 / 13.5 / 40
//   6 x 512, 2 taps     7.7 / 9.9 / 23 / 58   ->  6.9 / 9.0 / 19 / 47 (a wave per head: MANY's registers leave too few waves, 51 at 8000)
constexpr int kPrepPairs = 4;
constexpr int kPrepGroups = 2048;     // workgroups that are resident together: eight on each CU

template <typename T, int R, int TAPS, bool MANY>
__global__ void __launch_bounds__(256) sm_attn_prep_pair_kernel(
    const int32_t* __restrict__ tok_seq, const int32_t* __restrict__ cu, const int32_t* __restrict__ positions,
    const int32_t* __restrict__ slots, int H, int G, int D, int Dv, int taps_, int bs,   // (14 words: they come with the wave)
    void* __restrict__ q_out_, const void* __restrict__ qkv_, const void* __restrict__ conv_w_, const void* state_,
    const void* __restrict__ q_norm_, const void* __restrict__ k_norm_, const float* __restrict__ freqs, int nrot, float mag,
    float eps, void* __restrict__ k_cache_, void* __restrict__ v_cache_, const int32_t* __restrict__ slot_mapping, void* tail_) {
  static_assert(TAPS > 0 || !MANY, "the next head's rows are read ahead");
  constexpr int NT = TAPS > 0 ? TAPS : 1;
  const int taps = TAPS > 0 ? TAPS : taps_;
  const int t = blockIdx.x, lane = threadIdx.x & 63;
  const int C = H * D + G * (D + Dv);
  const int b = tok_seq[t];
  const int tl = t - cu[b], pos = positions[t];
  const T* qkv = (const T*)qkv_;
  const T* w = (const T*)conv_w_;
  const T* st = (const T*)state_ + (size_t)slots[b] * (taps - 1) * C;
  typedef T pair __attribute__((ext_vector_type(2)));
  pair xn[R][NT], wn[R][NT];                           // a head's rows and weights
  auto channels = [&](int head, int& c0, int& n, int& kind) {   // kind 0 q, 1 k, 2 v
    if (head < H) c0 = head * D, n = D, kind = 0;
    else if (head < H + G) c0 = H * D + (head - H) * D, n = D, kind = 1;
    else c0 = H * D + G * D + (head - H - G) * Dv, n = Dv, kind = 2;
  };
  auto load = [&](int head) {                          // every load at once, off a place that is always there
    int c0, n, kind;
    channels(head, c0, n, kind);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int c = c0 + min(2 * (lane + 64 * r), n - 2);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        wn[r][j] = *reinterpret_cast<const pair*>(w + (size_t)j * C + c);
        xn[r][j] = *reinterpret_cast<const pair*>(conv_row(qkv, (long)C, st, t, tl, taps - 1 - j, taps, C) + c);
      }
    }
  };
  int head = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (head >= H + 2 * G) return;
  if constexpr (TAPS > 0) load(head);
  float cs[MANY ? R : 1], sn[MANY ? R : 1];            // one wave's heads share the angles
  bool angles = false;
  auto angle = [&](int i, float& c, float& s) {
    const float ang = (float)pos * freqs[i];
    c = cosf(ang) * mag, s = sinf(ang) * mag;
  };
  for (bool more = true; more; more = MANY && (head += 4 * (int)gridDim.y) < H + 2 * G) {
    int c0, n, kind;
    channels(head, c0, n, kind);
    float x[R][2];
    float ss = 0.f;
    if constexpr (TAPS > 0) {
      float xv[R][NT][2], wv[R][NT][2];
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int e = 0; e < 2; ++e) xv[r][j][e] = (float)xn[r][j][e], wv[r][j][e] = (float)wn[r][j][e];
      if constexpr (MANY) load(min(head + 4 * (int)gridDim.y, H + 2 * G - 1));   // the next head's under this one
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int e = 2 * (lane + 64 * r);
        x[r][0] = x[r][1] = 0.f;
        if (e < n) {
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            if (taps - 1 - j > pos) xv[r][j][0] = xv[r][j][1] = 0.f;
            else {
              x[r][0] = fmaf(wv[r][j][0], xv[r][j][0], x[r][0]);
              x[r][1] = fmaf(wv[r][j][1], xv[r][j][1], x[r][1]);
            }
            // one token per sequence: the tail moves up here
            if (tail_ && j > 0) stv<2>((T*)tail_ + ((size_t)slots[b] * (taps - 1) + j - 1) * C + c0 + e, xv[r][j]);
          }
          ss += fmaf(x[r][0], x[r][0], x[r][1] * x[r][1]);
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int e = 2 * (lane + 64 * r);
        x[r][0] = x[r][1] = 0.f;
        if (e < n) {
          for (int j = max(0, taps - 1 - pos); j < taps; ++j) {
            const pair xv = *reinterpret_cast<const pair*>(conv_row(qkv, (long)C, st, t, tl, taps - 1 - j, taps, C) + c0 + e);
            const pair wv = *reinterpret_cast<const pair*>(w + (size_t)j * C + c0 + e);
            x[r][0] = fmaf((float)wv[0], (float)xv[0], x[r][0]);
            x[r][1] = fmaf((float)wv[1], (float)xv[1], x[r][1]);
          }
          ss += fmaf(x[r][0], x[r][0], x[r][1] * x[r][1]);
        }
      }
    }
    if (kind == 2) {
      const int slot = slot_mapping[t];
      const int blk = slot / bs, off = slot - blk * bs;
      T* dst = (T*)v_cache_ + ((size_t)blk * G + (head - H - G)) * Dv * bs + off;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int e = 2 * (lane + 64 * r);
        if (e < n) stf(dst + (size_t)e * bs, x[r][0]), stf(dst + (size_t)(e + 1) * bs, x[r][1]);
      }
      continue;
    }
    T* dst;
    if (kind == 0) dst = (T*)q_out_ + ((size_t)t * H + head) * D;
    else {
      const int slot = slot_mapping[t];
      const int blk = slot / bs, off = slot - blk * bs;
      dst = (T*)k_cache_ + (((size_t)blk * G + (head - H)) * bs + off) * D;
    }
    if (MANY && !angles) {                             // (uniform)
      angles = true;
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (lane + 64 * r < nrot) angle(lane + 64 * r, cs[MANY ? r : 0], sn[MANY ? r : 0]);
    }
    ss = wave_sum(ss);
    const float inv = 1.0f / sqrtf(ss / (float)n + eps);
    const T* nw = (const T*)(kind == 0 ? q_norm_ : k_norm_);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = lane + 64 * r, e = 2 * i;
      if (e < n) {
        float g2[2], o[2];
        ldv<2>(nw + e, g2);
        float x0 = x[r][0] * inv * g2[0], x1 = x[r][1] * inv * g2[1];
        if (i < nrot) {
          if (!MANY) angle(i, cs[0], sn[0]);
          const float c = cs[MANY ? r : 0], s = sn[MANY ? r : 0];
          const float r0 = fmaf(x0, c, -(x1 * s)), r1 = fmaf(x1, c, x0 * s);   // (alike in every form)
          x0 = r0, x1 = r1;
        }
        o[0] = x0, o[1] = x1;
        stv<2>(dst + e, o);
      }
    }
  }
}

void sm_attn_prep(uintptr_t q_out, uintptr_t qkv, uintptr_t conv_w, uintptr_t state, uintptr_t q_norm,
                  uintptr_t k_norm, uintptr_t freqs, int nrot, float mag, float eps, uintptr_t k_cache,
                  uintptr_t v_cache, uintptr_t slot_mapping, uintptr_t cu, uintptr_t positions, uintptr_t tok_seq,
                  uintptr_t slots, int tokens, int seqs, int H, int G, int D, int Dv, int taps, int bs, int max_q_len, int f32,
                  uintptr_t stream) {
  if (tokens <= 0 || seqs <= 0) return;
  DLLM_HOST_CHECK(H > 0 && G >= 0 && D > 0 && Dv > 0 && taps >= 1 && bs > 0 && 2 * nrot <= D, "attn_prep sizes");
  DLLM_HOST_CHECK(G == 0 || (k_cache && v_cache && k_norm), "attn_prep caches");
  DLLM_HOST_CHECK(H + 2 * G <= 65535, "attn_prep heads");
  const int C = H * D + G * (D + Dv);
  const size_t lds = (size_t)std::max(D, Dv) * sizeof(float);
  const bool pairs = D % 2 == 0 && Dv % 2 == 0 && std::max(D, Dv) <= 128 * kPrepPairs;
  // one token per sequence: a channel of a sequence's tail is read and moved up by the one lane that convolves it, so the
  // tail needs no launch of its own (4.6 us)
  const bool tail = pairs && max_q_len == 1 && taps > 1 && taps <= kConvTaps;
  if (pairs) {
    const int most = (H + 2 * G + 3) / 4, r = std::max(D, Dv) <= 128 ? 1 : std::max(D, Dv) <= 256 ? 2 : kPrepPairs;
    const bool exact = taps >= 2 && taps <= kConvTaps;
    // workgroups per token: one per four heads while those fit the chip together, else fewer whose waves take as many heads each
    // (18 heads of 64 at 500 tokens: 5 workgroups 9.1 us, 4 whose first wave takes two heads each 9.3, 3 8.6)
    int gy = most;
    if (exact && r <= 2) {
      const int fit = std::max(1, kPrepGroups / tokens), each = (most + fit - 1) / fit;
      gy = (most + each - 1) / each;
    }
#define SM_PREP_M(T_, R_, N_, MANY_)                                                                                                \
  hipLaunchKernelGGL(HIP_KERNEL_NAME(sm_attn_prep_pair_kernel<T_, R_, N_, MANY_>), dim3(tokens, gy), dim3(256), 0,         \
                     (hipStream_t)stream, (const int32_t*)tok_seq, (const int32_t*)cu, (const int32_t*)positions,            \
                     (const int32_t*)slots, H, G, D, Dv, taps, bs, (void*)q_out, (const void*)qkv, (const void*)conv_w,      \
                     (const void*)state, (const void*)q_norm, (const void*)k_norm, (const float*)freqs, nrot, mag, eps,      \
                     (void*)k_cache, (void*)v_cache, (const int32_t*)slot_mapping, tail ? (void*)state : nullptr)
#define SM_PREP_N(T_, R_, N_) do { if (R_ <= 2 && gy < most) SM_PREP_M(T_, R_, N_, (R_ <= 2)); else SM_PREP_M(T_, R_, N_, false); } while (0)
#define SM_PREP(T_, R_)                                                                                                      \
  do {                                                                                                                       \
    if (!exact) SM_PREP_M(T_, R_, 0, false);                                                                                 \
    else if (taps == 2) SM_PREP_N(T_, R_, 2);                                                                                \
    else if (taps == 3) SM_PREP_N(T_, R_, 3);                                                                                \
    else SM_PREP_N(T_, R_, 4);                                                                                               \
  } while (0)
#define SM_PREP_R(T_) do { if (r == 1) SM_PREP(T_, 1); else if (r == 2) SM_PREP(T_, 2); else SM_PREP(T_, kPrepPairs); } while (0)
    if (f32) SM_PREP_R(float);
    else SM_PREP_R(bf16);
#undef SM_PREP_R
#undef SM_PREP
#undef SM_PREP_N
#undef SM_PREP_M
    DLLM_HIP_CHECK(hipGetLastError());
  }
  else
  SM_DISPATCH(f32, sm_attn_prep_kernel, dim3(tokens, H + 2 * G), dim3(64), lds, stream, (void*)q_out, (const void*)qkv,
              (const void*)conv_w, (const void*)state, (const void*)q_norm, (const void*)k_norm, (const float*)freqs,
              nrot, mag, eps, (void*)k_cache, (void*)v_cache, (const int32_t*)slot_mapping, (const int32_t*)cu,
              (const int32_t*)positions, (const int32_t*)tok_seq, (const int32_t*)slots, H, G, D, Dv, taps, bs);
  // the projection's last taps - 1 rows of every sequence become its new tail
  if (taps > 1 && !tail)
    launch_conv_state(state, qkv, (long)C, cu, positions, slots, seqs, C, taps, f32, C % 8 == 0, stream);
}

// --------------------------------------------------------------------------- values of an attention input stage
template <typename T> __device__ __forceinline__ void add8(float (&x)[8], const T* p) {
  float b[8];
  ldv<8>(p, b);
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] += b[i];
}

// Appends one token's values v [G Dv] (+ vb, when given) to the transposed cache; with v_in (another layer's values of the
// token) v <- (1 - lam) v + lam v_in first; with v_out the values are also written there, row-major.  float32 arithmetic.
template <typename T>
__device__ __forceinline__ void append_values(const T* __restrict__ v, const T* __restrict__ vb, const T* __restrict__ v_in,
                                              T* __restrict__ v_out, float lam, T* __restrict__ vc, int blk, int off, int G,
                                              int Dv, int bs) {
  for (int e = threadIdx.x; e < G * Dv; e += blockDim.x) {
    const int g = e / Dv, c = e - g * Dv;
    float x = ldf(v + e);
    if (vb) x += ldf(vb + e);
    if (v_in) x = (1.0f - lam) * x + lam * ldf(v_in + e);
    T y;
    stf(&y, x);
    if (v_out) v_out[e] = y;
    vc[(((size_t)blk * G + g) * Dv + c) * bs + off] = y;
  }
}

// The same for `n` (1 .. 8) consecutive tokens of the batch by one workgroup, v of token j at v + j ld.  Eight tokens that
// take eight aligned places of one cache block leave as one piece per channel (a token alone touches a cache line
// per channel for 2 bytes of it).
template <typename T>
__device__ __forceinline__ void append_value_rows(const T* __restrict__ v, long ld, const T* __restrict__ vb,
                                                  const T* __restrict__ v_in, T* __restrict__ v_out, float lam,
                                                  T* __restrict__ vc, const int32_t* __restrict__ slots, int n, int G, int Dv,
                                                  int bs) {
  const int nv = G * Dv, slot0 = slots[0];
  bool run = n == 8 && slot0 % 8 == 0 && bs % 8 == 0;
  for (int j = 1; run && j < 8; ++j) run = slots[j] == slot0 + j;
  for (int e = threadIdx.x; e < nv; e += blockDim.x) {
    const int g = e / Dv, c = e - g * Dv;
    const float b = vb ? ldf(vb + e) : 0.f;
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = ldf(v + (size_t)min(j, n - 1) * ld + e) + b;
    if (v_in) {
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = (1.0f - lam) * x[j] + lam * ldf(v_in + (size_t)min(j, n - 1) * nv + e);
    }
    if (v_out) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (j < n) stf(v_out + (size_t)j * nv + e, x[j]);
    }
    if (run) {
      const int blk = slot0 / bs, off = slot0 - blk * bs;
      stv<8>(vc + (((size_t)blk * G + g) * Dv + c) * bs + off, x);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (j >= n) break;
        const int blk = slots[j] / bs, off = slots[j] - blk * bs;
        stf(vc + (((size_t)blk * G + g) * Dv + c) * bs + off, x[j]);
      }
    }
  }
}

// Tokens per workgroup of the value rows: one while all workgroups run at once, else eight
static int value_rows(int tokens) { return tokens <= 1024 ? 1 : 8; }

// --------------------------------------------------------------------------- attention input: row norm + half-split rotation + append
// From a fused projection row [.. | q (H D) | k (G D) | v (G Dv) | ..] (row stride ld, q at column `col0`):
// an RMS norm over the WHOLE q projection and over the whole k projection (all heads at once, plain
// weights qw [H D] / kw [G D]; both null: no norm), then the half-split rotation of the first 2 nrot
// dimensions of every head: dimension i < nrot is paired with dimension i + nrot, the pair turns by
// float(pos) * freqs[i] (cos and sin times `mag`).  q goes to q_out [T, H, D]; k and v (unchanged) are appended
// at slot_mapping to caches k [NB, G, BS, D] / v [NB, G, Dv, BS].  `v_from_k`: the row has no v columns and
// the values are the k columns as projected, before norm and rotation (Dv = D).  `pb` (or null): biases of the projected
// q | k | v columns, added before anything else; v_in / v_out / lam: values shared between layers (append_values).
// One workgroup per token; norms, angles and the rotation are float32.
template <typename T>
__global__ void __launch_bounds__(256) sm_rownorm_rope_kernel(
    void* __restrict__ q_out_, const void* __restrict__ qkv_, long ld, int col0, const void* __restrict__ qw_,
    const void* __restrict__ kw_, const float* __restrict__ freqs, int nrot, float eps, void* __restrict__ k_cache_,
    void* __restrict__ v_cache_, const int32_t* __restrict__ slot_mapping, const int32_t* __restrict__ positions, int H,
    int G, int D, int Dv, int bs, float mag, int v_from_k, const void* __restrict__ pb_, const void* __restrict__ v_in_,
    void* __restrict__ v_out_, float lam) {
  __shared__ float red[16];
  extern __shared__ float csn[];                   // cos | sin of the token's nrot angles
  const int t = blockIdx.x, tid = threadIdx.x;
  const float fpos = (float)positions[t];
  for (int i = tid; i < nrot; i += 256) {
    const float ang = fpos * freqs[i];
    csn[i] = cosf(ang) * mag;
    csn[nrot + i] = sinf(ang) * mag;
  }
  const T* q = (const T*)qkv_ + (size_t)t * ld + col0;
  const T* k = q + (size_t)H * D;
  const T* v = v_from_k ? k : k + (size_t)G * D;
  const T* qw = (const T*)qw_;
  const T* kw = (const T*)kw_;
  const int nq = H * D, nk = G * D, nv = G * Dv;
  const T* qb = (const T*)pb_;
  const T* kb = qb ? qb + nq : nullptr;
  auto at = [](const T* p, const T* b, int e) { return b ? ldf(p + e) + ldf(b + e) : ldf(p + e); };
  float iq = 1.f, ik = 1.f;
  if (qw) {
    float sq = 0.f, sk = 0.f;
    for (int e = tid; e < nq; e += 256) { const float x = at(q, qb, e); sq += x * x; }
    for (int e = tid; e < nk; e += 256) { const float x = at(k, kb, e); sk += x * x; }
    sq = block_sum(sq, red);
    sk = block_sum(sk, red);
    iq = 1.0f / sqrtf(sq / (float)nq + eps), ik = 1.0f / sqrtf(sk / (float)nk + eps);
  } else {
    __syncthreads();                               // csn is complete
  }
  const int slot = slot_mapping[t], blk = slot / bs, off = slot - blk * bs;
  T* q_out = (T*)q_out_ + (size_t)t * nq;
  T* kc = (T*)k_cache_;
  T* vc = (T*)v_cache_;
  for (int e = tid; e < nq + nk; e += 256) {
    const bool isq = e < nq;
    const int ee = isq ? e : e - nq;
    const T* src = isq ? q : k;
    const T* sb = isq ? qb : kb;
    const T* w = isq ? qw : kw;
    const float inv = isq ? iq : ik;
    const int hd = ee / D, d = ee - hd * D;
    float x = at(src, sb, ee);
    if (w) x = x * inv * ldf(w + ee);
    if (d < 2 * nrot) {
      const int i = d < nrot ? d : d - nrot;
      const int pe = d < nrot ? ee + nrot : ee - nrot;          // the pair's other dimension
      float y = at(src, sb, pe);
      if (w) y = y * inv * ldf(w + pe);
      const float cs = csn[i], sn = csn[nrot + i];
      x = d < nrot ? x * cs - y * sn : x * cs + y * sn;
    }
    if (isq) stf(q_out + ee, x);
    else stf(kc + (((size_t)blk * G + hd) * bs + off) * D + d, x);
  }
  append_values<T>(v, kb ? kb + nk : nullptr, v_in_ ? (const T*)v_in_ + (size_t)t * nv : nullptr,
                   v_out_ ? (T*)v_out_ + (size_t)t * nv : nullptr, lam, vc, blk, off, G, Dv, bs);
}

// The same with 8 consecutive dimensions per lane (16-byte loads and stores for bf16): head size, rotated
// half, row stride and first column are multiples of 8, so a lane's 8 dimensions and their 8 partners are
// one aligned piece each.
template <typename T>
__global__ void __launch_bounds__(256) sm_rownorm_rope_vec_kernel(
    void* __restrict__ q_out_, const void* __restrict__ qkv_, long ld, int col0, const void* __restrict__ qw_,
    const void* __restrict__ kw_, const float* __restrict__ freqs, int nrot, float eps, void* __restrict__ k_cache_,
    void* __restrict__ v_cache_, const int32_t* __restrict__ slot_mapping, const int32_t* __restrict__ positions, int H,
    int G, int D, int Dv, int bs, float mag, int v_from_k, const void* __restrict__ pb_, const void* __restrict__ v_in_,
    void* __restrict__ v_out_, float lam, int tokens, int vt) {
  __shared__ float red[32];
  extern __shared__ float csn[];                   // cos | sin of the token's nrot angles
  const int nq = H * D, nk = G * D, nv = G * Dv;
  const T* pb = (const T*)pb_;
  if ((int)blockIdx.x >= tokens) {                 // value rows: vt tokens of the batch
    const int t0 = (blockIdx.x - tokens) * vt;
    append_value_rows<T>((const T*)qkv_ + (size_t)t0 * ld + col0 + nq + (v_from_k ? 0 : nk), ld, pb ? pb + nq + nk : nullptr,
                         v_in_ ? (const T*)v_in_ + (size_t)t0 * nv : nullptr,
                         v_out_ ? (T*)v_out_ + (size_t)t0 * nv : nullptr, lam, (T*)v_cache_, slot_mapping + t0,
                         min(vt, tokens - t0), G, Dv, bs);
    return;
  }
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const float fpos = (float)positions[t];
  for (int i = tid; i < nrot; i += 256) {
    const float ang = fpos * freqs[i];
    csn[i] = cosf(ang) * mag;
    csn[nrot + i] = sinf(ang) * mag;
  }
  const T* q = (const T*)qkv_ + (size_t)t * ld + col0;
  const bool normed = qw_ != nullptr;
  float sq = 0.f, sk = 0.f;
  if (normed) {
    for (int e = tid * 8; e < nq + nk; e += 2048) {
      float x[8];
      ldv<8>(q + e, x);
      if (pb) add8(x, pb + e);
      float a = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) a += x[i] * x[i];
      if (e < nq) sq += a; else sk += a;
    }
    sq = wave_sum(sq);
    sk = wave_sum(sk);
    if (lane == 0) red[wid] = sq, red[4 + wid] = sk;
  }
  __syncthreads();                                 // also: csn is complete
  float iq = 1.f, ik = 1.f;
  if (normed) {
    sq = red[0] + red[1] + red[2] + red[3];
    sk = red[4] + red[5] + red[6] + red[7];
    iq = 1.0f / sqrtf(sq / (float)nq + eps), ik = 1.0f / sqrtf(sk / (float)nk + eps);
  }
  const int slot = slot_mapping[t], blk = slot / bs, off = slot - blk * bs;
  T* q_out = (T*)q_out_ + (size_t)t * nq;
  T* kc = (T*)k_cache_;
  for (int e = tid * 8; e < nq + nk; e += 2048) {
    const bool isq = e < nq;
    const int ee = isq ? e : e - nq;
    const T* w = (isq ? (const T*)qw_ : (const T*)kw_) + ee;
    const float inv = isq ? iq : ik;
    const int hd = ee / D, d = ee - hd * D;
    float x[8], g[8];
    ldv<8>(q + e, x);
    if (pb) add8(x, pb + e);
    if (normed) {
      ldv<8>(w, g);
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] *= inv * g[i];
    }
    if (d < 2 * nrot) {
      const bool first = d < nrot;
      const int po = first ? nrot : -nrot, i0 = first ? d : d - nrot;
      float y[8], gy[8];
      ldv<8>(q + e + po, y);
      if (pb) add8(y, pb + e + po);
      if (normed) {
        ldv<8>(w + po, gy);
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] *= inv * gy[i];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float cs = csn[i0 + i], sn = csn[nrot + i0 + i];
        x[i] = first ? x[i] * cs - y[i] * sn : x[i] * cs + y[i] * sn;
      }
    }
    if (isq) stv<8>(q_out + ee, x);
    else stv<8>(kc + (((size_t)blk * G + hd) * bs + off) * D + d, x);
  }
}

void sm_rownorm_rope(uintptr_t q_out, uintptr_t qkv, long ld, int col0, uintptr_t q_norm, uintptr_t k_norm,
                     uintptr_t freqs, int nrot, float eps, uintptr_t k_cache, uintptr_t v_cache, uintptr_t slot_mapping,
                     uintptr_t positions, int tokens, int H, int G, int D, int Dv, int bs, float mag, int v_from_k,
                     uintptr_t bias, uintptr_t v_in, uintptr_t v_out, float lam, int f32, uintptr_t stream) {
  if (tokens <= 0) return;
  DLLM_HOST_CHECK(H > 0 && G > 0 && D > 0 && Dv > 0 && bs > 0 && nrot >= 0 && 2 * nrot <= D && col0 >= 0 &&
                      ld >= col0 + (long)H * D + (long)G * D + (v_from_k ? 0 : (long)G * Dv) && (!v_from_k || Dv == D),
                  "rownorm_rope sizes");
  DLLM_HOST_CHECK(!v_from_k || (!bias && !v_in && !v_out), "rownorm_rope values from keys");
  DLLM_HOST_CHECK(q_out && k_cache && v_cache && (!q_norm == !k_norm) && (nrot == 0 || freqs), "rownorm_rope arguments");
  const int esz = f32 ? 4 : 2;
  if (D % 8 == 0 && nrot % 8 == 0 && ld % 8 == 0 && col0 % 8 == 0 && qkv % (8 * esz) == 0 && q_norm % (8 * esz) == 0 &&
      k_norm % (8 * esz) == 0 && q_out % (8 * esz) == 0 && k_cache % (8 * esz) == 0 && v_cache % (8 * esz) == 0 && bias % (8 * esz) == 0) {
    const int vt = value_rows(tokens);
    SM_DISPATCH(f32, sm_rownorm_rope_vec_kernel, dim3(tokens + (tokens + vt - 1) / vt), dim3(256), 2 * (size_t)nrot * sizeof(float), stream,
                (void*)q_out, (const void*)qkv, ld, col0, (const void*)q_norm, (const void*)k_norm, (const float*)freqs, nrot,
                eps, (void*)k_cache, (void*)v_cache, (const int32_t*)slot_mapping, (const int32_t*)positions, H, G, D, Dv, bs,
                mag, v_from_k, (const void*)bias, (const void*)v_in, (void*)v_out, lam, tokens, vt);
    return;
  }
  SM_DISPATCH(f32, sm_rownorm_rope_kernel, dim3(tokens), dim3(256), 2 * (size_t)nrot * sizeof(float), stream, (void*)q_out, (const void*)qkv, ld, col0,
              (const void*)q_norm, (const void*)k_norm, (const float*)freqs, nrot, eps, (void*)k_cache, (void*)v_cache,
              (const int32_t*)slot_mapping, (const int32_t*)positions, H, G, D, Dv, bs, mag, v_from_k,
              (const void*)bias, (const void*)v_in, (void*)v_out, lam);
}

// --------------------------------------------------------------------------- attention input: per-head norm, paired rotation, append
// From a fused projection row [.. | q (H D) | k (G D) | v (G Dv) | ..] (row stride ld, q at column `col0`): every q and
// k head is divided by its root mean square over D (times the plain weight qw / kw [D] shared by the heads, when
// given) before or -- `norm_last` -- after the rotation of its first 2 nrot dimensions, pairs (2i, 2i + 1) turning by
// float(pos) * freqs[i].  q is then multiplied by q_mul[h] (when given) and, with temp_every > 0, by
// 1 + temp_coef ln(floor((pos + 1) / temp_every) + 1).  q goes to q_out [T, H, D]; k and v (unchanged) are appended at
// slot_mapping to caches k [NB, G, BS, D] / v [NB, G, Dv, BS].  Norms, angles and factors are float32.  `pb` (or null):
// biases of the projected q | k | v columns, added before anything else; v_in / v_out / lam: values shared between
// layers (append_values).
//
// One workgroup per token; 8 consecutive dimensions per lane, a head on an aligned group of `lph` lanes (a power of
// two, 8 lph >= D): the mean square is a butterfly inside the group, the rotation stays inside a lane.
__device__ __forceinline__ float query_temp(int pos, float coef, int every) {
  return every > 0 ? 1.0f + coef * logf((float)((pos + 1) / every) + 1.0f) : 1.0f;
}

template <typename T>
__global__ void __launch_bounds__(256) sm_head_norm_rope_vec_kernel(
    void* __restrict__ q_out_, const void* __restrict__ qkv_, long ld, int col0, const void* __restrict__ qw_,
    const void* __restrict__ kw_, const float* __restrict__ freqs, int nrot, int norm_last, float eps,
    const float* __restrict__ q_mul, float temp_coef, int temp_every, void* __restrict__ k_cache_,
    void* __restrict__ v_cache_, const int32_t* __restrict__ slot_mapping, const int32_t* __restrict__ positions, int H,
    int G, int D, int Dv, int bs, int lph, const void* __restrict__ pb_, const void* __restrict__ v_in_,
    void* __restrict__ v_out_, float lam, int tokens, int vt) {
  extern __shared__ float csn[];                   // cos | sin of the token's nrot angles
  const int nq = H * D, nk = G * D, nv = G * Dv;
  const T* pb = (const T*)pb_;
  if ((int)blockIdx.x >= tokens) {                 // value rows: vt tokens of the batch
    const int t0 = (blockIdx.x - tokens) * vt;
    append_value_rows<T>((const T*)qkv_ + (size_t)t0 * ld + col0 + nq + nk, ld, pb ? pb + nq + nk : nullptr,
                         v_in_ ? (const T*)v_in_ + (size_t)t0 * nv : nullptr,
                         v_out_ ? (T*)v_out_ + (size_t)t0 * nv : nullptr, lam, (T*)v_cache_, slot_mapping + t0,
                         min(vt, tokens - t0), G, Dv, bs);
    return;
  }
  const int t = blockIdx.x, tid = threadIdx.x, pos = positions[t];
  const float fpos = (float)pos;
  for (int i = tid; i < nrot; i += 256) {
    const float ang = fpos * freqs[i];
    csn[i] = cosf(ang);
    csn[nrot + i] = sinf(ang);
  }
  const T* q = (const T*)qkv_ + (size_t)t * ld + col0;
  const int slot = slot_mapping[t], blk = slot / bs, off = slot - blk * bs;
  T* q_out = (T*)q_out_ + (size_t)t * nq;
  T* kc = (T*)k_cache_;
  const float qt = query_temp(pos, temp_coef, temp_every);
  const int sub = tid & (lph - 1), d = sub * 8;
  if (nrot > 0) __syncthreads();                   // uniform: csn is complete
  // every lane of a wave runs the same number of passes: the butterfly below needs whole groups
  for (int h0 = 0; h0 < H + G; h0 += 256 / lph) {
    const int head = h0 + tid / lph;
    const bool ok = head < H + G && d < D;
    const bool isq = head < H;
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = 0.f;
    if (ok) {
      ldv<8>(q + (size_t)head * D + d, x);
      if (pb) add8(x, pb + head * D + d);
    }
    float ss = 0.f;
    auto turn = [&]() {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int pr = (d >> 1) + i;
        if (pr < nrot) {
          const float cs = csn[pr], sn = csn[nrot + pr], a = x[2 * i], b = x[2 * i + 1];
          x[2 * i] = a * cs - b * sn;
          x[2 * i + 1] = b * cs + a * sn;
        }
      }
    };
    if (norm_last) turn();
#pragma unroll
    for (int i = 0; i < 8; ++i) ss += x[i] * x[i];
    for (int m = lph >> 1; m > 0; m >>= 1) ss += __shfl_xor(ss, m, 64);
    const float inv = 1.0f / sqrtf(ss / (float)D + eps);
    const T* w = (const T*)(isq ? qw_ : kw_);
    if (w && ok) {
      float g[8];
      ldv<8>(w + d, g);
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] *= inv * g[i];
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] *= inv;
    }
    if (!norm_last) turn();
    if (!ok) continue;
    if (isq) {
      const float f = q_mul ? qt * q_mul[head] : qt;
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] *= f;
      stv<8>(q_out + (size_t)head * D + d, x);
    } else {
      stv<8>(kc + (((size_t)blk * G + (head - H)) * bs + off) * D + d, x);
    }
  }
}

// The same for any head size: a wave per (token, head), the head's values in LDS.
template <typename T>
__global__ void __launch_bounds__(64) sm_head_norm_rope_kernel(
    void* __restrict__ q_out_, const void* __restrict__ qkv_, long ld, int col0, const void* __restrict__ qw_,
    const void* __restrict__ kw_, const float* __restrict__ freqs, int nrot, int norm_last, float eps,
    const float* __restrict__ q_mul, float temp_coef, int temp_every, void* __restrict__ k_cache_,
    void* __restrict__ v_cache_, const int32_t* __restrict__ slot_mapping, const int32_t* __restrict__ positions, int H,
    int G, int D, int Dv, int bs, int, const void* __restrict__ pb_, const void* __restrict__ v_in_,
    void* __restrict__ v_out_, float lam) {
  extern __shared__ float hv[];                    // the head's values [D]
  const int t = blockIdx.x, head = blockIdx.y, lane = threadIdx.x, pos = positions[t];
  const T* q = (const T*)qkv_ + (size_t)t * ld + col0;
  const T* pb = (const T*)pb_;
  const int slot = slot_mapping[t], blk = slot / bs, off = slot - blk * bs;
  if (head >= H + G) {                             // a value head
    const int g = head - H - G;
    const size_t v0 = ((size_t)t * G + g) * Dv;          // this head's place in the shared values
    append_values<T>(q + (size_t)(H + G) * D + (size_t)g * Dv, pb ? pb + (H + G) * D + g * Dv : nullptr,
                     v_in_ ? (const T*)v_in_ + v0 : nullptr, v_out_ ? (T*)v_out_ + v0 : nullptr, lam,
                     (T*)v_cache_ + (size_t)g * Dv * bs, blk * G, off, 1, Dv, bs);
    return;
  }
  const bool isq = head < H;
  const T* src = q + (size_t)head * D;
  const T* w = (const T*)(isq ? qw_ : kw_);
  T* dst = isq ? (T*)q_out_ + ((size_t)t * H + head) * D
               : (T*)k_cache_ + (((size_t)blk * G + (head - H)) * bs + off) * D;
  const float fpos = (float)pos;
  auto turn = [&]() {                              // a lane turns its own pairs
    for (int i = lane; i < nrot; i += 64) {
      const float ang = fpos * freqs[i], cs = cosf(ang), sn = sinf(ang), a = hv[2 * i], b = hv[2 * i + 1];
      hv[2 * i] = a * cs - b * sn;
      hv[2 * i + 1] = b * cs + a * sn;
    }
    __syncthreads();
  };
  for (int e = lane; e < D; e += 64) hv[e] = ldf(src + e) + (pb ? ldf(pb + head * D + e) : 0.f);
  __syncthreads();
  if (norm_last) turn();
  float ss = 0.f;
  for (int e = lane; e < D; e += 64) ss += hv[e] * hv[e];
  const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)D + eps);
  for (int e = lane; e < D; e += 64) hv[e] *= w ? inv * ldf(w + e) : inv;
  __syncthreads();
  if (!norm_last) turn();
  float f = 1.f;
  if (isq) {
    f = query_temp(pos, temp_coef, temp_every);
    if (q_mul) f *= q_mul[head];
  }
  for (int e = lane; e < D; e += 64) stf(dst + e, hv[e] * f);
}

void sm_head_norm_rope(uintptr_t q_out, uintptr_t qkv, long ld, int col0, uintptr_t q_norm, uintptr_t k_norm,
                       uintptr_t freqs, int nrot, int norm_last, float eps, uintptr_t q_mul, float temp_coef, int temp_every,
                       uintptr_t k_cache, uintptr_t v_cache, uintptr_t slot_mapping, uintptr_t positions, int tokens, int H,
                       int G, int D, int Dv, int bs, uintptr_t bias, uintptr_t v_in, uintptr_t v_out, float lam, int f32,
                       uintptr_t stream) {
  if (tokens <= 0) return;
  DLLM_HOST_CHECK(H > 0 && G > 0 && D > 0 && Dv > 0 && bs > 0 && nrot >= 0 && 2 * nrot <= D && col0 >= 0 && temp_every >= 0 &&
                      H + 2 * G <= 65535 && D <= 8192 && ld >= col0 + (long)H * D + (long)G * (D + Dv),
                  "head_norm_rope sizes");
  DLLM_HOST_CHECK(q_out && qkv && k_cache && v_cache && slot_mapping && positions && (nrot == 0 || freqs) &&
                      (!q_norm == !k_norm),
                  "head_norm_rope arguments");
  const int esz = f32 ? 4 : 2;
  if (D % 8 == 0 && D <= 512 && ld % 8 == 0 && col0 % 8 == 0 && qkv % (8 * esz) == 0 && q_norm % (8 * esz) == 0 &&
      k_norm % (8 * esz) == 0 && q_out % (8 * esz) == 0 && k_cache % (8 * esz) == 0 && v_cache % (8 * esz) == 0 && bias % (8 * esz) == 0) {
    int lph = 1;
    while (8 * lph < D) lph *= 2;
    const int vt = value_rows(tokens);
    SM_DISPATCH(f32, sm_head_norm_rope_vec_kernel, dim3(tokens + (tokens + vt - 1) / vt), dim3(256), 2 * (size_t)nrot * sizeof(float), stream,
                (void*)q_out, (const void*)qkv, ld, col0, (const void*)q_norm, (const void*)k_norm, (const float*)freqs, nrot,
                norm_last, eps, (const float*)q_mul, temp_coef, temp_every, (void*)k_cache, (void*)v_cache,
                (const int32_t*)slot_mapping, (const int32_t*)positions, H, G, D, Dv, bs, lph,
                (const void*)bias, (const void*)v_in, (void*)v_out, lam, tokens, vt);
    return;
  }
  SM_DISPATCH(f32, sm_head_norm_rope_kernel, dim3(tokens, H + 2 * G), dim3(64), (size_t)D * sizeof(float), stream,
              (void*)q_out, (const void*)qkv, ld, col0, (const void*)q_norm, (const void*)k_norm, (const float*)freqs, nrot,
              norm_last, eps, (const float*)q_mul, temp_coef, temp_every, (void*)k_cache, (void*)v_cache,
              (const int32_t*)slot_mapping, (const int32_t*)positions, H, G, D, Dv, bs, 0, (const void*)bias, (const void*)v_in,
              (void*)v_out, lam);
}

// --------------------------------------------------------------------------- averaged blocks of old keys
// For every block of `pool` positions whose LAST position p (p + 1 a multiple of pool) is a token of this
// step: the float32 mean of the block's keys and of its values AS THE CACHES HOLD THEM (k [NB, G, BS, D],
// v [NB, G, Dv, BS], read through the sequence's block table; earlier steps may have written some of them)
// goes to entry b = (p + 1) / pool - 1 of the averaged caches kp [NB, G, PB, D] / vp [NB, G, Dv, PB] (entry b
// at block b / PB of the same table, place b % PB).  One workgroup per (block that a chunk may complete, K/V
// head, sequence); V consecutive key dimensions per lane.  Runs after the step's append.
template <typename T, int V>
__global__ void __launch_bounds__(128) sm_pool_blocks_kernel(const void* __restrict__ k_cache_,
                                                             const void* __restrict__ v_cache_, void* __restrict__ kp_,
                                                             void* __restrict__ vp_,
                                                             const int32_t* __restrict__ block_tables, int max_blocks,
                                                             const int32_t* __restrict__ cu,
                                                             const int32_t* __restrict__ positions, int G, int D, int Dv,
                                                             int bs, int pb, int pool) {
  const int s = blockIdx.z, g = blockIdx.y;
  const int lo = cu[s], n = cu[s + 1] - lo;
  if (n <= 0) return;
  const int start = positions[lo], end = start + n - 1;          // positions of the chunk's tokens
  const int b = (start + pool) / pool - 1 + (int)blockIdx.x;     // first block whose last position is >= start
  if ((long)b * pool + pool - 1 > end) return;
  const int32_t* bt = block_tables + (size_t)s * max_blocks;
  const T* kc = (const T*)k_cache_;
  const T* vc = (const T*)v_cache_;
  const int pblk = bt[b / pb], poff = b % pb;
  T* kp = (T*)kp_ + (((size_t)pblk * G + g) * pb + poff) * D;
  T* vp = (T*)vp_ + ((size_t)pblk * G + g) * Dv * pb + poff;
  const float fpool = (float)pool;
  const int j0 = b * pool;
  for (int c = threadIdx.x * V; c < D; c += 128 * V) {
    float a[V];
#pragma unroll
    for (int i = 0; i < V; ++i) a[i] = 0.f;
    for (int j = j0; j < j0 + pool; ++j) {
      float x[V];
      ldv<V>(kc + (((size_t)bt[j / bs] * G + g) * bs + j % bs) * D + c, x);
#pragma unroll
      for (int i = 0; i < V; ++i) a[i] += x[i];
    }
#pragma unroll
    for (int i = 0; i < V; ++i) a[i] /= fpool;
    stv<V>(kp + c, a);
  }
  for (int c = threadIdx.x; c < Dv; c += 128) {
    float a = 0.f;
    for (int j = j0; j < j0 + pool; ++j) a += ldf(vc + (((size_t)bt[j / bs] * G + g) * Dv + c) * bs + j % bs);
    stf(vp + (size_t)c * pb, a / fpool);
  }
}

void sm_pool_blocks(uintptr_t k_cache, uintptr_t v_cache, uintptr_t kp_cache, uintptr_t vp_cache, uintptr_t block_tables,
                    int max_blocks, uintptr_t cu, uintptr_t positions, int seqs, int max_q_len, int G, int D, int Dv,
                    int bs, int pb, int pool, int f32, uintptr_t stream) {
  if (seqs <= 0 || max_q_len <= 0) return;
  DLLM_HOST_CHECK(G > 0 && G <= 65535 && seqs <= 65535 && D > 0 && Dv > 0 && bs > 0 && pb > 0 && pool > 0 &&
                      (long)pb * pool >= bs && max_blocks > 0 && k_cache && v_cache && kp_cache && vp_cache && cu && positions,
                  "pool_blocks arguments");
  const int esz = f32 ? 4 : 2;
  const bool vec = D % 8 == 0 && k_cache % (8 * esz) == 0 && kp_cache % (8 * esz) == 0;
  // a chunk of n tokens completes at most (n + pool - 1) / pool blocks
  SM_DISPATCH_V(f32, vec, sm_pool_blocks_kernel, dim3((max_q_len + pool - 1) / pool, G, seqs), dim3(128), 0, stream,
                (const void*)k_cache, (const void*)v_cache, (void*)kp_cache, (void*)vp_cache,
                (const int32_t*)block_tables, max_blocks, (const int32_t*)cu, (const int32_t*)positions, G, D, Dv, bs, pb,
                pool);
}

}  // namespace dllm
