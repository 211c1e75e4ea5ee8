// A token's choice of experts from its router logits: softmax -> top-k -> renormalise, by one thread.
#pragma once
#include "common.h"

namespace dllm {

// p: the logits' f32 sums, rounded to bf16 here as a product's output is
template <int E>
__device__ __forceinline__ void moe_top(float (&p)[E], int t, int k, float* __restrict__ topk_w, int* __restrict__ topk_ids) {
  float mx = -INFINITY;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    p[e] = bf2f(f2bf(p[e]));
    mx = fmaxf(mx, p[e]);
  }
  float sum = 0.f;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    p[e] = __expf(p[e] - mx);
    sum += p[e];
  }
  // (places known to the compiler throughout: an array that is indexed at run time lies in scratch memory)
  int ids[8];
  float ws[8];
  float tot = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    if (j >= k) break;
    int best = 0;
    float bv = -1.f;
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (p[e] > bv) { bv = p[e]; best = e; }
    ids[j] = best;
    ws[j] = bv / sum;
    tot += ws[j];
#pragma unroll
    for (int e = 0; e < E; ++e) p[e] = e == best ? -2.f : p[e];
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    if (j >= k) break;
    topk_ids[t * k + j] = ids[j];
    topk_w[t * k + j] = ws[j] / tot;
  }
}

}  // namespace dllm
