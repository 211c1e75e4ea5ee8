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

// Up to 64 (token, choice) pairs: where they lie sorted by expert, from the choices themselves, a pair per lane.  A launch that made counts, offsets and
// slot lists of them stood between the router and the experts; a wave has them from one load and two ballots, in place of the two
// dependent loads of those: 5 us a layer, and the experts' launches no longer (16 rows, traced 279 + 138 us either way; 4 rows 215 + 108
// -> 208 + 106).
constexpr int kPickPairs = 64;
struct MoePick {
  int cnt, off, list;       // the expert's pairs, the slot of the first of them, lane i: the token of the i-th
};
__device__ __forceinline__ int moe_pair(const int* __restrict__ ids, int pairs, int lane) {
  const int id = ids[lane < pairs ? lane : 0];
  return lane < pairs ? id : 0x7fffffff;
}
__device__ __forceinline__ MoePick moe_pick(const int* __restrict__ ids, int pairs, int top, int e, int lane) {
  const int id = moe_pair(ids, pairs, lane);
  const uint64_t mine = __ballot(id == e), below = (1ull << lane) - 1;
  MoePick r;
  r.cnt = __popcll(mine);
  r.off = __popcll(__ballot(id < e));
  // (every lane sends to a place of its own: the expert's pairs first)
  const int to = id == e ? __popcll(mine & below) : r.cnt + __popcll(~mine & below);
  r.list = __builtin_amdgcn_ds_permute(4 * to, lane / top);
  return r;
}
// the slot of pair i (uniform), id: moe_pair of the lane
__device__ __forceinline__ int moe_slot(int id, int i) {
  const int own = __builtin_amdgcn_readlane(id, i);
  return __popcll(__ballot(id < own)) + __popcll(__ballot(id == own) & ((1ull << i) - 1));
}

}  // namespace dllm
