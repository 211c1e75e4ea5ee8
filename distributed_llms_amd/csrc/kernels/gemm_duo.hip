// Decode products of 65 to 512 rows: C[M, N] = A[M, K] . B[N, K]^T, bf16 in, f32 accumulate, as split-K slabs or through a SwiGLU.
// Tiles of 128 / 192 / 256 rows x 128 columns, four waves that multiply and four that stage.
//
// What bounds it: the requests of a CU for lines of 128 bytes, some 256 of them under way whatever the ring's depth, cache policy or
// number of waves.  A K-tile of 256 activation rows takes 0.27 us of them (out of the L2), its 128 weight rows 0.55 (memory), and the two add up:
// 28672 x 4096 with nothing but its staging loads 50 us, 36 without the activations.  gemm_wide, whose eight waves multiply and
// stage, took 62-69 us for it: a wave that waits for room to issue a load issues no products either, and loads strewn among
// products come as activations and weights in turn, which alone makes the staging 56 us instead of 50.  Here the waves that stage
// issue a K-tile's activations, then its weights, as soon as a slot is free, and those that multiply wait for nothing but
// the K-tile's one barrier: 57-62 us.  us, gemm_wide / this, slabs with the sum and norm behind them:
//   28672 x 4096, SwiGLU   M = 96 / 128 / 192         46.3 / 46.8 / 53.6 -> 44.5 / 45.8 / 52.8
//   4096 x 14336           192 / 256                  35.3 / 40.1 -> 34.4 / 38.6
//   4096 x 4096            160 / 256 / 300 / 512      16.0 / 18.4 / 31.9 / 28.5 -> 15.1 / 17.6 / 23.6 / 27.4
//   6144 x 4096            160 / 200 / 256            18.5 / 22.2 / 23.4 -> 18.2 / 19.7 / 21.5
//   8192 x 8192            160 / 256                  40.3 / 45.4 -> 39.5 / 43.6
// It needs the CUs: 2048 x 2048 in 64 workgroups, 256 rows 12.0 -> 14.1 (ops/gemm.duo_fits has the rule).
//
// The order of a K-tile: the waves that multiply hold its K-half 0 in registers, read K-half 1 among half 0's products, and at the barrier
// behind these every wave has the whole K-tile in registers (its slot is free) and the next one has landed (the staging waves'
// counted vmcnt); the next one's K-half 0 is read among half 1's products.  Three slots: two are 25 % slower (256 rows 74.8
// us), four and five of shorter tiles no faster.
//
// Slabs.  Slices under 24 K-tiles store them through to memory (sc1): the launch that sums them runs on other XCDs and waits for what the
// kernel's end writes back otherwise (6144 x 4096 at 256 rows with its sum 22.6 -> 21.5, 4096 x 4096 18.0 -> 17.6), and leave
// the weights in the caches' default policy; in longer ones the stores are a smaller part and nontemporal weights gain more (4096 x 14336
// 41.4 -> 38.6).
// The sums have gemm_wide's order: equal bits.  A SwiGLU that gemm_pp would run (like_pp) has that kernel's instead: K from its start on every
// XCD, gate and up rounded to bf16 in front of the SiLU.  us, gemm_pp / this / with gemm_wide's bits, 200 and 256 rows: 28672 x 4096
// 60.9 / 58.2 / 58.1 and 62.1 / 60.6 / 59.5, 32768 x 4096 71.3 / 65.6 / 58.6 and 68.7 / 66.6 / 61.8, 28672 x 3072 52.9 / 51.6 / 51.7 and 49.4 / 48.1 / 48.6,
// 27648 x 5120 74.5 / 72.0 / 72.8 and 77.8 / 76.3 / 76.9.
//
// An XCD has the column tiles of a slice next to each other: its L2 then holds one slice of the activations, where the slices of a column tile
// beside each other had every XCD fetch all of them (7 MiB of 4096 x 14336 at 256 rows, eight times, beside 112 MiB of weights).  With the sum
// and norm behind them, 4096 x 14336 at 256 / 384 / 512 rows 42.4 / 56.5 / 64.8 -> 41.2 / 54.3 / 60.2 us, 1024 x 8192 at 512 in 8 slices 19.9 ->
// 17.8, 2560 x 7680 at 400 27.6 -> 26.4; in a decode step of 256 requests on 8B the down projection 40.7 -> 35.8.
#include "gemm_pp_common.h"
#include "launchers.h"

namespace dllm {

// Row tile 32 RT.  GLU: SwiGLU C [M, N / 2] of B = [gate; up] in alternating 16-row groups (pp_b_row), else slabs P [S, M, N].  LONG: long slices.
template <int RT, bool GLU, bool LONG>
__global__ void __launch_bounds__(512, 1) gemm_duo_kernel(const bf16* __restrict__ B, const bf16* __restrict__ A, int M, int N, int K,
                                                          int kts, int nsplit, bool like_pp, bf16* __restrict__ C, float* __restrict__ P) {
  constexpr int BM = 32 * RT, BN = 128, CT = 4, TM = 16 * RT, TN = 64, NB = 3;   // waves that multiply: 2 x 2 of TM x TN
  constexpr int SLOT = (BM + BN) * PBK;
  constexpr int GA = BM / 32, GB = BN / 32, G = GA + GB;       // pieces of 8 rows per staging wave and K-tile
  static_assert(NB * SLOT * 2 <= 160 * 1024 && (NB - 1) * G <= 63, "ring");
  __shared__ __attribute__((aligned(16))) bf16 smem[NB * SLOT];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int b = blockIdx.x;
  {   // row tiles of a column tile, then column tiles of a slice on one XCD
    const int q = gridDim.x >> 3, r = gridDim.x & 7, x = b & 7;
    b = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + (b >> 3);
  }
  const int mtiles = (M + BM - 1) / BM;
  const int m_t = b % mtiles, rest = b / mtiles, ntiles = N / BN, split = rest / ntiles, n_t = rest - split * ntiles;
  const int m0 = m_t * BM;
  const int ks0 = split * kts, nt = min(K / PBK, ks0 + kts) - ks0;               // >= 1 (host)
  if (wv >= 4) {
    const int lw = wv - 4;
    // (unsplit: K from another place on each XCD, gemm_wide's rotation)
    const int rot = !like_pp && nsplit == 1 && mtiles == 1 && nt >= 16 ? ((int)(blockIdx.x & 7) * nt) >> 3 : 0;
    uint32_t off[G];
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const bool act = j < GA;
      const int q = act ? lw * GA + j : lw * GB + j - GA, r = 8 * q + (lane >> 3);
      const int row = act ? min(m0 + r, M - 1) : pp_b_row<BN, GLU>(8 * q, n_t, N / 2) + (lane >> 3);
      off[j] = (uint32_t)row * (uint32_t)(K * 2) + (uint32_t)(pswz(r, lane & 7) * 16);
    }
    const auto ra = __builtin_amdgcn_make_buffer_rsrc((void*)(reinterpret_cast<const char*>(A) + (size_t)ks0 * 128), (short)0,
                                                      (int)(unsigned)((long)M * K * 2 - (long)ks0 * 128), 0x00020000);
    const auto rb = __builtin_amdgcn_make_buffer_rsrc((void*)(reinterpret_cast<const char*>(B) + (size_t)ks0 * 128), (short)0,
                                                      (int)(unsigned)((long)N * K * 2 - (long)ks0 * 128), 0x00020000);
    auto stage = [&](int slot, int t) {
      const int k = (t + rot >= nt ? t + rot - nt : t + rot) * 128;
      bf16* base = smem + slot * SLOT;
#pragma unroll
      for (int j = 0; j < GA; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_vptr_p)(base + (lw * GA + j) * 512), 16, (int)off[j], k, 0, 0);
#pragma unroll
      for (int j = 0; j < GB; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_vptr_p)(base + BM * PBK + (lw * GB + j) * 512), 16, (int)off[GA + j], k, 0,
                                                 GLU || LONG ? 2 : 0);
    };
#pragma unroll
    for (int j = 0; j < NB; ++j)
      if (j < nt) stage(j, j);
    if (nt >= NB) pp_vm<(NB - 1) * G>();
    else pp_vm<0>();
    __builtin_amdgcn_s_barrier();                      // K-tile 0 has landed
    int slot = 0;
    for (int t = 0; t < nt; ++t) {
      if (t + NB <= nt) pp_vm<(NB - 2) * G>();         // K-tile t + 1
      else pp_vm<0>();
      __builtin_amdgcn_s_barrier();
      if (t + NB < nt) stage(slot, t + NB);
      slot = slot == NB - 1 ? 0 : slot + 1;
    }
    return;
  }
  const int wm = wv >> 1, wn = wv & 1;
  const uint32_t lds_base = (uint32_t)(size_t)(lds_vptr_p)smem;
  uint32_t lane_off[2];
#pragma unroll
  for (int kh = 0; kh < 2; ++kh)
    lane_off[kh] = (uint32_t)((lane & 15) * 128 + ((4 * kh + (lane >> 4)) ^ (((lane & 15) >> 1) & 7)) * 16);
  const uint32_t a_off = lds_base + (uint32_t)(wm * TM * 128), b_off = lds_base + (uint32_t)(BM * 128 + wn * TN * 128);
  f32x4 acc[RT][CT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+a"(acc[i][j]));
    }
  // fragments of a K-half: CT of B, then RT of A; one is read behind every EV products
  constexpr int NMF = RT * CT, NR = RT + CT, EV = 2 * NR <= NMF ? 2 : 1;
  bf16x8 f0[NR], f1[NR];
  auto rd = [&](bf16x8& f, uint32_t at, auto mc) {
    constexpr int m = decltype(mc)::value;
    if constexpr (m < CT) f = pp_frag<m * 2048>(at + b_off);
    else f = pp_frag<(m - CT) * 2048>(at + a_off);
  };
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  pp_static_for<NR>([&](auto mc) { rd(f0[decltype(mc)::value], lane_off[0], mc); });
  __builtin_amdgcn_sched_barrier(0);
  int slot = 0;
  for (int t = 0; t < nt; ++t) {
    const int nslot = slot == NB - 1 ? 0 : slot + 1;
    const uint32_t at1 = (uint32_t)(slot * SLOT * 2) + lane_off[1], at0 = (uint32_t)(nslot * SLOT * 2) + lane_off[0];
    pp_static_for<NMF>([&](auto ic) {
      constexpr int i = decltype(ic)::value, r = i / CT, c = i % CT;
      if constexpr (c == 0) {                          // a row's A fragment (the first one's: every B) has landed
        constexpr int w = (RT - 1 - r) + (i / EV < NR ? i / EV : NR);
        pp_lgkm<(w > 15 ? 15 : w)>();
      }
      acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f0[c], f0[CT + r], acc[r][c], 0, 0, 0);
      if constexpr (i % EV == EV - 1 && i / EV < NR) rd(f1[i / EV], at1, std::integral_constant<int, i / EV>{});
      __builtin_amdgcn_sched_barrier(0);
    });
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    // (past the last K-tile: what its slot holds, never used)
    pp_static_for<NMF>([&](auto ic) {
      constexpr int i = decltype(ic)::value, r = i / CT, c = i % CT;
      acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f1[c], f1[CT + r], acc[r][c], 0, 0, 0);
      if constexpr (i % EV == EV - 1 && i / EV < NR) rd(f0[i / EV], at0, std::integral_constant<int, i / EV>{});
      __builtin_amdgcn_sched_barrier(0);
    });
    slot = nslot;
  }
  // the reads past the last K-tile: their registers are nobody else's before they have landed
#pragma unroll
  for (int i = 0; i < NR; ++i) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f0[i])::"memory");

  // acc[r][c] lane l: C[m0 + wm TM + 16 r + (l & 15)][columns 16 c + 4 (l >> 4) .. + 3 of the wave's 64]; two fragments' 4-column pieces
  // are exchanged between 16-lane rows, so that a lane stores 8 consecutive columns (gemm_pp.hip)
  const int lr = lane & 15, lq = lane >> 4;
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  [[maybe_unused]] const auto rp = __builtin_amdgcn_make_buffer_rsrc((void*)P, (short)0, 0x7fffffff, 0x00020000);
#pragma unroll
  for (int r = 0; r < RT; ++r) {
#pragma unroll
    for (int c = 0; c < CT; ++c) asm volatile("" : "+a"(acc[r][c]));
    const int m = m0 + wm * TM + r * 16 + lr;
#if DLLM_PART_TYPE != 2
    if constexpr (!GLU) {
#pragma unroll
      for (int c = 0; c < CT; ++c)
        if (m < M) part_store4(P, ((size_t)split * M + m) * N + n_t * BN + wn * TN + 16 * c + 4 * lq, acc[r][c]);
      continue;
    }
#endif
    constexpr int NQ = GLU ? CT / 2 : CT;
    u32x2 q[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      if constexpr (GLU) {
        bf16x4 h;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          float g = acc[r][2 * i][v], u = acc[r][2 * i + 1][v];
          if (like_pp) g = bf2f(f2bf(g)), u = bf2f(f2bf(u));
          h[v] = f2bf(silu_f(g) * u);
        }
        q[i] = __builtin_bit_cast(u32x2, h);
      } else {
        f16x4 h;
#pragma unroll
        for (int v = 0; v < 4; ++v) h[v] = (_Float16)(acc[r][i][v] * kPartScale);
        q[i] = __builtin_bit_cast(u32x2, h);
      }
    }
#pragma unroll
    for (int pr = 0; pr < NQ / 2; ++pr) {
      u32x2 x = q[2 * pr], y = q[2 * pr + 1];
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const auto sw = __builtin_amdgcn_permlane16_swap(x[d], y[d], false, false);
        x[d] = sw[0];
        y[d] = sw[1];
      }
      if (m < M) {
        const u32x4 o = {x[0], x[1], y[0], y[1]};
        const int col = 32 * pr + 16 * (lq & 1) + 8 * (lq >> 1);
        if constexpr (GLU) *reinterpret_cast<u32x4*>(C + (size_t)m * (N / 2) + n_t * (BN / 2) + wn * (TN / 2) + col) = o;
        else __builtin_amdgcn_raw_buffer_store_b128(o, rp, (int)((((size_t)split * M + m) * N + n_t * BN + wn * TN + col) * 2), 0, LONG ? 0 : 16);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// glu: SwiGLU c [m, n / 2] of b = [gate; up], unsplit; else slabs [S, m, n] of `splits` K slices in ws (S > 1).  bm: row tile 128, 192 or 256.
// like_pp: a SwiGLU with gemm_pp's bits, else with gemm_wide's.  Returns the number of slices S.
int gemm_duo(uintptr_t c, uintptr_t a, uintptr_t b, uintptr_t ws, long ws_floats, int M, int N, int K, int splits, bool glu, int bm,
             uintptr_t stream, bool like_pp) {
  DLLM_HOST_CHECK(M >= 1 && N > 0 && N % 128 == 0 && K % PBK == 0 && K >= PBK && splits >= 1, "N a multiple of 128, K of 64");
  DLLM_HOST_CHECK((long)M * K * 2 < (1L << 32) && (long)N * K * 2 < (1L << 32), "operands must be < 4 GiB");
  DLLM_HOST_CHECK(bm == 128 || bm == 192 || bm == 256, "row tile 128, 192 or 256");
  const int kt = K / PBK, kts = (kt + splits - 1) / splits, S = (kt + kts - 1) / kts;
  DLLM_HOST_CHECK(glu ? S == 1 && c : S > 1, "a SwiGLU unsplit, slabs of a K split");
  DLLM_HOST_CHECK(glu || (ws != 0 && (long)S * M * N <= ws_floats && (long)S * M * N < (1L << 29)), "split-K workspace too small");
  DLLM_HOST_CHECK((a | b) % 16 == 0 && (c | ws) % 16 == 0, "alignment");
  const long grid = (long)(N / 128) * S * ((M + bm - 1) / bm);
  DLLM_HOST_CHECK(grid < (1L << 31), "grid");
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(512), 0, reinterpret_cast<hipStream_t>(stream), (const bf16*)b, (const bf16*)a, M,
                       N, K, kts, S, like_pp, (bf16*)c, (float*)ws);
  };
#define DLLM_DUO(RT_)                                     \
  do {                                                    \
    if (glu) go(gemm_duo_kernel<RT_, true, true>);        \
    else if (kts >= 24) go(gemm_duo_kernel<RT_, false, true>); \
    else go(gemm_duo_kernel<RT_, false, false>);          \
  } while (0)
  if (bm == 128) DLLM_DUO(4);
  else if (bm == 192) DLLM_DUO(6);
  else DLLM_DUO(8);
#undef DLLM_DUO
  DLLM_HIP_CHECK(hipGetLastError());
  return S;
}

}  // namespace dllm
