// Prompt GEMM of fp8 (W8A8) operands: C = diag(sa) A B^T diag(sb), A [M, K] and B [N, K] OCP e4m3 bytes, per-row scales, f32
// accumulate, bf16 out, or its SwiGLU with B = [Bg; Bu] -- gemm_wide_fp8's products in its order (equal bits) for prompt sizes.
//
// What bounds it.  gemm_wide_fp8's 256 x 128 tile of eight waves reads 128 KB of fragments from LDS per K-tile of 128 and stages 48 KB
// into it, 0.6 us of the LDS's 0.3 TB/s per CU against 0.43 us of MFMAs at the nominal rate: a K-tile took 0.75 us (1.9 PFLOP/s).  Here,
// as in gemm_pf (gemm_pp.hip, whose tile walk, staging and stores these are), four waves hold 128 x 128 of a 256 x 256 tile: the same
// fragment bytes for twice the products, and two thirds of the staged ones.  An e4m3 K-tile of 128 has the bytes of a bf16 one of 64
// and the cycles of it, so the ring and its two barriers per K-tile are gemm_pf's; but v_mfma_f32_16x16x128_f8f6f4 takes
// 32 bytes per lane and operand, all of the K-tile at once, so the fragments of two K-tiles (2 x 128 registers) do not fit beside
// 256 accumulators: Pf8Sched orders a K-tile's products so that one set is enough.
// us, before -> now, 2560 rows: 28672 x 4096 with its SwiGLU 315 -> 221, 4096 x 14336 169 -> 103 (160 rows: one full round), 6144 x
// 4096 68 -> 48, 4096 x 4096 54 -> 35; 28672 x 4096 at 8192 rows 956 -> 629 (3.06 PFLOP/s, at a clock that falls as the matrix
// cores fill: a K-tile takes 1.0 us while half of the CUs are busy and 1.29 on all of them).
// The scales of a tile's rows and columns come into LDS beside its first K-tile, 2 KB: loaded in the epilogue they would
// wait for every staged piece in flight.
// Row tile 32 RT (160 .. 256): the shorter ones for grids that they fit into fewer or cheaper rounds (ops/quant._pf8_plan); 160 rows
// leave room for a third slot.
#include "gemm_pp_common.h"
#include "launchers.h"

#include <atomic>
#include <type_traits>

namespace dllm {

namespace {
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));

// One K-tile of 128 is NMF = 8 RT products of a 16 x 128 by 128 x 16 fragment.  A wave's RT fragments of A come in two parts,
// Aa (RA) and Ab (RB), its 8 of B in two of four, F and S, and the products go Aa F, Aa S, Ab S, Ab F -- the last two by columns
// -- so that the fragments fall free in the order in which the next K-tile, with F and S exchanged, asks for them: each is read
// into its own registers again, and one set of fragments is enough (two do not fit beside 256 accumulators).
// Read m of the next K-tile (two of 16 bytes per fragment: Aa, its F, its S, Ab) goes out behind product pos(m); those past the
// last product in the K-tile itself.
template <int RT>
struct Pf8Sched {
  static constexpr int RA = (RT + 1) / 2, RB = RT / 2, NMF = 8 * RT, NRD = 2 * RT + 16;
  static constexpr int Q2 = 4 * RA, Q3 = 8 * RA, Q4 = 8 * RA + 4 * RB;
  static constexpr int L = NMF - 24;                           // the next K-tile has landed: reads from here on
  static constexpr int last_use(int m) {                       // of the fragment that read m replaces
    const int f = m / 2;
    if (f < RA) return Q2 + 4 * f + 3;
    if (f < RA + 4) return Q3 + RB * (f - RA) + RB - 1;        // the next F is this S
    if (f < RA + 8) return Q4 + RB * (f - RA - 4) + RB - 1;
    return Q4 + 3 * RB + (f - RA - 8);
  }
  static constexpr int pos(int m) {
    int p = L;
    for (int k = 0; k <= m; ++k) p = p + 1 > last_use(k) ? p + 1 : last_use(k);
    return p;
  }
  static constexpr int read_at(int p) {                        // the read behind product p (next K-tile's from NMF on), or -1
    for (int m = 0; m < NRD; ++m)
      if (pos(m) == p) return m;
    return -1;
  }
  static constexpr int issued(int p) {                         // reads out before product p
    int n = 0;
    for (int m = 0; m < NRD; ++m) n += pos(m) < p;
    return n;
  }
  static constexpr int early() { return issued(NMF); }
  static constexpr int IB1 = pos(NRD - 1) - NMF + 5;           // every read of the K-tile has returned: its slot is free
  // product i of the first row waits for column i's fragment, and with it for all of Aa
  static constexpr int wait(int i) {
    const int n = issued(NMF + i) - 1 - (2 * RA + 2 * i + 1);
    return n < 0 ? 0 : n > 15 ? 15 : n;
  }
  static constexpr int row(int i) { return i < Q3 ? (i % Q2) / 4 : RA + (i < Q4 ? i - Q3 : i - Q4) % RB; }
  static constexpr int col(int i, int par) {                   // par 1: F and S exchanged
    const bool first = i < Q2 || i >= Q4;
    const int c = i < Q3 ? i % 4 : (i < Q4 ? i - Q3 : i - Q4) / RB;
    return (first != (par != 0) ? 0 : 4) + c;
  }
  static_assert(IB1 > 0 && IB1 < Q2 && L > IB1, "a K-tile's reads end in its first part");
};
}  // namespace

template <bool SWIGLU, int RT>
__global__ void __launch_bounds__(256, 1) gemm_pf8_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B,
                                                          const float* __restrict__ sa, const float* __restrict__ sb,
                                                          bf16* __restrict__ C, int M, int N, int K) {
  using SC = Pf8Sched<RT>;
  constexpr int NW = 4, NWN = 2, TM = 16 * RT, BM = 2 * TM, BN = 256, TN = BN / NWN, CT = TN / 16, BK = 128;
  constexpr int SLOT = (BM + BN) * BK, NB = RT > 5 ? 2 : 3;    // bytes
  constexpr int GA = BM * BK / 1024 / NW, GB = BN * BK / 1024 / NW, G = GA + GB;
  constexpr int OUTW = SWIGLU ? BN / 2 : BN;
  constexpr int NMF = SC::NMF, IB1 = SC::IB1, IB3 = SC::L;
  constexpr int GE = (NMF - 2 - IB1) / G > 1 ? (NMF - 2 - IB1) / G : 1;
  constexpr int PB3 = (IB3 - IB1 - 1) / GE + 1 < G ? (IB3 - IB1 - 1) / GE + 1 : G;   // pieces issued by IB3
  constexpr int VC = (NB - 2) * G + PB3;
  static_assert(CT == 8 && IB1 + 1 + GE * (G - 1) < NMF && VC <= 63, "schedule");
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  constexpr int SCALES = 512;                          // floats per tile: 256 of its rows, 256 of its columns
  static_assert(NB * SLOT + 2 * SCALES * 4 <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(16))) uint8_t smem[NB * SLOT + 2 * SCALES * 4];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wv / NWN, wn = wv % NWN;
  const int ldc = SWIGLU ? N / 2 : N;
  const int mtiles = (M + BM - 1) / BM;
  const int ntn = N / BN, tiles = ntn * mtiles;
  const int P = gridDim.x;                             // a multiple of 8 (host)
  const int w = (int)(blockIdx.x & 7) * (P >> 3) + (int)(blockIdx.x >> 3);
  const int mine = w < tiles ? (tiles - 1 - w) / P + 1 : 0;
  if (mine == 0) return;                               // uniform: before any load or barrier
  constexpr int GM = 8;                                // row tiles per group of the tile order
  const int nt = K / BK, per = GM * ntn;
  auto tile_mn = [&](int tau, int& m_t, int& n_t) {
    const int g = tau / per, first = g * GM, gsz = min(mtiles - first, GM), q = tau - g * per;
    m_t = first + q % gsz;
    n_t = q / gsz;
  };

  const __amdgpu_buffer_rsrc_t rsA =
      __builtin_amdgcn_make_buffer_rsrc((void*)A, (short)0, (int)(unsigned)((long)M * K), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsB =
      __builtin_amdgcn_make_buffer_rsrc((void*)B, (short)0, (int)(unsigned)((long)N * K), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsC =
      __builtin_amdgcn_make_buffer_rsrc((void*)C, (short)0, (int)(unsigned)((long)M * ldc * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsSa = __builtin_amdgcn_make_buffer_rsrc((void*)sa, (short)0, M * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsSb = __builtin_amdgcn_make_buffer_rsrc((void*)sb, (short)0, N * 4, 0x00020000);
  uint32_t chunk_q[2], offB[2], offA[GA], offBv[GB];
#pragma unroll
  for (int par = 0; par < 2; ++par) {
    chunk_q[par] = (uint32_t)(pswz(8 * par + (lane >> 3), lane & 7) * 16);
    offB[par] = (uint32_t)(lane >> 3) * (uint32_t)K + chunk_q[par];
  }
  int s_i = 0, s_kt = 0;
  // staging side onto my i-th tile: its rows' offsets (past M: the last row again) and its scales, into the buffer that the
  // tile before last has left (nt >= 4: every wave has passed a barrier of the tile in between since)
  auto set_stage = [&](int i) {
    int m_t, n_t;
    tile_mn(w + i * P, m_t, n_t);
    const int r0 = m_t * BM;
#pragma unroll
    for (int j = 0; j < GA; ++j) {
      const int q = wv * GA + j, r = 8 * q + (lane >> 3);
      offA[j] = (uint32_t)min(r0 + r, M - 1) * (uint32_t)K + chunk_q[q & 1];
    }
#pragma unroll
    for (int j = 0; j < GB; ++j)
      offBv[j] = (uint32_t)pp_b_row<BN, SWIGLU>(8 * (wv * GB + j), n_t, N / 2) * (uint32_t)K + offB[j & 1];
    uint8_t* sc = smem + NB * SLOT + (i & 1) * SCALES * 4 + wv * 256;
    const int j = 64 * wv + lane;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsSa, (lds_vptr_p)sc, 4, min(r0 + j, M - 1) * 4, 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsSb, (lds_vptr_p)(sc + 1024), 4, pp_b_row<BN, SWIGLU>(j, n_t, N / 2) * 4, 0, 0, 0);
  };
  // piece p of the staging K-tile into ring slot `slot`
  auto piece = [&](int slot, int p) {
    uint8_t* base = smem + slot * SLOT;
    if (p < GA) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsA, (lds_vptr_p)(base + (wv * GA + p) * 1024), 16, (int)offA[p], s_kt * BK, 0,
                                               0);
    } else {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsB, (lds_vptr_p)(base + BM * BK + (wv * GB + p - GA) * 1024), 16,
                                               (int)offBv[p - GA], s_kt * BK, 0, 0);
    }
  };
  // next staging K-tile; past my last tile: K-tile nt - 1 of it again (into a slot nobody reads again, so that every K-tile
  // issues exactly G pieces: static vmcnt counts)
  auto advance = [&]() {
    if (++s_kt == nt) {
      if (s_i + 1 < mine) {
        s_kt = 0;
        set_stage(++s_i);
      } else {
        s_kt = nt - 1;
      }
    }
  };

  // a lane's 32 bytes of a fragment's row: chunks 2 (l >> 4) and the next, of row l & 15 (K in the order of gemm_wide_fp8)
  const uint32_t lds_base = (uint32_t)(size_t)(lds_vptr_p)smem;
  uint32_t a_off[2], b_off[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint32_t l = (uint32_t)((lane & 15) * 128 + ((2 * (lane >> 4) + h) ^ (((lane & 15) >> 1) & 7)) * 16);
    a_off[h] = lds_base + l + wm * TM * BK;
    b_off[h] = lds_base + l + BM * BK + wn * TN * BK;
  }
  f32x4 acc[RT][CT];
  i32x4 fa[RT][2], fb[CT][2];
  // read m of the K-tile of parity PAR in the slot `at` bytes on
  auto rd = [&](uint32_t at, auto mc, auto parc) {
    constexpr int m = decltype(mc)::value, f = m / 2, h = m % 2, par = decltype(parc)::value;
    if constexpr (f < SC::RA || f >= SC::RA + 8) {
      constexpr int r = f < SC::RA ? f : f - 8;
      fa[r][h] = __builtin_bit_cast(i32x4, pp_frag<r * 16 * BK>(at + a_off[h]));
    } else {
      constexpr int c = (f - SC::RA) ^ (par ? 4 : 0);
      fb[c][h] = __builtin_bit_cast(i32x4, pp_frag<c * 16 * BK>(at + b_off[h]));
    }
  };

  set_stage(0);
#pragma unroll
  for (int j = 0; j < NB; ++j) {
#pragma unroll
    for (int p = 0; p < G; ++p) piece(j, p);
    advance();
  }
  pp_vm<(NB - 1) * G>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  pp_static_for<SC::early()>([&](auto mc) { rd(0u, mc, std::integral_constant<int, 0>{}); });
  __builtin_amdgcn_sched_barrier(0);

  const int lr = lane & 15, lq = lane >> 4;
  int slot = 0;
  auto ktile = [&](auto parc) {
    constexpr int par = decltype(parc)::value;
    const int nslot = slot == NB - 1 ? 0 : slot + 1;
    const uint32_t cur = (uint32_t)(slot * SLOT), next = (uint32_t)(nslot * SLOT);
    pp_static_for<NMF>([&](auto ic) {
      constexpr int i = decltype(ic)::value, r = SC::row(i), c = SC::col(i, par);
      if constexpr (i < 4) pp_lgkm<SC::wait(i)>();
      const i32x8 a = __builtin_shufflevector(fa[r][0], fa[r][1], 0, 1, 2, 3, 4, 5, 6, 7);
      const i32x8 b = __builtin_shufflevector(fb[c][0], fb[c][1], 0, 1, 2, 3, 4, 5, 6, 7);
      acc[r][c] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(b, a, acc[r][c], 0, 0, 0, 0, 0, 0);
      if constexpr (SC::read_at(NMF + i) >= 0) rd(cur, std::integral_constant<int, SC::read_at(NMF + i)>{}, parc);
      if constexpr (i == IB1) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
      }
      if constexpr (i > IB1 && (i - IB1 - 1) % GE == 0 && (i - IB1 - 1) / GE < G) piece(slot, (i - IB1 - 1) / GE);
      if constexpr (i == IB3) {
        pp_vm<VC>();
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
      }
      if constexpr (SC::read_at(i) >= 0)
        rd(next, std::integral_constant<int, SC::read_at(i)>{}, std::integral_constant<int, 1 - par>{});
      __builtin_amdgcn_sched_barrier(0);
    });
    advance();
    slot = nslot;
  };
  for (int ti = 0; ti < mine; ++ti) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        asm volatile("" : "+a"(acc[i][j]));            // zeroed in place, in AGPRs
      }
    for (int t = 0; t < nt; t += 2) {                  // (nt even: host)
      ktile(std::integral_constant<int, 0>{});
      ktile(std::integral_constant<int, 1>{});
    }
    // acc[r][c] lane l = C[row wm TM + 16 r + (l & 15)][col wn TN + 16 c + 4 (l >> 4) + v] (SwiGLU: fragments 2 cp (gate) and
    // 2 cp + 1 (up) hold the same output columns); the scales of its columns and rows
    int m_t, n_t;
    tile_mn(w + ti * P, m_t, n_t);
    f32x4 sc[CT];
    float sr[8];
    {
      const uint32_t at = lds_base + NB * SLOT + (ti & 1) * SCALES * 4;
      asm volatile(
          "ds_read_b128 %0, %16\n\tds_read_b128 %1, %16 offset:64\n\tds_read_b128 %2, %16 offset:128\n\t"
          "ds_read_b128 %3, %16 offset:192\n\tds_read_b128 %4, %16 offset:256\n\tds_read_b128 %5, %16 offset:320\n\t"
          "ds_read_b128 %6, %16 offset:384\n\tds_read_b128 %7, %16 offset:448\n\t"
          "ds_read_b32 %8, %17\n\tds_read_b32 %9, %17 offset:64\n\tds_read_b32 %10, %17 offset:128\n\t"
          "ds_read_b32 %11, %17 offset:192\n\tds_read_b32 %12, %17 offset:256\n\tds_read_b32 %13, %17 offset:320\n\t"
          "ds_read_b32 %14, %17 offset:384\n\tds_read_b32 %15, %17 offset:448\n\ts_waitcnt lgkmcnt(0)"
          : "=&v"(sc[0]), "=&v"(sc[1]), "=&v"(sc[2]), "=&v"(sc[3]), "=&v"(sc[4]), "=&v"(sc[5]), "=&v"(sc[6]), "=&v"(sc[7]),
            "=&v"(sr[0]), "=&v"(sr[1]), "=&v"(sr[2]), "=&v"(sr[3]), "=&v"(sr[4]), "=&v"(sr[5]), "=&v"(sr[6]), "=&v"(sr[7])
          : "v"(at + 1024 + (wn * TN + 4 * lq) * 4), "v"(at + (wm * TM + lr) * 4)
          : "memory");
    }
    __builtin_amdgcn_sched_barrier(0);
    // (the stores as in gemm_pf: 8 consecutive columns per lane, rows past M dropped by the range check)
    const uint32_t colb = (uint32_t)(n_t * OUTW + wn * (OUTW / NWN) + 16 * (lq & 1) + 8 * (lq >> 1)) * 2;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
#pragma unroll
      for (int c = 0; c < CT; ++c) asm volatile("" : "+a"(acc[r][c]));
      const int row = m_t * BM + wm * TM + r * 16 + lr;
      const uint32_t vo = row < M ? (uint32_t)row * (uint32_t)(ldc * 2) + colb : 0x80000000u;
      constexpr int NQ = SWIGLU ? CT / 2 : CT;
      u32x2 q[NQ];
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        bf16x4 hq;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          if constexpr (SWIGLU) {
            const float g = acc[r][2 * i][v] * (sr[r] * sc[2 * i][v]), u = acc[r][2 * i + 1][v] * (sr[r] * sc[2 * i + 1][v]);
            hq[v] = f2bf(silu_f(g) * u);
          } else {
            hq[v] = f2bf(acc[r][i][v] * (sr[r] * sc[i][v]));
          }
        }
        q[i] = __builtin_bit_cast(u32x2, hq);
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
        const u32x4 o = {x[0], x[1], y[0], y[1]};
        __builtin_amdgcn_raw_buffer_store_b128(o, rsC, (int)(vo + pr * 64), 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // the last K-tiles' surplus pieces must land before the workgroup's LDS is released
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// C = diag(a_scale) A B^T diag(b_scale) (mode 0) or its SwiGLU (mode 1, C [M, N / 2], B = [Bg; Bu]); K in elements (= bytes).
// bm: row tile 160, 192, 224 or 256.
void gemm_pf8(uintptr_t c, uintptr_t a, uintptr_t a_scale, uintptr_t b, uintptr_t b_scale, int M, int N, int K, int mode, int bm,
              uintptr_t stream) {
  DLLM_HOST_CHECK(M >= 1, "M >= 1");
  DLLM_HOST_CHECK(K % 256 == 0 && K >= 512, "K must be a multiple of 256, at least 512");
  DLLM_HOST_CHECK(N >= 256 && N % 256 == 0, "N must be a multiple of 256");
  DLLM_HOST_CHECK(mode == 0 || mode == 1, "mode 0 (plain) or 1 (SwiGLU)");
  DLLM_HOST_CHECK(a && b && c && a_scale && b_scale && (a | b | c) % 16 == 0 && (a_scale | b_scale) % 4 == 0, "operands");
  // rows past M are dropped by giving their stores the offset 0x80000000, which has to lie outside the output's range
  DLLM_HOST_CHECK((long)M * K < (1L << 32) && (long)N * K < (1L << 32) && (long)M * (mode ? N / 2 : N) * 2 < (1L << 31),
                  "operands must be < 4 GiB, the output < 2 GiB");
  DLLM_HOST_CHECK(bm == 256 || bm == 224 || bm == 192 || bm == 160, "row tile 160, 192, 224 or 256");
  static std::atomic<int> cus_of[64];                  // per device (a benign race: every thread stores the same value)
  int dev = 0;
  DLLM_HIP_CHECK(hipGetDevice(&dev));
  int cus = dev >= 0 && dev < 64 ? cus_of[dev].load(std::memory_order_relaxed) : 0;
  if (cus == 0) {
    int n = 0;
    DLLM_HIP_CHECK(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev));
    cus = n > 0 ? n : 256;
    if (dev >= 0 && dev < 64) cus_of[dev].store(cus, std::memory_order_relaxed);
  }
  const long tiles = (long)(N / 256) * ((M + bm - 1) / bm);
  DLLM_HOST_CHECK(tiles < (1L << 30), "tiles");
  const long grid = ((tiles < cus ? tiles : cus) + 7) / 8 * 8;
#define DLLM_PF8(SW_, RT_)                                                                                              \
  hipLaunchKernelGGL((gemm_pf8_kernel<SW_, RT_>), dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, (const uint8_t*)a, \
                     (const uint8_t*)b, (const float*)a_scale, (const float*)b_scale, (bf16*)c, M, N, K)
#define DLLM_PF8_BM(SW_)                      \
  do {                                        \
    if (bm == 256) DLLM_PF8(SW_, 8);          \
    else if (bm == 224) DLLM_PF8(SW_, 7);     \
    else if (bm == 192) DLLM_PF8(SW_, 6);     \
    else DLLM_PF8(SW_, 5);                    \
  } while (0)
  if (mode == 1) DLLM_PF8_BM(true);
  else DLLM_PF8_BM(false);
#undef DLLM_PF8_BM
#undef DLLM_PF8
  DLLM_HIP_CHECK(hipGetLastError());
}

}  // namespace dllm
