// Mid-sized products: see k_gemm_ring.  Included by gemm.hip (GemmEpilogue, f32x16).
#pragma once
#include <type_traits>

#define RING_THREADS 512
#define RING_SETS 4        // register sets: the stages on their way from global memory

// Stage t of an operand as this lane's 16-byte groups; a stage behind the last one is an out-of-range offset, which the
// buffer hardware answers with zeros without going to memory (every trip of the loop issues the same requests, so
// the compiler can count them).
template <int ROWS, int BK, bool KC>
struct RingOperand {
  static constexpr int NG = ROWS * BK / 4 / RING_THREADS;        // 16-byte groups per lane and stage
  static_assert(NG * RING_THREADS * 4 == ROWS * BK, "whole groups per lane");
  static constexpr int PITCH = KC ? BK + 4 : ROWS + 4;            // floats; 4 mod 8 (see k_gemm_ring)
  static constexpr int FLOATS = KC ? ROWS * PITCH : BK * PITCH;
  __amdgpu_buffer_rsrc_t rsrc;
  unsigned voff[NG];
  unsigned step, last;
  __device__ __forceinline__ void init(const float* P, unsigned bytes, int ld, int row0, int K, int tid) {
    rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)P, 0, (int)bytes, 0x00020000);
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      const int f = tid + u * RING_THREADS;
      voff[u] = KC ? 4u * ((unsigned)(row0 + f / (BK / 4)) * (unsigned)ld + 4u * (unsigned)(f % (BK / 4)))
                   : 4u * ((unsigned)(f / (ROWS / 4)) * (unsigned)ld + (unsigned)row0 + 4u * (unsigned)(f % (ROWS / 4)));
    }
    const unsigned per_k = KC ? 4u : 4u * (unsigned)ld;
    step = BK * per_k;
    last = (unsigned)(K - BK) * per_k;
  }
  __device__ __forceinline__ void fetch(int t, int nst, f32x4 (&r)[NG]) const {
    const unsigned at = (unsigned)t * step;                       // (without a branch: the loop stays one block)
    const unsigned so = (at < last ? at : last) | ((unsigned)(nst - 1 - t) & 0x80000000u);
#pragma unroll
    for (int u = 0; u < NG; ++u)
      r[u] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)voff[u], (int)so, 0));
  }
  __device__ __forceinline__ static void stash(float* S, int tid, const f32x4 (&r)[NG]) {
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      const int f = tid + u * RING_THREADS;
      float* d = KC ? S + (f / (BK / 4)) * PITCH + 4 * (f % (BK / 4)) : S + (f / (ROWS / 4)) * PITCH + 4 * (f % (ROWS / 4));
      *reinterpret_cast<f32x4*>(d) = r[u];
    }
  }
  // v[4 u + j] = operand(row, k0 + u * KU + j), u < 2, j < 4
  template <int KU>
  __device__ __forceinline__ static void frag(const float* S, int row, int k0, float (&v)[8]) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (KC) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(S + row * PITCH + k0 + KU * u);
        v[4 * u] = x.x; v[4 * u + 1] = x.y; v[4 * u + 2] = x.z; v[4 * u + 3] = x.w;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[4 * u + j] = S[(k0 + KU * u + j) * PITCH + row];
      }
    }
  }
};

__device__ __forceinline__ f32x16 ring_mfma(float b, float a, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(b, a, c, 0, 0, 0); }
__device__ __forceinline__ f32x4 ring_mfma(float b, float a, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(b, a, c, 0, 0, 0); }

// Products of a few hundred to a few thousand per side (the layers of a net at its batch size): their outputs
// make one or two tiles per CU at best, so a workgroup is alone with its latencies, and what bounds the older kernels
// there is how few bytes they keep in flight (k_gemm: three 16-deep slabs, 0.33 us per slab where its MFMAs take
// 0.21) or how many they ask the L2s for (k_gemm_small: 32 x 32 blocks straight from global memory).
//
// RING_THREADS lanes = 8 wavefronts own a BM x BN tile of C.  A stage is BK terms of the reduction: registers take stages
// from global memory four stages ahead of their use (RING_SETS), LDS holds two, and the fragments of a stage are read
// one stage ahead of its MFMAs, so that a trip of the loop is one barrier, one stage of MFMAs and nothing that waits.
// The tile is BM/TB x BN/TB blocks of TB x TB outputs; the wavefronts that are left over split the stage's terms KS
// ways and meet in LDS at the end, in a fixed order: a small tile, of which there are enough to cover the chip,
// still has eight wavefronts' worth of MFMAs per stage.  Nothing is masked in the loop: a tile that hangs over the
// edge moves back inside the matrix and stores only its own outputs; the last stage moves back likewise (it ends at
// K) and leaves out the terms that were taken already.  16-byte requests at any 4-byte boundary serve odd leading
// dimensions.
// LDS rows: [row][BK + 4] for a K-contiguous operand, [k][rows + 4] for the other kind, both free of bank conflicts
// for the order of terms that `frag` reads (pitch 4 mod 8).
// Tiles are numbered so that each XCD gets a contiguous run of them, along the shorter side first (shared panels
// meet in its L2).
// Measured (us, before -> now; before: the best of the other kernels), first operand transposed / neither / second:
//   1500 x 300 x 1001   22.1 -> 13.6  24.1 -> 13.6  26.0 -> 13.6      64 x 32 tiles (floor at 157 TFLOP/s: 5.7)
//   2001 x 1003 x 250   16.1 -> 13.9  20.3 -> 14.5  20.3 -> 14.6      64 x 64
//   1024 x 100 x 2304   16.1 -> 9.3   14.2 -> 10.0  14.9 -> 11.2      32 x 16
//   814 x 263 x 1038    11.1 -> 8.0   13.6 -> 8.5   14.9 -> 8.7       32 x 32
//   1000 x 1000 x 1000  26.9 -> 21.3  23.5 -> 19.9  23.8 -> 20.2      64 x 64
// What is left above the MFMAs' time at 64 x 64 is 4.3 us: launch 2.4, the first trip to memory, the sum over the
// wavefronts and the stores.  The smaller tiles run at what the L2s give (20 TB/s over the chip).
struct RingArgs {
  const float* A; const float* B;
  float* C;
  unsigned a_bytes, b_bytes;
  int lda, ldb, ldc, M, N, K, gx, gy;
  float alpha, beta;
};

template <int TB, int BM, int BN, int BK, bool A_KC, bool B_KC>
__global__ void __launch_bounds__(RING_THREADS, 4) k_gemm_ring(RingArgs g, GemmEpilogue epi) {
  float* C = g.C;
  const int ldc = g.ldc, M = g.M, N = g.N, K = g.K, gx = g.gx, gy = g.gy;
  const float alpha = g.alpha, beta = g.beta;
  constexpr int WM = BM / TB, WN = BN / TB, KS = 8 / (WM * WN), KW = BK / KS;
  static_assert(KW == 512 / TB, "eight MFMAs per wavefront and stage");
  using acc_t = std::conditional_t<TB == 32, f32x16, f32x4>;
  constexpr int NACC = TB * TB / 64, KU = TB == 32 ? 4 : 16;
  using OA = RingOperand<BM, BK, A_KC>;
  using OB = RingOperand<BN, BK, B_KC>;
  constexpr int STAGE = OA::FLOATS + OB::FLOATS, RED = KS * BM * BN;
  constexpr int LDS = 2 * STAGE > RED ? 2 * STAGE : RED;
  __shared__ __attribute__((aligned(16))) float lds[LDS];
  const int tid = threadIdx.x, lane = tid & 63, li = lane % TB, lk = lane / TB;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wv % WM, wn = (wv / WM) % WN, ks = wv / (WM * WN);
  // contiguous runs of tiles per XCD, along the shorter side of the grid first: the tiles of an XCD share operand panels
  const int tiles = gx * gy, run = (tiles + 7) >> 3;
  const int t = (int)(blockIdx.x & 7) * run + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= run || t >= tiles) return;
  const int bx = gx >= gy ? t / gy : t % gx, by = gx >= gy ? t % gy : t / gx;
  // a tile over the edge moves back inside; the outputs it shares with its neighbour are that one's to store
  const int m_lo = bx * BM, n_lo = by * BN;
  const int m0 = m_lo + BM <= M ? m_lo : M - BM, n0 = n_lo + BN <= N ? n_lo : N - BN;
  const int nst = (K + BK - 1) / BK;

  OA oa; OB ob;
  oa.init(g.A, g.a_bytes, g.lda, m0, K, tid);
  ob.init(g.B, g.b_bytes, g.ldb, n0, K, tid);
  f32x4 ra[RING_SETS][OA::NG], rb[RING_SETS][OB::NG];
#define RING_FETCH(SET, T) do { oa.fetch(T, nst, ra[SET]); ob.fetch(T, nst, rb[SET]); } while (0)
#define RING_STASH(BUF, SET) do { OA::stash(lds + (BUF) * STAGE, tid, ra[SET]); OB::stash(lds + (BUF) * STAGE + OA::FLOATS, tid, rb[SET]); } while (0)
  const int arow = wm * TB + li, brow = wn * TB + li, fk = ks * KW + (TB == 32 ? 8 : 4) * lk;
#define RING_FRAG(BUF, AV, BV) do { OA::template frag<KU>(lds + (BUF) * STAGE, arow, fk, AV); OB::template frag<KU>(lds + (BUF) * STAGE + OA::FLOATS, brow, fk, BV); } while (0)
  // stage s sits in register set (s + 2) % 4 until it is written to LDS[s & 1]
  RING_FETCH(2, 0); RING_FETCH(3, 1); RING_FETCH(0, 2); RING_FETCH(1, 3);
  constexpr int EPL = BM * BN / RING_THREADS;
  float cold[EPL];
  const int em = m0 + tid % BM, en0 = n0 + tid / BM;
  if (beta != 0.f) {
#pragma unroll
    for (int u = 0; u < EPL; ++u) cold[u] = C[(size_t)(en0 + u * (RING_THREADS / BM)) * ldc + em];
  }
  RING_STASH(0, 2); RING_FETCH(2, 4);
  RING_STASH(1, 3); RING_FETCH(3, 5);
  acc_t acc;
#pragma unroll
  for (int v = 0; v < NACC; ++v) acc[v] = 0.f;
  float fa[2][8], fb[2][8];
  __syncthreads();
  RING_FRAG(0, fa[0], fb[0]);
  __syncthreads();
  int s = 0;
  for (; s + 4 < nst; s += 4) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      RING_FRAG((q + 1) & 1, fa[(q + 1) & 1], fb[(q + 1) & 1]);
      RING_STASH(q & 1, q);
      RING_FETCH(q, s + q + 6);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc = ring_mfma(fb[q & 1][j], fa[q & 1][j], acc);
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        if (g >= 4) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        if (g >= 4) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // the last one to four stages; the last one overlaps its predecessor by nst * BK - K terms, which it leaves out
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (s + q < nst) {
      const int kmin = s + q == nst - 1 ? nst * BK - K : 0;
      if (s + q + 1 < nst) RING_FRAG((q + 1) & 1, fa[(q + 1) & 1], fb[(q + 1) & 1]);
      if (s + q + 2 < nst) RING_STASH(q & 1, q);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const bool in = fk + KU * (j >> 2) + (j & 3) >= kmin;
        acc = ring_mfma(in ? fb[q & 1][j] : 0.f, in ? fa[q & 1][j] : 0.f, acc);
      }
      __syncthreads();
    }
  }
  // acc[v] is the tile's (m, n) = (32 wm + li, 32 wn + 8 (v / 4) + 4 lk + v % 4); partial tiles are [n][m]
  float* part = lds + ks * (BM * BN);
#pragma unroll
  for (int v = 0; v < NACC; ++v) part[(wn * TB + 8 * (v >> 2) + 4 * lk + (v & 3)) * BM + wm * TB + li] = acc[v];
  __syncthreads();
#pragma unroll
  for (int u = 0; u < EPL; ++u) {
    const int e = tid + RING_THREADS * u, en = en0 + u * (RING_THREADS / BM);
    float sum = lds[e];
#pragma unroll
    for (int w = 1; w < KS; ++w) sum += lds[w * (BM * BN) + e];
    if (em >= m_lo && en >= n_lo) {
      const size_t off = (size_t)en * ldc + em;
      float out = gemm_finish(small_axpby(beta, beta != 0.f ? cold[u] : 0.f, alpha, sum), em, off, epi);
      const unsigned int i = (unsigned int)off;
      if (epi.sample && epi.drop) out = out * gemm_draw_mask(gemm_draw_fetch(i, true, epi), i, epi);
      C[off] = out;
      if (epi.sample && !epi.drop) gemm_draw_store(gemm_draw_fetch(i, true, epi), i, out, epi);
    }
  }
  if (t == 0) gemm_draw_idle_streams(tid, RING_THREADS, epi);
#undef RING_FETCH
#undef RING_STASH
#undef RING_FRAG
}

// The tile that is expected to be fastest, with its time in us; cfg < 0: none fits (a tile has to lie inside the
// matrices and a stage inside the reduction; offsets are 31 bits).
struct RingPlan { int cfg; double us; };
static const struct { int bm, bn, bk; double stage; } g_ring_cfgs[] = {
    // us per stage, measured with one tile on every CU
    {64, 64, 32, 0.43}, {64, 32, 64, 0.52}, {32, 64, 64, 0.52}, {32, 32, 64, 0.25}, {32, 16, 128, 0.31}, {16, 32, 128, 0.33}};
static RingPlan ring_plan(int M, int N, int K, size_t a_bytes, size_t b_bytes, int cus) {
  RingPlan best = {-1, 0.};
  if (a_bytes >= (1ull << 31) || b_bytes >= (1ull << 31)) return best;
  for (int c = 0; c < (int)(sizeof(g_ring_cfgs) / sizeof(g_ring_cfgs[0])); ++c) {
    const auto& f = g_ring_cfgs[c];
    if (M < f.bm || N < f.bn || K < f.bk) continue;
    const long long tiles = (long long)((M + f.bm - 1) / f.bm) * ((N + f.bn - 1) / f.bn);
    const double rounds = (double)((tiles + cus - 1) / cus);
    // a CU holds two workgroups; from the third on a tile's first trip to memory is not hidden
    const double us = 4.2 + rounds * ((K + f.bk - 1) / f.bk) * f.stage + (rounds > 2 ? 1.3 * (rounds - 2) : 0.);
    if (best.cfg < 0 || us < best.us) best = {c, us};
  }
  return best;
}

template <int TB, int BM, int BN, int BK>
static void ring_launch_cfg(bool a_kc, bool b_kc, RingArgs g, const GemmEpilogue& epi) {
  g.gx = (g.M + BM - 1) / BM; g.gy = (g.N + BN - 1) / BN;
  const dim3 grid((unsigned)(8 * ((g.gx * g.gy + 7) / 8)));
#define RING_GO(AK, BK_) hipLaunchKernelGGL((k_gemm_ring<TB, BM, BN, BK, AK, BK_>), grid, dim3(RING_THREADS), 0, dn_stream(), g, epi)
  if (a_kc && b_kc) RING_GO(true, true);
  else if (a_kc) RING_GO(true, false);
  else if (b_kc) RING_GO(false, true);
  else RING_GO(false, false);
#undef RING_GO
}
static void ring_launch(int cfg, bool a_kc, bool b_kc, const RingArgs& g, const GemmEpilogue& epi) {
  switch (cfg) {
    case 0: ring_launch_cfg<32, 64, 64, 32>(a_kc, b_kc, g, epi); break;
    case 1: ring_launch_cfg<32, 64, 32, 64>(a_kc, b_kc, g, epi); break;
    case 2: ring_launch_cfg<32, 32, 64, 64>(a_kc, b_kc, g, epi); break;
    case 3: ring_launch_cfg<16, 32, 32, 64>(a_kc, b_kc, g, epi); break;
    case 4: ring_launch_cfg<16, 32, 16, 128>(a_kc, b_kc, g, epi); break;
    default: ring_launch_cfg<16, 16, 32, 128>(a_kc, b_kc, g, epi); break;
  }
}
