// Mid-sized products: see k_gemm_ring.  Included by gemm.hip (GemmEpilogue, f32x16).
#pragma once
#include "ring_tile.h"
#include "gemm_ring_plan.h"

// Stage t of an operand as this lane's 16-byte groups.  Every trip of the loop issues the same requests, so that the
// compiler can count them; those of a stage behind the last one go to a buffer of no bytes, which answers with zeros
// and does not go to memory.  An offset beyond the buffer would do as well, the lanes' or the scalar one (both take part in
// the range check: measured on buffers inside a larger allocation, loads and stores); a bit in the lanes' offsets is
// a vector instruction per request (dense 1001 x 1500 x 300, three products: 46.4 against 49.0 us).
template <class Tile>
struct RingOperand : Tile {
  using Tile::NG;
  static constexpr int BK = Tile::BK;
  static constexpr bool KC = Tile::KC;
  const float* P0;
  unsigned voff[NG];
  unsigned n_bytes, step, last;
  __device__ __forceinline__ void init(const float* P, unsigned bytes, int ld, int row0, int K, int tid) {
    P0 = P; n_bytes = bytes;
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      const unsigned row = (unsigned)(row0 + Tile::group_row(tid, u)), k = (unsigned)Tile::group_k(tid, u);
      voff[u] = KC ? 4u * (row * (unsigned)ld + k) : 4u * (k * (unsigned)ld + row);
    }
    const unsigned per_k = KC ? 4u : 4u * (unsigned)ld;
    step = BK * per_k;
    last = (unsigned)(K - BK) * per_k;
  }
  __device__ __forceinline__ void fetch(int t, int nst, f32x4 (&r)[NG]) const {
    const unsigned at = (unsigned)t * step;                       // (without a branch: the loop stays one block)
    const unsigned in = ~(unsigned)((nst - 1 - t) >> 31), so = (at < last ? at : last) & in;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)P0, 0, (int)(n_bytes & in), 0x00020000);
#pragma unroll
    for (int u = 0; u < NG; ++u)
      r[u] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)voff[u], (int)so, 0));
  }
};

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
// Measured (us, operands from memory, before -> now; before: the best of the other kernels), first operand transposed /
// neither / second:
//   1500 x 300 x 1001   23.3 -> 15.7  24.5 -> 16.5  27.0 -> 17.1      32 x 32 tiles (floor at 157 TFLOP/s: 5.7)
//   2001 x 1003 x 250   17.4 -> 17.0  20.5 -> 17.1  21.6 -> 17.0      64 x 64
//   1024 x 100 x 2304   17.2 -> 10.8  16.6 -> 13.3  17.8 -> 15.7      32 x 16
//   814 x 263 x 1038    11.7 -> 8.7   13.7 -> 9.0   15.2 -> 9.4       32 x 32
//   1000 x 1000 x 1000  26.9 -> 21.2  27.0 -> 21.4  26.7 -> 21.6      64 x 64
//   2074 x 464 x 912    34.4 -> 22.0                                  64 x 32
//   726 x 2749 x 1091                 81.1 -> 51.6                    32 x 64
// What is left above the MFMAs' time at 64 x 64 is 4.3 us: launch 2.4, the first trip to memory, the sum over the
// wavefronts and the stores.  The smaller tiles run at what the L2s give: a stage of a 32 x 16 tile is 24.6 KB in 0.31 us on
// every CU, 20 TB/s over the chip.
struct RingArgs {
  const float* A; const float* B;
  float* C;
  unsigned a_bytes, b_bytes;
  int lda, ldb, ldc, M, N, K, gx, gy;
  float alpha, beta;
};

// The second product of a pair into one C: C = beta*C + alpha*op(A)*op(B), then C = C + alpha*op(A2)*op(B2), each rounded as by
// itself (no epilogue).  A null: none.
struct RingSecond { const float* A; const float* B; unsigned a_bytes, b_bytes; int lda, ldb; float alpha; };

// Tile `block` of a product.
template <int TB, int BM, int BN, int BK, bool A_KC, bool B_KC>
struct RingProduct {
  using OA = RingOperand<RingTile<BM, BK, A_KC>>;
  using OB = RingOperand<RingTile<BN, BK, B_KC>>;
  using Shape = RingShape<TB, BM, BN, BK, OA, OB>;
  template <bool PAIRS>
  __device__ __forceinline__ static void run(float* lds, const RingArgs& g, const GemmEpilogue& epi, const RingSecond& second, int block) {
    float* C = g.C;
    const int ldc = g.ldc, M = g.M, N = g.N, K = g.K, gx = g.gx, gy = g.gy;
    const float alpha = g.alpha, beta = g.beta;
    constexpr int EPL = Shape::EPL;
    const int tid = ring_tid<PAIRS>();
    // contiguous runs of tiles per XCD, along the shorter side of the grid first: the tiles of an XCD share operand panels
    const int tiles = gx * gy, run = (tiles + 7) >> 3;
    const int t = (block & 7) * run + (block >> 3);
    if ((block >> 3) >= run || t >= tiles) return;
    const int bx = gx >= gy ? t / gy : t % gx, by = gx >= gy ? t % gy : t / gx;
    // a tile over the edge moves back inside; the outputs it shares with its neighbour are that one's to store
    const int m_lo = bx * BM, n_lo = by * BN;
    const int m0 = m_lo + BM <= M ? m_lo : M - BM, n0 = n_lo + BN <= N ? n_lo : N - BN;
    const int nst = (K + BK - 1) / BK;

    OA oa; OB ob;
    oa.init(g.A, g.a_bytes, g.lda, m0, K, tid);
    ob.init(g.B, g.b_bytes, g.ldb, n0, K, tid);
    float cold[EPL], sum[EPL];
    const int em = m0 + tid % BM, en0 = n0 + tid / BM;
    // the last stage overlaps its predecessor by nst * BK - K terms, which it leaves out
    Shape::template run<true, PAIRS>(lds, oa, ob, nst, nst * BK - K, sum, [&] {
      if (beta != 0.f) {
#pragma unroll
        for (int u = 0; u < EPL; ++u) cold[u] = C[(size_t)(en0 + u * (RING_THREADS / BM)) * ldc + em];
      }
    });
#pragma unroll
    for (int u = 0; u < EPL; ++u) sum[u] = small_axpby(beta, beta != 0.f ? cold[u] : 0.f, alpha, sum[u]);
    if (PAIRS && second.A) {
      oa.init(second.A, second.a_bytes, second.lda, m0, K, tid);
      ob.init(second.B, second.b_bytes, second.ldb, n0, K, tid);
      __syncthreads();                                      // (the first product's sums have been read)
#pragma unroll
      for (int u = 0; u < EPL; ++u) cold[u] = sum[u];
      Shape::template run<true, PAIRS>(lds, oa, ob, nst, nst * BK - K, sum, [] {});
#pragma unroll
      for (int u = 0; u < EPL; ++u) sum[u] = small_axpby(1.f, cold[u], second.alpha, sum[u]);
    }
#pragma unroll
    for (int u = 0; u < EPL; ++u) {
      const int en = en0 + u * (RING_THREADS / BM);
      if (em >= m_lo && en >= n_lo) {
        const size_t off = (size_t)en * ldc + em;
        float out = gemm_finish(sum[u], em, off, epi);
        const unsigned int i = (unsigned int)off;
        if (!PAIRS && epi.sample && epi.drop) out = out * gemm_draw_mask(gemm_draw_fetch(i, true, epi), i, epi);
        C[off] = out;
        if (!PAIRS && epi.sample && !epi.drop) gemm_draw_store(gemm_draw_fetch(i, true, epi), i, out, epi);
      }
    }
    if (!PAIRS && t == 0) gemm_draw_idle_streams(tid, RING_THREADS, epi);
  }
};

template <int TB, int BM, int BN, int BK, bool A_KC, bool B_KC>
__global__ void __launch_bounds__(RING_THREADS, 4) k_gemm_ring(RingArgs g, GemmEpilogue epi) {
  using P = RingProduct<TB, BM, BN, BK, A_KC, B_KC>;
  __shared__ __attribute__((aligned(16))) float lds[P::Shape::LDS];
  P::template run<false>(lds, g, epi, RingSecond{}, (int)blockIdx.x);
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

// Several products, and sums along rows, that have nothing to do with each other, in one launch (the open group, see
// dn_group_*): a layer's forward product, its input gradient and its weight gradient come one after the other in a step, each
// is one or two tiles per CU, and by itself spends a third of its time on the launch, the first trip to memory and a last
// round that leaves most CUs idle.  Tiles are those the products have alone (same bits); those that take longest come first.
// Measured (us, launched one by one -> as a group): the three products of a 1001 x 1500 layer, batch 300, 46.4 -> 36.1; the step
// of a 2001 x 1003 RBM, batch 250, whose two statistics are one pass over the weights with the sums beside it, 84.6 -> 75.6.
// What is left of the layer is what the tiles ask the L2s for, 303 MB.
#define RING_GROUP 4
struct RingJob { RingArgs g; GemmEpilogue epi; RingSecond second; int variant, end; };     // end: behind its last workgroup
struct RingGroup { int sums_end, sums_blocks; RowSumJobs sums; RingJob job[RING_GROUP]; };

template <int CFG, bool A_KC, bool B_KC> struct RingOf;
#define RING_OF(C, ...) template <bool A_KC, bool B_KC> struct RingOf<C, A_KC, B_KC> : RingProduct<__VA_ARGS__, A_KC, B_KC> {};
RING_OF(0, 32, 64, 64, 32) RING_OF(1, 32, 64, 32, 64) RING_OF(2, 32, 32, 64, 64)
RING_OF(3, 16, 32, 32, 64) RING_OF(4, 16, 32, 16, 128) RING_OF(5, 16, 16, 32, 128)
#undef RING_OF
template <int CFG> static int ring_lds_bytes(bool a_kc, bool b_kc) {
  return 4 * (a_kc ? (b_kc ? RingOf<CFG, true, true>::Shape::LDS : RingOf<CFG, true, false>::Shape::LDS)
                   : (b_kc ? RingOf<CFG, false, true>::Shape::LDS : RingOf<CFG, false, false>::Shape::LDS));
}

// (of two kinds of tile: with the 12 loops of three the compiler spills hundreds of registers)
template <int C0, int C1>
__global__ void __launch_bounds__(RING_THREADS, 4) k_gemm_group(RingGroup G) {
  extern __shared__ __attribute__((aligned(16))) float group_lds[];
  const int block = (int)blockIdx.x;
  if (block < G.sums_end) {
    if (block < G.sums_blocks) rows_sum_jobs_body(G.sums, block);
    return;
  }
  int j = 0, first = G.sums_end;
  while (block >= G.job[j].end) first = G.job[j++].end;     // (the last one ends with the grid)
  const RingJob& J = G.job[j];
#define RING_BODY(AT, C, AK, BK_) case AT: RingOf<C, AK, BK_>::template run<true>(group_lds, J.g, J.epi, J.second, block - first); break;
#define RING_BODIES(AT, C) RING_BODY(AT, C, false, false) RING_BODY(AT + 1, C, false, true) RING_BODY(AT + 2, C, true, false) RING_BODY(AT + 3, C, true, true)
  switch (J.variant) { RING_BODIES(0, C0) RING_BODIES(4, C1) }
#undef RING_BODIES
#undef RING_BODY
}
// Launches G, whose jobs have the tiles of g_ring_cfgs c0 < c1; LDS for the largest of them.
static void ring_group_launch(int c0, int c1, const RingGroup& G, int blocks) {
  int lds = 0;
  auto room = [&](int bytes) { lds = bytes > lds ? bytes : lds; };
#define RING_GROUP_GO(A, B)                                                                                                  \
  if (c0 == A && c1 == B) {                                                                                                  \
    for (int j = 0; j == 0 || G.job[j - 1].end < blocks; ++j) {                                                              \
      const int v = G.job[j].variant;                                                                                        \
      room(v < 4 ? ring_lds_bytes<A>((v & 2) != 0, (v & 1) != 0) : ring_lds_bytes<B>((v & 2) != 0, (v & 1) != 0));           \
    }                                                                                                                        \
    hipLaunchKernelGGL((k_gemm_group<A, B>), dim3((unsigned)blocks), dim3(RING_THREADS), (unsigned)lds, dn_stream(), G); \
    return;                                                                                                                  \
  }
  RING_GROUP_GO(0, 1) RING_GROUP_GO(0, 2) RING_GROUP_GO(0, 3) RING_GROUP_GO(0, 4) RING_GROUP_GO(0, 5)
  RING_GROUP_GO(1, 2) RING_GROUP_GO(1, 3) RING_GROUP_GO(1, 4) RING_GROUP_GO(1, 5)
  RING_GROUP_GO(2, 3) RING_GROUP_GO(2, 4) RING_GROUP_GO(2, 5)
  RING_GROUP_GO(3, 4) RING_GROUP_GO(3, 5) RING_GROUP_GO(4, 5)
#undef RING_GROUP_GO
}
