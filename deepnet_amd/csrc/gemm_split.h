// Larger products: see k_gemm_split.  Included by gemm.hip behind gemm_ring.h.
#pragma once
#include "split_tile.h"

// Products that gemm_split_wins expects to be faster here (from about 160 tiles of 128 x 128 and 200 terms on): see split_tile.h for
// the arithmetic.  8 wavefronts own a 128 x 128 tile of C, 64 x 32 outputs each; a stage is 32 terms, which are 96 MFMAs and
// about 250 vector instructions (taking 8192 numbers apart) on each SIMD.  An MFMA leaves room for two of those and
// every further one takes its four cycles: the matrix cores are busy for 58 % of the cycles and the issue of vector instructions
// for 53, of which 15 are the MFMAs' own (4096 x 4096 x 4096, at a clock of 1.75 GHz).  Smaller tiles take more
// numbers apart per product (128 x 64 tiles, two workgroups per CU, 2048 x 2048 x 2048: 111 us against 91), larger ones
// do not fit the registers with two accumulators each (256 x 128, 4096 x 4096 x 4096: 690 us with 50 registers spilled,
// against 670).  A stage takes 1.05 to 1.3 us, of which the MFMAs have 0.64.
// Measured (us, operands from memory, before -> now): 4096 x 4096 x 4096 950 -> 670 to 705 (195 to 205 TFLOP/s of fp32 products; 770
// to 880 on a card whose power limit leaves less), 2048 x 2048 x 2048 140 -> 90, 3904 x 800 x 1568 112 -> 70, 1152 x 2208 x 256 21.4 -> 20.2.
// Edges, alignment and the numbering of the tiles as in k_gemm_ring.
#define SPLIT_THREADS 512
template <bool A_KC, bool B_KC>
__global__ void __launch_bounds__(SPLIT_THREADS, 2) k_gemm_split(RingArgs g, GemmEpilogue epi) {
  constexpr int BM = SPLIT_BM, BN = SPLIT_BM, BK = SPLIT_BK, NT = SPLIT_THREADS;
  float* C = g.C;
  const int ldc = g.ldc, M = g.M, N = g.N, K = g.K, gx = g.gx, gy = g.gy;
  const float alpha = g.alpha, beta = g.beta;
  using OA = RingOperand<SplitTile<BM, BK, A_KC, NT>>;
  using OB = RingOperand<SplitTile<BN, BK, B_KC, NT>>;
  using Shape = SplitShape<BM, BN, BK, 2, 4, 1, 2, OA, OB>;
  constexpr int EPL = Shape::EPL;
  __shared__ __attribute__((aligned(16))) char lds[Shape::LDS];
  const int tid = threadIdx.x;
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
  const int em = m0 + tid % BM, en0 = n0 + tid / BM;
  // the last stage overlaps its predecessor by nst * BK - K terms, which it leaves out
  Shape::template run<true>(lds, oa, ob, nst, nst * BK - K, [] {});
  constexpr int EP = EPL < 16 ? EPL : 16;
#pragma unroll
  for (int u0 = 0; u0 < EPL; u0 += EP) {
    float cold[EP];
    if (beta != 0.f) {
#pragma unroll
      for (int u = 0; u < EP; ++u) cold[u] = C[(size_t)(en0 + (u0 + u) * (NT / BM)) * ldc + em];
    }
#pragma unroll
    for (int u = 0; u < EP; ++u) {
      const int en = en0 + (u0 + u) * (NT / BM);
      if (em >= m_lo && en >= n_lo) {
        const size_t off = (size_t)en * ldc + em;
        C[off] = gemm_finish(small_axpby(beta, beta != 0.f ? cold[u] : 0.f, alpha, Shape::sum(lds, tid, u0 + u)), em, off, epi);
      }
    }
  }
}

static void split_launch(bool a_kc, bool b_kc, RingArgs g, const GemmEpilogue& epi) {
  g.gx = (g.M + SPLIT_BM - 1) / SPLIT_BM; g.gy = (g.N + SPLIT_BM - 1) / SPLIT_BM;
  const dim3 grid((unsigned)(8 * ((g.gx * g.gy + 7) / 8)));
#define SPLIT_GO(AK, BK_) hipLaunchKernelGGL((k_gemm_split<AK, BK_>), grid, dim3(SPLIT_THREADS), 0, dn_stream(), g, epi)
  if (a_kc && b_kc) SPLIT_GO(true, true);
  else if (a_kc) SPLIT_GO(true, false);
  else if (b_kc) SPLIT_GO(false, true);
  else SPLIT_GO(false, false);
#undef SPLIT_GO
}
