// Which products run on k_gemm_ring, and on which of its tiles, and which on k_gemm_split (host code without HIP; the tests
// build it by itself).
#pragma once
#include <stddef.h>

// The tile that is expected to be fastest, with its time in us; cfg < 0: none fits (a tile has to lie inside the
// matrices and a stage inside the reduction; offsets are 31 bits).
struct RingPlan { int cfg; double us; };
static const struct { int bm, bn, bk; double stage; } g_ring_cfgs[] = {
    // us per stage, measured with one tile on every CU
    {64, 64, 32, 0.43}, {64, 32, 64, 0.52}, {32, 64, 64, 0.52}, {32, 32, 64, 0.25}, {32, 16, 128, 0.31}, {16, 32, 128, 0.33}};
static inline RingPlan ring_plan(int M, int N, int K, size_t a_bytes, size_t b_bytes, int cus) {
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

// The same for products that k_gemm_ring is to take; cfg < 0: another kernel is expected to be faster.  The alternatives, as
// measured: 16 x 16 blocks take 2.9 us + 2.8 us per 1024 terms and round of the CUs (500 x 100 x 784 4.7 us against 5.6,
// 300 x 300 x 300 4.0 against 4.5; two rounds of 500 terms, 784 x 100 x 500, 5.5 against 5.1); slices of K with a second
// kernel 12 us + 1.5 us per 1e8 multiply-adds (few outputs over very long reductions); 128 x 128 tiles reach the same rate
// per output as 64 x 64 ones here (2000 x 2000 x 2000 130 us both) and win where their count fills the CUs as evenly.
// vec: the columns of both operands start at 16-byte boundaries, and one of them or both have the product's rows or columns
// along theirs.  The other kernels read those in 16-byte groups (the ring any), and short reductions are faster there.
static inline RingPlan gemm_ring_plan(int M, int N, int K, size_t a_bytes, size_t b_bytes, int cus, bool vec) {
  const RingPlan none = {-1, 0.}, ring = ring_plan(M, N, K, a_bytes, b_bytes, cus);
  if (ring.cfg < 0) return none;
  auto tiles = [&](int side) { return (long long)((M + side - 1) / side) * ((N + side - 1) / side); };
  auto rounds = [&](long long t) { return (t + cus - 1) / cus; };
  const double t16_us = 2.9 + 2.8 * (double)rounds(tiles(16)) * K / 1024.0;
  const double sliced_us = 12.0 + 1.5e-8 * (double)M * (double)N * (double)K;
  if (tiles(16) <= 2ll * cus && ring.us >= t16_us) return none;
  if (ring.us >= sliced_us) return none;
  // Strips of 17 to 31 rows or columns: the second 16-wide tile is nearly empty, a 32 x 32 block is not, and while those
  // fit one round of the CUs they take 3.8 us + 5 us per 1024 terms (operands from memory, us, ring -> blocks: 5899 x 21 x
  // 312 8.3 -> 7.3, 23 x 4407 x 250 6.2 -> 5.4, 4585 x 22 x 381 8.1 -> 7.2, 28 x 4655 x 180 5.9 -> 5.2).  Longer ones wait
  // for what a CU can pull in and win on the ring (from the caches, 6434 x 20 x 1675 16.2 against 21.9, 7038 x 19 x 743 9.3
  // against 11.6).
  const int thin = M < N ? M : N;
  if (thin > 16 && thin < 32 && K <= 512 && tiles(32) <= cus && ring.us >= 3.8 + 5.0 * K / 1024.0) return none;
  // Of 33 to 63 the 64-wide tile does not fit and the second 32-wide one mostly repeats the first.  From one and a half
  // 64 x 64 tiles per CU on the slab loop, whose tiles may hang over, is at least as fast (operands from memory, us, ring ->
  // slab loop: 57 x 25160 x 149 17.2 -> 12.7, 44 x 38103 x 167 21.4 -> 17.6, 26761 x 44 x 168 17.9 -> 15.4, 27552 x 55 x 239
  // 20.9 -> 21.2; fewer, 19399 x 49 x 252, 17.1 against 21.3).
  if (thin > 32 && thin < 64 && 20 * tiles(64) >= 29ll * cus) return none;
  // So does the second 64-wide tile of 65 to 85, more than two tiles per CU, as long as the reduction is short (23636 x 81 x
  // 243 25.3 -> 22.0, 17144 x 80 x 135 16.2 -> 14.5; longer ones, 77 x 21204 x 262, 24.9 against 28.8).
  if (thin > 64 && thin < 86 && tiles(64) > 2ll * cus && K <= 256) return none;
  // Strips of 17 to 31: one 64 x 64 tile per CU takes 5.9 us + 1.15 us per 100 terms, two 6.5 us + 3 us (12800 x 18 x 288
  // 11.2 -> 8.9, 15488 x 25 x 160 9.9 -> 7.9, 24200 x 25 x 144 13.7 -> 10.8; 20000 x 25 x 256 11.7 against 14.2).
  if (thin > 16 && thin < 32 && K <= 400 && 2 * tiles(64) <= 3ll * cus &&
      ring.us >= (tiles(64) <= cus ? 5.9 + 0.0115 * K : 6.5 + 0.03 * K)) return none;
  if (vec) {
    // More than two 64 x 64 tiles per CU: five workgroups of the slab loop share one and hide each other's waits (16384 x 147 x
    // 160 20.6 -> 16.0, 12800 x 200 x 208 25.7 -> 20.6, 10368 x 196 x 240 23.7 -> 19.4, 128 x 18880 x 240 24.3 -> 20.4;
    // of 546 the geometric means are, on the ring / there, 1.08 up to 256 terms, 1.01 up to 400, and 0.95 from 513 on).
    if (ring.cfg < 3 && tiles(64) > 2ll * cus && K <= (ring.cfg == 0 ? 400 : 256)) return none;
    // Strips of 33 to 63 from half a 64 x 64 tile per CU on (18432 x 49 x 208 15.7 -> 13.5, 10000 x 50 x 208 11.0 -> 9.3).
    if (thin > 32 && thin < 64 && K <= 256 && 2 * tiles(64) > cus) return none;
    // One round of 32 x 32 blocks of four stages at most: the blocks over eight wavefronts take the whole reduction at once
    // (1648 x 96 x 224 5.4 -> 4.6, 176 x 912 x 256 5.4 -> 4.8).
    if (ring.cfg == 3 && tiles(32) <= cus && K > 192 && K <= 256) return none;
  }
  if (tiles(128) >= cus && 4 * rounds(tiles(128)) <= rounds(tiles(64))) return none;
  return ring;
}

// Whether k_gemm runs a product on 128 x 128 tiles (see gemm()), else on 64 x 64.  Since k_gemm_split has most of what these were
// made for, strips are left: 33 to 191 rows or columns by more than 32768, and operands of 2 GiB and more.  Of 96 such strips those
// of 64 to 127 are as fast on either on average, long reductions faster here (us, 128 x 128 / 64 x 64: 57467 x 105 x 2173 279 /
// 392, 119 x 61225 x 1591 278 / 324); 33 to 63 would take 0.60 of the time on 64 x 64 tiles, 128 to 191 0.78.
static inline bool gemm_slab_big(int M, int N, int K, bool beta, int cus) {
  auto tiles = [&](int side) { return (long long)((M + side - 1) / side) * ((N + side - 1) / side); };
  auto fill = [&](long long t) { return (double)t / (double)(((t + cus - 1) / cus) * cus); };
  // 128 x 128 tiles (two workgroups per CU) against 64 x 64 tiles (five), as measured:
  // short reductions are mostly prologue and epilogue, which more resident workgroups hide
  // (4096 x 4096 x 128, beta = 1: 71 us against 60 us; up to K = 512 when C is also read, K = 256 otherwise); and
  // a tile count that leaves the last round of a CU half empty costs more than the smaller
  // tile's lower matrix-core rate of about 0.92 (3072 x 3072 x 2048: 404 us against 336 us).
  // (with the present main loop: 4096 x 4096 x 256 84 us on 64 x 64 tiles against 88 us, x 512 even, x 1024 268 us
  // against 254 us; fewer than two big tiles per CU leave the CU to one or two workgroups, and the small
  // tiles win up to K = 1024: 2048 x 2048 x 256 24.2 us against 30.3 us, x 512 39.6 against 46.7, x 1024 71.4
  // against 75.5)
  const int kmax64 = tiles(128) < 2ll * cus ? 1024 : beta ? 512 : 256;
  return tiles(128) >= cus && K > kmax64 && fill(tiles(128)) >= 0.92 * fill(tiles(64));
}

#define SPLIT_BM 128       // k_gemm_split's tile, and its stage of the reduction
#define SPLIT_BK 32
#define GEMM_SAMPLE_OUTPUTS (16 * 96 * 128)      // most outputs of a product that draws a sample of them (gemm.hip)

// What a product takes on k_gemm_split, in us: fitted to 462 measured products of 128 to 90000 per side and 32 to 5000 terms
// (rms 8 %).  A workgroup is alone on its CU, so what a tile costs besides its stages (first trip to memory, sums to
// memory) is not hidden; from the third round on the clock is what the matrix cores' power leaves.  < 0: no tile fits.
static inline double split_us(int M, int N, int K, size_t a_bytes, size_t b_bytes, int cus) {
  if (M < SPLIT_BM || N < SPLIT_BM || K < SPLIT_BK || a_bytes >= (1ull << 31) || b_bytes >= (1ull << 31)) return -1.;
  const long long tiles = (long long)((M + SPLIT_BM - 1) / SPLIT_BM) * ((N + SPLIT_BM - 1) / SPLIT_BM);
  const double rounds = tiles <= 3 * cus ? (double)((tiles + cus - 1) / cus) : 0.5 + (double)tiles / cus;
  return 4. + rounds * (1.05 * ((K + SPLIT_BK - 1) / SPLIT_BK) + 8.) * (rounds > 2. ? 1.18 : 1.);
}

// Whether k_gemm_split is expected to be faster than `ring` or, where that is none, than k_gemm (fitted to the same
// products).  Of the 462 it takes 99, which were 1.31 times as fast on average (4096 x 4096 x 4096 950 -> 670 us, 2048 x
// 2048 x 2048 140 -> 90, 3904 x 800 x 1568 112 -> 70, 3278 x 3637 x 1110 279 -> 170); the best choice for each would have
// gained 1 % more over all.  Cards differ: of random products that it takes, 300 took 0.75 times as long as before on one (three
// were more than 3 % slower, by 5 at most; the best choice for each 0.753 -> 0.753), 760 0.85 on one whose bf16 products take 18 %
// longer (44, by 21 at most: 11456 x 268 x 2000 146 -> 177, 496 x 5720 x 208 17.9 -> 21.5; 0.851 -> 0.847).  Estimates that suit
// the second card (1.37 us a stage) cost 3 % on the first and gain nothing on the second.  Strips of 129 to 191, whose second tile is mostly a repeat, have to win by more (169 x 54443 x
// 552 117 -> 137).
static inline bool gemm_split_wins(int M, int N, int K, bool beta, size_t a_bytes, size_t b_bytes, const RingPlan& ring, int cus) {
  auto tiles = [&](int side) { return (long long)((M + side - 1) / side) * ((N + side - 1) / side); };
  const double us = split_us(M, N, K, a_bytes, b_bytes, cus);
  if (us < 0. || K < 200) return false;               // (short ones are mostly first trip and stores: 4349 x 2436 x 86 36 -> 43)
  // A product that may draw a sample stays on the kernels that can, with and without one: the bits are those of the
  // calls one by one.  (On 256 CUs the estimates never differ on these; on 32 they would, 435 x 429 x 2008.)
  if ((long long)M * N <= GEMM_SAMPLE_OUTPUTS) return false;
  const int slabs = (K + 15) / 16;
  double other;
  if (ring.cfg >= 0) {
    other = 1.12 * ring.us;
  } else if (tiles(32) <= 2ll * cus) {
    return false;                                     // small products, or few outputs over a long reduction
  } else if (gemm_slab_big(M, N, K, beta, cus)) {
    const long long t = tiles(128);
    other = 8. + (t <= 3 * cus ? (double)((t + cus - 1) / cus) : 0.5 + (double)t / cus) * (1.16 * slabs + 3.);
  } else {
    other = 9. + 0.38 * slabs * (double)tiles(64) / cus;
  }
  const int thin = M < N ? M : N;
  return us * (thin > SPLIT_BM && 2 * thin < 3 * SPLIT_BM ? 1.3 : 1.05) < other;
}
