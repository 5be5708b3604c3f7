// Convolution passes on the tile loop of ring_tile.h: see k_conv_ring.  Included by conv.hip (ConvArgs).
#pragma once
#include "split_tile.h"
#include "conv_ring_plan.h"

// A term of the reduction, as the workgroup keeps it in LDS for its reduction (one entry per term for Up, per four
// for Down and Outp): the byte offset that it adds to a lane's, and which filter rows (bits 0-14) and columns (15-29)
// have to be inside (Up, Down: `mask` of the entry has to be part of the lane's) or are inside (Outp: the other way
// round).  RING_FAR stands in no lane's mask: such a term reads as zero.  Of filters that are no multiple of four, the last
// entry of a tap (RING_LAST in its mask) moves back to the last four, and leaves out those that the entry before has.
#define RING_FAR 0x80000000u
#define RING_LAST 0x40000000u
static_assert(2 * RING_MAX_SIDE <= 30, "masks below RING_LAST");
static_assert(RING_AHEAD >= RING_SETS + 3, "fetch() looks one stage ahead, the loop RING_SETS + 2");

struct ConvRingArgs {
  const float* a; const float* b;
  float* out;
  unsigned a_bytes, b_bytes;
  int N, H, HH, Mx, M, k, kk2, s, pad0, Cg, Fg, F, G;
  int local;                    // one filter bank per module
  int rows, cols;               // of one period: a tile lies inside one (one module or pixel, or everything)
  int periods, gx, gy, gz;      // tiles per period down the rows, across; Up / Down: groups; Outp: chunks x splits x groups
  int K;                        // Outp: terms of a chunk
  // (What only Outp has, and only DownM: side of a block of pixels, blocks per side of a map.  64 bytes more of arguments are 0.15 us
  // a launch, and so is a line of 64 that a pass reads for one of them only: what every tile needs of the divisors lies next to ldc.)
  union { int m_count, block; };
  union { int splits, lines; };
  int split_stages;
  FastDiv dN;
  union { FastDiv dMx, dlines; };                                        // all others; DownM
  union { FastDiv dk, dblock; };
  union { FastDiv dkk2, dblock2; };
  FastDiv dH, dFg4, dgx, dgy, dper;
  union { FastDiv dsplits, ds; };                                        // Outp; Down
  FastDiv dG;
  __host__ __device__ int Fg4() const { return (Fg + 3) & ~3; }          // filters of a group in whole fours
  long long ldc, out_stride;    // of a column; Outp: of a (chunk, split)
};

// Operand of a convolution stage: offsets and masks from the table of the workgroup's reduction.
// KIND 0: rows are (module | pixel, image) groups, a table entry per PER terms (A of Up and Down)
//      1: rows are filters, terms in order of memory (B of Up)
//      2: rows are colours, four filters of a tap per entry (B of Down)
//      3: rows are filters, terms (module, image) in order of memory (A of Outp)
//      4: rows are taps, four images of a module per entry (B of Outp)
//   On tiles of one module or pixel every entry is an offset into each operand, or RING_FAR behind the last term:
//      5, 6: A (x of an entry) and B (y) of Up and A of Down
//      7: B of Down
//      9: A of DownM (its mask: RING_LAST where the lane's term of a tap's last entry is taken by the one before)
//      8: B of DownM: rows are (colour, row and column of a pixel in its block), which have a tap for some entries (tab1: masks as above)
template <int KIND, class Tile, int PER>
struct ConvRingOperand : Tile {
  static_assert(Tile::KC == ((KIND >= 2 && KIND <= 4) || KIND == 7 || KIND == 8), "terms or rows in order of memory");
  static_assert(Tile::REACH == 1 || KIND == 1 || KIND == 3 || KIND >= 5, "the table ends with the last stage");
  using Tile::NG;
  static constexpr int BK = Tile::BK;
  // an entry per group, else one per lane and stage
  static constexpr bool ENT = (KIND == 0 || KIND == 5 || KIND == 6 || KIND == 9) && !(Tile::KPACK >= NG && NG <= PER);
  static constexpr bool LOOKS = KIND != 1 && KIND != 3;
  __amdgpu_buffer_rsrc_t rsrc;
  unsigned off[NG], mask[NG];
  unsigned step;                                                          // KIND 1
  int left;                                                               // KIND 3: terms behind the lane's first one
  const uint2* tab;                                                       // KIND 0, 4 .. 7
  const unsigned* tab1;                                                   // KIND 2, 8, 9
  uint2 ent[ENT ? NG : 1];
  __device__ __forceinline__ void look(int t, int nst) {
    const int at = (t < nst ? t : nst - 1) * (BK / PER);
    if (KIND == 0) {
#pragma unroll
      for (int u = 0; u < (ENT ? NG : 1); ++u) ent[u] = tab[at + Tile::group_k(threadIdx.x, u) / PER];
    }
    if (KIND == 2) ent[0].x = tab1[at + Tile::group_k(threadIdx.x, 0) / PER];
    if (KIND == 4) ent[0] = tab[at + Tile::group_k(threadIdx.x, 0) / PER];
    const int free = t * (BK / PER);                                      // (the table of these reaches over what is asked for)
    if (KIND == 5 || KIND == 6) {
#pragma unroll
      for (int u = 0; u < (ENT ? NG : 1); ++u) {
        const uint2* e = tab + free + Tile::group_k(threadIdx.x, u) / PER;
        ent[u].x = KIND == 5 ? e->x : e->y;
      }
    }
    if (KIND == 7) ent[0].x = tab[free + Tile::group_k(threadIdx.x, 0) / PER].y;
    if (KIND == 9) {
#pragma unroll
      for (int u = 0; u < (ENT ? NG : 1); ++u) {
        const int e = free + Tile::group_k(threadIdx.x, u) / PER;
        ent[u] = make_uint2(tab[e].x, tab1[e]);
      }
    }
    if (KIND == 8) {
      const int e = free + Tile::group_k(threadIdx.x, 0) / PER;
      ent[0] = make_uint2(tab[e].y, tab1[e]);
    }
  }
  __device__ __forceinline__ void fetch(int t, int nst, ring_f32x4 (&r)[NG]) {
    const unsigned behind = (unsigned)(nst - 1 - t) & RING_FAR;           // a stage behind the last one goes nowhere
    if (LOOKS && t == 0) look(0, nst);
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      unsigned o;
      if (KIND == 0) {
        const uint2 e = ent[ENT ? u : 0];
        const unsigned need = e.y | behind;
        o = (mask[u] & need) == need ? off[u] + e.x : RING_FAR;
      } else if (KIND == 1) {
        o = off[u] + (unsigned)t * step;                                  // (beyond the last term: beyond the buffer)
      } else if (KIND == 2) {
        o = (off[u] + ent[0].x) | behind;
      } else if (KIND == 3) {
        o = t * BK < left ? off[u] + (unsigned)(t * BK * 4) : RING_FAR;
      } else if (KIND == 8) {
        o = (mask[u] & ent[0].y) == ent[0].y ? off[u] + ent[0].x : RING_FAR;
      } else if (KIND == 9) {
        o = mask[u] & ent[ENT ? u : 0].y ? RING_FAR : off[u] + ent[ENT ? u : 0].x;
      } else if (KIND >= 5) {
        o = off[u] + ent[ENT ? u : 0].x;
      } else {
        const unsigned have = behind ? 0u : ent[0].y;
        o = (mask[u] & have) == mask[u] ? off[u] + ent[0].x : RING_FAR;
      }
      r[u] = __builtin_bit_cast(ring_f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)o, 0, 0));
    }
    if (LOOKS) look(t + 1, nst);
  }
};

// An output of Down by itself, (y, x) counted from the padding's edge, where the product has terms that this sum has not, with a
// zero for one factor: modules that reach a block but not this pixel (DownM), filters that a tap's last entry repeats (DownM, DownO).
// Where the other factor is not finite, neither is the product's output, whatever this sum is.
__device__ __forceinline__ float conv_down_one(const ConvRingArgs& p, int g, int c, int y, int x, int n) {
  float acc = 0.f;
  const int top = (int)fd_div((uint32_t)y, p.ds), right = (int)fd_div((uint32_t)x, p.ds);
#pragma unroll 1
  for (int my = top < p.Mx - 1 ? top : p.Mx - 1; my >= 0 && y - my * p.s < p.k; --my)
#pragma unroll 1
    for (int mx = right < p.Mx - 1 ? right : p.Mx - 1; mx >= 0 && x - mx * p.s < p.k; --mx) {
      const float* h = p.a + (size_t)p.N * ((size_t)p.M * (g * p.Fg) + my * p.Mx + mx) + n;
      const float* w = p.b + (size_t)p.F * ((c * p.k + y - my * p.s) * p.k + x - mx * p.s) + g * p.Fg;
#pragma unroll 1
      for (int f = 0; f < p.Fg; ++f) acc += h[(size_t)p.N * p.M * f] * w[f];
    }
  return acc;
}

// A convolution pass as a product on the tile loop of ring_tile.h (see there and k_gemm_ring): layers on small and
// mid-sized maps, locally connected layers, and batches that are no multiple of 16, in one launch each.  What bounded
// these on k_conv_mfma: one or two workgroups of four wavefronts per CU that wait for every slab, reductions split over
// workgroups and summed by a second launch, copies of batches and filter counts to whole groups, outputs in blocks of
// 128 rows.  Here the rows of a tile are any run of (module | pixel, image) groups, the loads of four stages are in flight,
// the wavefronts of a workgroup split the stage, and the offset of every 16-byte group is a lane's base plus
// an entry of a table in LDS (what a term of the reduction adds, and a mask for the padding): five vector
// instructions per group and stage.  Tiles of one module or pixel (SINGLE: locally connected layers, batches that are no
// multiple of 4 or that the tile divides) need no masks and leave out the taps beyond the edge.
// convOutp splits its reduction over workgroups and is summed by k_conv_outp_finish*.
// convDown onto few colours (DownM) fills a tile's columns with the pixels of a block beside the colours: k + (b - 1) s rows of taps
// a line where a pixel has k / s, for b s times as many columns; strided layers take tiles of one pixel or one block too, which
// have the taps that exist and no others.  What these took before: a product of all taps and a gather of its outputs
// (a patch matrix, 5 passes over the maps), phases of 128 images, copies of batches and filters to whole groups, or one lane per output.
// Measured, us, operands in the caches, before -> now:
//   96 -> 112 colours 7 x 7, stride 2, 10 x 10, batch 128   131 -> 17      1 -> 64 of 11 x 11, stride 2, 223 x 223, 100    2044 -> 506
//   84 -> 148 of 5 x 5, stride 2, 11 x 11, 100    120 -> 36                3 -> 32 of 5 x 5, 18 x 18, 100     21 -> 11
//   24 -> 93 of 7 x 7, 31 x 31, 151 (whole fours of filters)    645 -> 339
// Filters, colours, images or taps that are fewer than any tile has (13 filters, 9 taps) run on tiles larger than them as well: 60 ->
// 13 colours 7 x 7, 11 x 11, 100 61 -> 23 us Up, 54 -> 21 Outp (before: a copy to 16 filters, or one lane per output).
// Of the random layers that these tiles take about one in forty is more than 4 % slower than before (see conv_pixels_choice); half are
// nearly twice as fast.  (3 -> 96 of 11 x 11, stride 4, 224 x 224, 128, as fast either way, stays on phases of 128 images.)
// Measured, us Up / Down / Outp, operands from memory, before -> now (with the copies and sums):
//   64 -> 64 colours 5 x 5, 13 x 13, batch 100      70 / 62 / 65 -> 46 / 45 / 39      (22 each at 157 TFLOP/s)
//   64 -> 64 colours 3 x 3, 17 x 17, batch 100      69 / 57 / 55 -> 27 / 27 / 32      (14)
//   local 64 -> 64 colours 3 x 3, 8 x 8, batch 128  21 / 20 / 26 -> 11 / 10 / 14      (4)
//   local 48 -> 64 colours 3 x 3, 14 x 14, 100      39 / 37 / 4630 -> 21 / 31 / 27    (7)
//   96 -> 256 colours 5 x 5, 2 groups, 27 x 27, 128 Up 500 -> 412 (9 % of its taps are padding), Outp 532 -> 446; Down
//   449 on k_conv_mfma (48 columns)
// The MFMAs are busy for 81 (Up) and 83 % (Outp) of the time of the last layer, without bank conflicts; without the masks a
// stage takes as long as with them.
// Layers with enough outputs for tiles of 128 x 48 to 128 x 128 (64 x 64 in a few cases) run on the bf16 matrix cores
// (ConvSplitCfg, split_tile.h), where taking the operands apart is as much work as the MFMAs: a number of a map is used by
// as many columns as the tile is wide.  Measured as above, fp32 tile or other kernel -> now:
//   96 -> 256 colours 5 x 5, 2 groups, 27 x 27, 128   Up 413 -> 290 (128 x 128), Down 457 -> 415 (128 x 48), Outp 450 -> 306
//   3 -> 96 colours 11 x 11, stride 4, 224 x 224, 128 Up 260 -> 217 (128 x 96), Outp 237 -> 170 (96 x 128)
//   32 -> 128 colours 3 x 3, 32 x 32, 128             Up 95 -> 68, Outp 91 -> 75
//   64 -> 64 colours 5 x 5, 24 x 24, 128              Outp 128 -> 107 (64 x 128), Up and Down 124 and 118 -> 117 and 117: stay
// Of random passes that they take, 400 took 0.84 times as long as before on one card, one of them more than 3 % longer (6 %);
// 761 0.90 on one whose bf16 products take a sixth longer, 76 more than 3 % longer (22 % at most, 100 images, 72 -> 96 colours 5 x 5,
// 7 x 7, Outp).  Margins for that card cost 2 % on the other.
template <int TB, int BM_, int BN_, int BK_>
struct ConvRingCfg {
  static constexpr int BM = BM_, BN = BN_, BK = BK_, THREADS = RING_THREADS, WAVES = 4;
  static constexpr bool SPLIT = false;
  template <int ROWS, bool KC> using Tile = RingTile<ROWS, BK, KC>;
  template <class OA, class OB> using Shape = RingShape<TB, BM, BN, BK, OA, OB>;
};
// (on the bf16 matrix cores: see split_tile.h)
template <int BM_, int BN_, int BK_, int WM, int WN, int KS, int SETS, int WAVES_>
struct ConvSplitCfg {
  static constexpr int BM = BM_, BN = BN_, BK = BK_, THREADS = 64 * WM * WN * KS, WAVES = WAVES_;
  static constexpr bool SPLIT = true;
  template <int ROWS, bool KC> using Tile = SplitTile<ROWS, BK, KC, THREADS>;
  template <class OA, class OB> using Shape = SplitShape<BM, BN, BK, WM, WN, KS, SETS, OA, OB>;
};
// LOOSE: of a tile that may be larger than all rows or columns there are.  (Instances of their own: with the bounds that it needs
// convUp of the locally connected layer above takes 8.80 us instead of 8.70.)
template <int MODE, bool SINGLE, bool LOOSE, class Cfg>
__global__ void __launch_bounds__(Cfg::THREADS, Cfg::WAVES) k_conv_ring(ConvRingArgs p) {
  constexpr int PER = MODE == CONV_UP ? 1 : 4, BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK, THREADS = Cfg::THREADS;
  using OA = ConvRingOperand<MODE == CONV_OUTP ? 3 : MODE == CONV_DOWNM ? 9 : SINGLE ? 5 : 0, typename Cfg::template Tile<BM, MODE == CONV_OUTP>, PER>;
  using OB = ConvRingOperand<MODE == CONV_UP ? (SINGLE ? 6 : 1) : MODE == CONV_OUTP ? 4 : MODE == CONV_DOWNM ? 8 : SINGLE ? 7 : 2,
                             typename Cfg::template Tile<BN, MODE != CONV_UP>, PER>;
  using Shape = typename Cfg::template Shape<OA, OB>;
  constexpr int EPL = Shape::EPL, LDS = Cfg::SPLIT ? Shape::LDS : 4 * Shape::LDS;
  static_assert(LDS == (Cfg::SPLIT ? conv_split_lds(BM, BN, BK) : conv_ring_lds(MODE, BM, BN, BK)) && LDS + RING_TABLE_BYTES <= RING_CU_LDS,
                "as planned");
  if constexpr (Cfg::SPLIT && SINGLE) {
    constexpr int reach = OA::REACH > OB::REACH ? OA::REACH : OB::REACH;
    static_assert(RING_AHEAD >= Shape::AHEAD + 1 + reach, "fetch() looks one stage ahead, and a lane's entry may lie reach - 1 stages behind that");
  }
  __shared__ __attribute__((aligned(16))) char lds[LDS];
  extern __shared__ uint2 table[];
  const int tid = threadIdx.x;
  const int N = p.N, H = p.H, Mx = p.Mx, k = p.k;
  // each XCD gets a contiguous run of tiles, the column tiles of a row tile one after the other
  const int tiles = p.periods * p.gx * p.gy * p.gz, run = (tiles + 7) >> 3;
  int t = (int)(blockIdx.x & 7) * run + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= run || t >= tiles) return;
  auto div = [](int v, const FastDiv& d) { return (int)fd_div((uint32_t)v, d); };
  int rest = div(t, p.dgy);
  const int by = t - rest * p.gy;
  t = rest; rest = div(t, p.dgx);
  const int bx = t - rest * p.gx, z = div(rest, p.dper), per = rest - z * p.periods;
  // a tile over the edge moves back inside; the outputs it shares with its neighbour are that one's to store (of a tile larger than
  // all there is, rows and columns behind the last are computed from what stands there, or zeros, and not stored)
  const int m_lo = bx * BM, n_lo = by * BN;
  const int m0 = m_lo + BM <= p.rows || (LOOSE && p.rows < BM) ? m_lo : p.rows - BM;
  const int n0 = n_lo + BN <= p.cols || (LOOSE && p.cols < BN) ? n_lo : p.cols - BN;

  OA oa; OB ob;
  int nst, g = z;
  float* out = p.out;
  if constexpr (SINGLE) {
    // One module or pixel: taps that leave the image, or reach no module, are left out.  Up: the others are rows ky0 ..
    // ky0 + ny - 1 and columns kx0 .. kx0 + nx - 1 of the filter.  Down: modules my0, my0 - 1 .. my0 - ny + 1 (of a line) have the
    // pixel at rows ky0, ky0 + s ..; a block of pixels: the tap of its first pixel there, which may lie outside the filter.
    constexpr bool UP = MODE == CONV_UP, MERGED = MODE == CONV_DOWNM, ONE = MODE == CONV_DOWN;      // ONE: of stride 1
    const int s = ONE ? 1 : p.s, blocks = MERGED ? div(p.block, p.ds) : 1;
    const int line = div(per, UP ? p.dMx : MERGED ? p.dlines : p.dH), at = per - line * (UP ? Mx : MERGED ? p.lines : H);
    const int y = UP ? line * s + p.pad0 : MERGED ? line * p.block : line - p.pad0, x = UP ? at * s + p.pad0 : MERGED ? at * p.block : at - p.pad0;
    auto range = [&](int v, int* first, int* m_first) {
      if (UP) {
        *first = -v > 0 ? -v : 0;
        return (H - v < k ? H - v : k) - *first;
      }
      if (ONE) {
        *first = v - Mx + 1 > 0 ? v - Mx + 1 : 0;
        *m_first = v - *first;
        return (v + 1 < k ? v + 1 : k) - *first;
      }
      const int top = div(v, p.ds) + blocks - 1, m = top < Mx - 1 ? top : Mx - 1, reach = MERGED ? k + s * (blocks - 1) : k;
      *m_first = m;
      *first = v - s * m;                                               // (from -s (blocks - 1) on)
      const int n = *first < k ? div(reach - 1 - (*first + s * (blocks - 1)), p.ds) + 1 : 0;
      return n < m + 1 ? n : m + 1;
    };
    int ky0, kx0, my0 = 0, mx0 = 0;
    int ny = range(y, &ky0, &my0), nx = range(x, &kx0, &mx0);
    if (ny <= 0 || nx <= 0) { ny = 0; nx = 1; }
    const int Fg4 = MERGED ? p.Fg4() : p.Fg, area = ny * nx, K = area * (UP ? p.Cg : Fg4);
    nst = K > BK ? (K + BK - 1) / BK : 1;
    unsigned* tab1 = reinterpret_cast<unsigned*>(table + (nst + RING_AHEAD) * (BK / PER));
    // exact for dividends below 2^12 and divisors up to RING_MAX_SIDE^2
    const unsigned inv_nx = 65536u / (unsigned)nx + 1u, inv_area = (1u << 20) / (unsigned)(area > 0 ? area : 1) + 1u;
    const unsigned Nu = (unsigned)N, Fu = (unsigned)p.F;
    for (int e = tid; e < (nst + RING_AHEAD) * (BK / PER); e += THREADS) {
      uint2 t2 = make_uint2(RING_FAR, RING_FAR);
      unsigned need = 0u;
      if (PER * e < K) {
        const int c = UP ? (int)((unsigned)e * inv_area >> 20) : 0;
        const int tap = UP ? e - c * area : div(4 * e, p.dFg4);
        const int ty = (int)((unsigned)tap * inv_nx >> 16), tx = tap - ty * nx;
        if (UP) {
          const int bank = p.local ? per : 0, ky = ky0 + ty, kx = kx0 + tx;
          t2.x = 4u * Nu * (unsigned)((g * p.Cg + c) * p.HH + (y + ky) * H + x + kx);
          t2.y = 4u * Fu * (unsigned)((bank * p.Cg + c) * p.kk2 + ky * k + kx);
        } else {
          const int ky = ky0 + s * ty, kx = kx0 + s * tx, m = ONE ? (y - ky) * Mx + x - kx : (my0 - ty) * Mx + mx0 - tx;
          int f = 4 * e - tap * Fg4;
          if (MERGED && f + 4 > p.Fg) { f = p.Fg - 4; need = RING_LAST; }
          t2.x = 4u * Nu * (unsigned)(p.M * (g * p.Fg + f) + m);
          t2.y = 4u * ((unsigned)f + Fu * (unsigned)(ky * k + kx + p.Cg * p.kk2 * (p.local ? m : 0)));
          // (the first pixel's row and column, from -s (blocks - 1) on, in steps of s; a lane's mask says with which its own has a tap)
          if (MERGED) need |= 1u << (div(ky + s * (blocks - 1), p.ds)) | 1u << (RING_MAX_SIDE + div(kx + s * (blocks - 1), p.ds));
        }
      }
      table[e] = t2;
      if (MERGED) tab1[e] = need;
    }
    oa.tab = ob.tab = table;
    const int n = m0 + OA::group_row(tid, 0);
#pragma unroll
    for (int u = 0; u < OA::NG; ++u) {
      oa.off[u] = 4u * (unsigned)(n + (PER == 4 ? N * p.M * (OA::group_k(tid, u) % 4) : 0));
      if (MERGED) oa.mask[u] = OA::group_k(tid, u) % 4 < Fg4 - p.Fg ? RING_LAST : 0u;
    }
#pragma unroll
    for (int u = 0; u < OB::NG; ++u) {
      const int col = n0 + OB::group_row(tid, u);
      if (MERGED) {
        const int c = div(col, p.dblock2), q = col - c * p.block * p.block, py = div(q, p.dblock), px = q - py * p.block;
        ob.off[u] = 4u * (unsigned)(g * p.Fg + p.F * (c * p.kk2 + py * k + px));
        // rows 0 <= first + py < k of the filter, first = s (t - blocks + 1), as bits t
        auto taps = [&](int q0) {
          const int back = s * (blocks - 1) - q0;                       // first + q0 = s t - back
          return ring_bits(back > 0 ? div(back + s - 1, p.ds) : 0, back + k > 0 ? div(back + k - 1, p.ds) + 1 : 0);
        };
        ob.mask[u] = col < p.cols ? taps(py) | taps(px) << RING_MAX_SIDE | RING_LAST : 0u;
      } else {
        ob.off[u] = 4u * (unsigned)(g * p.Fg + (MODE == CONV_UP ? col : p.F * p.kk2 * col));
      }
    }
    if (MERGED) oa.tab1 = ob.tab1 = tab1;
    ob.rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p.b, 0, (int)p.b_bytes, 0x00020000);
    if (MERGED) out += (long long)g * p.Cg * p.HH * N;
    else out += (long long)g * p.cols * p.ldc + (long long)per * p.rows;
  } else if constexpr (MODE == CONV_UP) {
    const int K = p.Cg * p.kk2;
    nst = (K + BK - 1) / BK;
    for (int e = tid; e < nst * BK; e += THREADS) {
      const int c = div(e, p.dkk2), tap = e - c * p.kk2, ky = div(tap, p.dk), kx = tap - ky * k;
      table[e] = e < K ? make_uint2(4u * (unsigned)N * (unsigned)(c * p.HH + ky * H + kx), 1u << ky | 1u << (RING_MAX_SIDE + kx))
                       : make_uint2(0u, RING_FAR);
    }
    const int r = m0 + OA::group_row(tid, 0);
    const int m = div(r, p.dN), n = r - m * N, my = div(m, p.dMx), mx = m - my * Mx;
    const int y = my * p.s + p.pad0, x = mx * p.s + p.pad0;
#pragma unroll
    for (int u = 0; u < OA::NG; ++u) {
      oa.off[u] = 4u * (unsigned)(n + N * (y * H + x + g * p.Cg * p.HH));
      oa.mask[u] = ring_bits(-y, H - y < k ? H - y : k) | ring_bits(-x, H - x < k ? H - x : k) << RING_MAX_SIDE;
    }
    oa.tab = table;
    ob.rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p.b, 0, (int)(4u * (unsigned)K * (unsigned)p.F), 0x00020000);
    ob.step = 4u * BK * (unsigned)p.F;
#pragma unroll
    for (int u = 0; u < OB::NG; ++u)
      ob.off[u] = 4u * (unsigned)(OB::group_k(tid, u) * p.F + g * p.Fg + n0 + OB::group_row(tid, u));
    out += (long long)g * p.Fg * p.ldc;
  } else if constexpr (MODE == CONV_DOWN || MODE == CONV_DOWNO) {
    constexpr bool ODD = MODE == CONV_DOWNO;
    const int Fg4 = ODD ? p.Fg4() : p.Fg, K = p.kk2 * Fg4;
    nst = (K + BK - 1) / BK;
    unsigned* tab1 = reinterpret_cast<unsigned*>(table + nst * (BK / 4));
    for (int e = tid; e < nst * (BK / 4); e += THREADS) {
      const int tap = div(4 * e, p.dFg4), f0 = 4 * e - tap * Fg4, f = ODD && f0 + 4 > p.Fg ? p.Fg - 4 : f0, ky = div(tap, p.dk), kx = tap - ky * k;
      const bool in = 4 * e < K;
      table[e] = make_uint2(4u * (unsigned)N * (unsigned)(p.M * f - ky * Mx - kx),
                            in ? 1u << ky | 1u << (RING_MAX_SIDE + kx) | (f < f0 ? RING_LAST : 0u) : RING_FAR);
      tab1[e] = in ? 4u * (unsigned)(f + p.F * tap) : RING_FAR;
    }
    const int r = m0 + OA::group_row(tid, 0);
    const int pix = div(r, p.dN), n = r - pix * N, yy = div(pix, p.dH), y = yy - p.pad0, x = pix - yy * H - p.pad0;
#pragma unroll
    for (int u = 0; u < OA::NG; ++u) {
      oa.off[u] = 4u * (unsigned)(n + N * (y * Mx + x + p.M * (g * p.Fg + OA::group_k(tid, u) % 4)));
      oa.mask[u] = ring_bits(y - Mx + 1, y + 1 < k ? y + 1 : k) | ring_bits(x - Mx + 1, x + 1 < k ? x + 1 : k) << RING_MAX_SIDE;
      if (ODD && OA::group_k(tid, u) % 4 >= Fg4 - p.Fg) oa.mask[u] |= RING_LAST;
    }
    oa.tab = table;
    ob.tab1 = tab1;
    ob.rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p.b, 0, (int)p.b_bytes, 0x00020000);
#pragma unroll
    for (int u = 0; u < OB::NG; ++u) ob.off[u] = 4u * (unsigned)(g * p.Fg + p.F * p.kk2 * (n0 + OB::group_row(tid, u)));
    out += (long long)g * p.Cg * p.ldc;
  } else {
    const int cz = div(z, p.dG), chunk = div(cz, p.dsplits), k_beg = (cz - chunk * p.splits) * p.split_stages * BK;
    g = z - cz * p.G;
    const int count = p.K - k_beg < p.split_stages * BK ? p.K - k_beg : p.split_stages * BK, first = chunk * p.m_count * N + k_beg;
    nst = (count + BK - 1) / BK;
    for (int e = tid; e < nst * (BK / 4); e += THREADS) {
      const int r = first + 4 * e, m = div(r, p.dN), n = r - m * N, my = div(m, p.dMx), mx = m - my * Mx;
      const int y = my * p.s + p.pad0, x = mx * p.s + p.pad0;
      table[e] = 4 * e < count ? make_uint2(4u * (unsigned)(n + N * (y * H + x)),
                                            ring_bits(-y, H - y < k ? H - y : k) | ring_bits(-x, H - x < k ? H - x : k) << RING_MAX_SIDE)
                               : make_uint2(0u, 0u);
    }
    const int kl = OA::group_k(tid, 0);
    oa.left = count - kl;
#pragma unroll
    for (int u = 0; u < OA::NG; ++u)
      oa.off[u] = 4u * ((unsigned)(g * p.Fg + m0 + OA::group_row(tid, u)) * (unsigned)(N * p.M) + (unsigned)(first + kl));
#pragma unroll
    for (int u = 0; u < OB::NG; ++u) {
      const int q = n0 + OB::group_row(tid, u), c = div(q, p.dkk2), tap = q - c * p.kk2, ky = div(tap, p.dk), kx = tap - ky * k;
      ob.off[u] = 4u * (unsigned)N * (unsigned)((g * p.Cg + c) * p.HH + ky * H + kx);
      ob.mask[u] = 1u << ky | 1u << (RING_MAX_SIDE + kx);
    }
    ob.tab = table;
    ob.rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p.b, 0, (int)p.b_bytes, 0x00020000);
    out += cz * p.out_stride + (p.splits > 1 ? (long long)g * p.Fg * p.cols : (long long)g * p.Fg);
  }
  oa.rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p.a, 0, (int)p.a_bytes, 0x00020000);
  __syncthreads();

  // output (em, en) of the tile: at column en, or (DownM) at the pixel that it stands for, which may lie outside the map
  const unsigned ms = (unsigned)((m0 + BM < p.rows ? m0 + BM : p.rows) - m_lo), ns = (unsigned)((n0 + BN < p.cols ? n0 + BN : p.cols) - n_lo);
  auto place = [&](int em, int en, long long* at) __attribute__((always_inline)) {
    if (LOOSE ? (unsigned)(em - m_lo) >= ms || (unsigned)(en - n_lo) >= ns : em < m_lo || en < n_lo) return false;
    if constexpr (MODE == CONV_DOWNM) {
      const int line = div(per, p.dlines), col = per - line * p.lines;
      const int c = div(en, p.dblock2), q = en - c * p.block * p.block, py = div(q, p.dblock), px = q - py * p.block;
      const int y = line * p.block + py + p.pad0, x = col * p.block + px + p.pad0;
      *at = (long long)(c * p.HH + y * H + x) * N + em;
      return (unsigned)y < (unsigned)H && (unsigned)x < (unsigned)H;
    }
    *at = (long long)en * p.ldc + em;
    return true;
  };
  constexpr bool AGAIN = MODE == CONV_DOWNM || MODE == CONV_DOWNO;        // see conv_down_one
  bool again = false;
  auto store = [&](int em, int en, float v) __attribute__((always_inline)) {
    long long at;
    if (!place(em, en, &at)) return;
    if (AGAIN) again |= !(__builtin_fabsf(v) < __builtin_inff());
    out[at] = v;
  };
  if constexpr (Cfg::SPLIT) {
    Shape::template run<false>(lds, oa, ob, nst, 0, [] {});
#pragma unroll
    for (int u = 0; u < EPL; ++u) {
      const int e = tid + THREADS * u;
      store(m0 + e % BM, n0 + e / BM, Shape::sum(lds, tid, u));
    }
  } else {
    float sum[EPL];
    Shape::template run<false, false>(reinterpret_cast<float*>(lds), oa, ob, nst, 0, sum, [] {});
    const int em = m0 + tid % BM, en0 = n0 + tid / BM;
#pragma unroll
    for (int u = 0; u < EPL; ++u) store(em, en0 + u * (THREADS / BM), sum[u]);
  }
  if (AGAIN && again) {
#pragma unroll 1
    for (int u = 0; u < EPL; ++u) {
      const int e = tid + THREADS * u, em = m0 + e % BM;
      long long at;
      if (!place(em, n0 + e / BM, &at) || __builtin_fabsf(out[at]) < __builtin_inff()) continue;
      // [colour][pixel][image], of a group's first colour on (ring_ok: 31 bits)
      const int row = (int)at / N, c = row / p.HH, pix = row - c * p.HH, y = pix / H, x = pix - y * H;
      out[at] = conv_down_one(p, g, c, y - p.pad0, x - p.pad0, (int)at - row * N);
    }
  }
}

// (of these modes there is no instance without LOOSE: their layers are of few colours, odd or strided, and mostly small)
static constexpr bool conv_always_loose(int mode) { return mode == CONV_DOWNM || mode == CONV_DOWNS || mode == CONV_DOWNO; }
template <int MODE, bool SINGLE, class Cfg>
static void conv_ring_go(const ConvRingArgs& p, dim3 grid, size_t tab) {
  constexpr bool may = conv_may_be_loose(MODE, Cfg::SPLIT), always = may && conv_always_loose(MODE);
  if constexpr (may) {
    if (always || p.rows < Cfg::BM || p.cols < Cfg::BN) {
      hipLaunchKernelGGL((k_conv_ring<MODE, SINGLE, true, Cfg>), grid, dim3(Cfg::THREADS), tab, dn_stream(), p);
      return;
    }
  }
  if constexpr (!always) hipLaunchKernelGGL((k_conv_ring<MODE, SINGLE, false, Cfg>), grid, dim3(Cfg::THREADS), tab, dn_stream(), p);
}

template <int MODE, bool SINGLE>
static void conv_ring_launch(const ConvRingPlan& plan, ConvRingArgs p) {
  const ConvRingTile f = conv_ring_cfg(MODE, plan.cfg);
  p.gx = (p.rows + f.bm - 1) / f.bm; p.gy = (p.cols + f.bn - 1) / f.bn;
  const long long tiles = (long long)p.periods * p.gx * p.gy * p.gz;
  const dim3 grid((unsigned)(8 * ((tiles + 7) / 8)));
  const int stages = MODE == CONV_OUTP ? plan.split_stages : (p.K + f.bk - 1) / f.bk;
  p.dN = make_fastdiv(p.N); p.dH = make_fastdiv(p.H); p.dFg4 = make_fastdiv(p.Fg4()); p.dG = make_fastdiv(p.G);
  p.dgx = make_fastdiv(p.gx); p.dgy = make_fastdiv(p.gy); p.dper = make_fastdiv(p.periods);
  p.dsplits = make_fastdiv(MODE == CONV_OUTP ? p.splits : p.s);
  p.dMx = make_fastdiv(MODE == CONV_DOWNM ? p.lines : p.Mx);
  p.dk = make_fastdiv(MODE == CONV_DOWNM ? p.block : p.k);
  p.dkk2 = make_fastdiv(MODE == CONV_DOWNM ? p.block * p.block : p.kk2);
  const size_t tab = (size_t)conv_ring_table(MODE, SINGLE, f.bk, stages);
#define CONV_RING(...) conv_ring_go<MODE, SINGLE, __VA_ARGS__>(p, grid, tab)
  switch (plan.cfg) {
    case 0: CONV_RING(ConvRingCfg<32, 64, 64, 32>); break;
    case 1: CONV_RING(ConvRingCfg<32, 64, 32, 64>); break;
    case 2: CONV_RING(ConvRingCfg<32, 32, 64, 64>); break;
    case 3: CONV_RING(ConvRingCfg<16, 32, 32, 64>); break;
    case 4: CONV_RING(ConvRingCfg<16, 32, 16, 128>); break;
    case 5: CONV_RING(ConvRingCfg<16, 16, 32, 128>); break;
    case 6: CONV_RING(ConvSplitCfg<128, 128, 32, 2, 4, 1, 2, 2>); break;
    case 7: if constexpr (MODE == CONV_OUTP) CONV_RING(ConvSplitCfg<96, 128, 32, 2, 4, 1, 2, 2>); else CONV_RING(ConvSplitCfg<128, 96, 32, 4, 2, 1, 2, 2>); break;
    case 8: if constexpr (MODE == CONV_OUTP) CONV_RING(ConvSplitCfg<64, 128, 32, 2, 4, 1, 2, 2>); else CONV_RING(ConvSplitCfg<128, 64, 32, 4, 2, 1, 2, 2>); break;
    case 9: CONV_RING(ConvSplitCfg<64, 64, 32, 2, 2, 1, 2, 3>); break;
    default: if constexpr (conv_ring_cfg(MODE, 10).bm != 0) CONV_RING(ConvSplitCfg<128, 48, 64, 4, 1, 2, 2, 2>); break;
  }
#undef CONV_RING
}
