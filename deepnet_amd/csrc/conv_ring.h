// Convolution passes on the tile loop of ring_tile.h: see k_conv_ring.  Included by conv.hip (ConvArgs).
#pragma once
#include "ring_tile.h"

// A term of the reduction, as the workgroup keeps it in LDS for its reduction (one entry per term for Up, per four
// for Down and Outp): the byte offset that it adds to a lane's, and which filter rows (bits 0-14) and columns (15-29)
// have to be inside (Up, Down: `mask` of the entry has to be part of the lane's) or are inside (Outp: the other way
// round).  RING_FAR stands in no lane's mask: such a term reads as zero.
#define RING_FAR 0x80000000u
#define RING_MAX_SIDE 15
__device__ __forceinline__ unsigned ring_bits(int lo, int hi) {      // bits lo .. hi - 1
  lo = lo < 0 ? 0 : lo;
  hi = hi < lo ? lo : hi;
  return ((1u << hi) - 1u) & ~((1u << lo) - 1u);
}

struct ConvRingArgs {
  const float* a; const float* b;
  float* out;
  unsigned a_bytes, b_bytes;
  int N, H, HH, Mx, M, k, kk2, s, pad0, Cg, Fg, F, G;
  int local;                    // one filter bank per module
  int rows, cols;               // of one period: a tile lies inside one (one module or pixel, or everything)
  int periods, gx, gy, gz;      // tiles per period down the rows, across; Up / Down: groups; Outp: chunks x splits x groups
  int K;                        // Outp: terms of a chunk
  int m_count, splits, split_stages;
  FastDiv dN, dMx, dk, dkk2, dH, dFg, dgx, dgy, dper, dsplits, dG;
  long long ldc, out_stride;    // of a column; Outp: of a (chunk, split)
};

// Operand of a convolution stage: offsets and masks from the table of the workgroup's reduction.
// KIND 0: rows are (module | pixel, image) groups, a table entry per PER terms (A of Up and Down)
//      1: rows are filters, terms in order of memory (B of Up)
//      2: rows are colours, four filters of a tap per entry (B of Down)
//      3: rows are filters, terms (module, image) in order of memory (A of Outp)
//      4: rows are taps, four images of a module per entry (B of Outp)
template <int KIND, int ROWS, int BK, int PER>
struct ConvRingOperand : RingTile<ROWS, BK, (KIND >= 2)> {
  using Tile = RingTile<ROWS, BK, (KIND >= 2)>;
  using Tile::NG;
  static constexpr bool ENT = KIND == 0;                                  // an entry per group, else one per lane and stage
  __amdgpu_buffer_rsrc_t rsrc;
  unsigned off[NG], mask[NG];
  unsigned step;                                                          // KIND 1
  int left;                                                               // KIND 3: terms behind the lane's first one
  const uint2* tab;                                                       // KIND 0, 4
  const unsigned* tab1;                                                   // KIND 2
  uint2 ent[ENT ? NG : 1];
  __device__ __forceinline__ void look(int t, int nst) {
    const int at = (t < nst ? t : nst - 1) * (BK / PER);
    if (KIND == 0) {
#pragma unroll
      for (int u = 0; u < NG; ++u) ent[u] = tab[at + Tile::group_k(threadIdx.x, u) / PER];
    }
    if (KIND == 2) ent[0].x = tab1[at + Tile::group_k(threadIdx.x, 0) / PER];
    if (KIND == 4) ent[0] = tab[at + Tile::group_k(threadIdx.x, 0) / PER];
  }
  __device__ __forceinline__ void fetch(int t, int nst, ring_f32x4 (&r)[NG]) {
    const unsigned behind = (unsigned)(nst - 1 - t) & RING_FAR;           // a stage behind the last one goes nowhere
    if (KIND == 0 || KIND == 2 || KIND == 4) { if (t == 0) look(0, nst); }
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      unsigned o;
      if (KIND == 0) {
        const unsigned need = ent[u].y | behind;
        o = (mask[u] & need) == need ? off[u] + ent[u].x : RING_FAR;
      } else if (KIND == 1) {
        o = off[u] + (unsigned)t * step;                                  // (beyond the last term: beyond the buffer)
      } else if (KIND == 2) {
        o = (off[u] + ent[0].x) | behind;
      } else if (KIND == 3) {
        o = t * BK < left ? off[u] + (unsigned)(t * BK * 4) : RING_FAR;
      } else {
        const unsigned have = behind ? 0u : ent[0].y;
        o = (mask[u] & have) == mask[u] ? off[u] + ent[0].x : RING_FAR;
      }
      r[u] = __builtin_bit_cast(ring_f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)o, 0, 0));
    }
    if (KIND == 0 || KIND == 2 || KIND == 4) look(t + 1, nst);
  }
};

// A convolution pass as a product on the tile loop of ring_tile.h (see there and k_gemm_ring): layers on small and
// mid-sized maps, locally connected layers, and batches that are no multiple of 16, in one launch each.  What bounded
// these on k_conv_mfma: one or two workgroups of four wavefronts per CU that wait for every slab, reductions split over
// workgroups and summed by a second launch, copies of batches and filter counts to whole groups, outputs in blocks of
// 128 rows.  Here the rows of a tile are any run of (module | pixel, image) groups, the loads of four stages are in flight,
// the wavefronts of a workgroup split the stage, and the offset of every 16-byte group is a lane's base plus
// an entry of a table in LDS (what a term of the reduction adds, and a mask for the padding): five vector
// instructions per group and stage.  Tiles of one module or pixel (locally connected layers, batches that are no
// multiple of 4) need the batch only to be as large as the tile; convDown then leaves out taps beyond the modules.
// convOutp splits its reduction over workgroups and is summed by k_conv_outp_finish*.
// Measured, us Up / Down / Outp, before -> now (with the copies and sums):
//   64 -> 64 colours 5 x 5, 13 x 13, batch 100      72 / 63 / 66 -> 49 / 48 / 39      (22 each at 157 TFLOP/s)
//   64 -> 64 colours 3 x 3, 17 x 17, batch 100      69 / 58 / 55 -> 25 / 26 / 29      (14)
//   local 64 -> 64 colours 3 x 3, 8 x 8, batch 128  20 / 19 / 25 -> 10 / 10 / 14      (4)
//   local 48 -> 64 colours 3 x 3, 14 x 14, 100      38 / 37 / 4570 -> 20 / 28 / 25    (7)
//   96 -> 256 colours 5 x 5, 2 groups, 27 x 27, 128 Outp 539 -> 470; Up 540 and Down 483 on either
// A stage takes 1.25 times its MFMAs: the offsets, and LDS reads of one value per lane for operands that are not
// contiguous along the reduction.
template <int MODE, int TB, int BM, int BN, int BK>
__global__ void __launch_bounds__(RING_THREADS, 4) k_conv_ring(ConvRingArgs p) {
  constexpr int PER = MODE == CONV_UP ? 1 : 4;
  using OA = ConvRingOperand<MODE == CONV_OUTP ? 3 : 0, BM, BK, PER>;
  using OB = ConvRingOperand<MODE == CONV_UP ? 1 : MODE == CONV_DOWN ? 2 : 4, BN, BK, PER>;
  using Shape = RingShape<TB, BM, BN, BK, OA, OB>;
  constexpr int EPL = Shape::EPL;
  __shared__ __attribute__((aligned(16))) float lds[Shape::LDS];
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
  // a tile over the edge moves back inside; the outputs it shares with its neighbour are that one's to store
  const int m_lo = bx * BM, n_lo = by * BN;
  const int m0 = m_lo + BM <= p.rows ? m_lo : p.rows - BM, n0 = n_lo + BN <= p.cols ? n_lo : p.cols - BN;

  OA oa; OB ob;
  int nst, g = z;
  float* out = p.out;
  if constexpr (MODE == CONV_UP) {
    const int K = p.Cg * p.kk2;
    nst = (K + BK - 1) / BK;
    for (int e = tid; e < nst * BK; e += RING_THREADS) {
      const int c = div(e, p.dkk2), tap = e - c * p.kk2, ky = div(tap, p.dk), kx = tap - ky * k;
      table[e] = e < K ? make_uint2(4u * (unsigned)N * (unsigned)(c * p.HH + ky * H + kx), 1u << ky | 1u << (RING_MAX_SIDE + kx))
                       : make_uint2(0u, RING_FAR);
    }
    const int r = per * p.rows + m0 + OA::group_row(tid, 0);
    const int m = div(r, p.dN), n = r - m * N, my = div(m, p.dMx), mx = m - my * Mx;
    const int y = my * p.s + p.pad0, x = mx * p.s + p.pad0;
#pragma unroll
    for (int u = 0; u < OA::NG; ++u) {
      oa.off[u] = 4u * (unsigned)(n + N * (y * H + x + g * p.Cg * p.HH));
      oa.mask[u] = ring_bits(-y, H - y < k ? H - y : k) | ring_bits(-x, H - x < k ? H - x : k) << RING_MAX_SIDE;
    }
    oa.tab = table;
    const int bank = p.local ? per : 0;
    const unsigned bank_bytes = 4u * (unsigned)K * (unsigned)p.F;
    ob.rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(p.b + (size_t)bank * K * p.F), 0, (int)bank_bytes, 0x00020000);
    ob.step = 4u * BK * (unsigned)p.F;
#pragma unroll
    for (int u = 0; u < OB::NG; ++u)
      ob.off[u] = 4u * (unsigned)(OB::group_k(tid, u) * p.F + g * p.Fg + n0 + OB::group_row(tid, u));
    out += (long long)g * p.Fg * p.ldc + (long long)per * p.rows;
  } else if constexpr (MODE == CONV_DOWN) {
    // a tile on one pixel leaves out the taps that reach no module: they are the rows and columns ky0.. and kx0.. of the filter
    int ky0 = 0, kx0 = 0, ny = k, nx = k;
    const int prow = div(per, p.dH), py = prow - p.pad0, px = per - prow * H - p.pad0;
    if (p.periods > 1) {
      ky0 = py - Mx + 1 > 0 ? py - Mx + 1 : 0; ny = (py + 1 < k ? py + 1 : k) - ky0;
      kx0 = px - Mx + 1 > 0 ? px - Mx + 1 : 0; nx = (px + 1 < k ? px + 1 : k) - kx0;
      if (ny <= 0 || nx <= 0) ny = 0, nx = 1;
    }
    const int K = ny * nx * p.Fg;
    nst = (K + BK - 1) / BK;
    if (nst < 1) nst = 1;
    const int inv_nx = 65536 / nx + 1;      // exact for tap < RING_MAX_SIDE^2
    unsigned* tab1 = reinterpret_cast<unsigned*>(table + nst * (BK / 4));
    for (int e = tid; e < nst * (BK / 4); e += RING_THREADS) {
      const int tap = div(4 * e, p.dFg), f = 4 * e - tap * p.Fg, ty = tap * inv_nx >> 16, ky = ky0 + ty, kx = kx0 + tap - ty * nx;
      const int bank = p.local ? (py - ky) * Mx + px - kx : 0;
      const bool in = 4 * e < K;
      table[e] = make_uint2(4u * (unsigned)N * (unsigned)(p.M * f - ky * Mx - kx), in ? 1u << ky | 1u << (RING_MAX_SIDE + kx) : RING_FAR);
      tab1[e] = in ? 4u * (unsigned)(f + p.F * (ky * k + kx + p.Cg * p.kk2 * bank)) : RING_FAR;
    }
    const int r = per * p.rows + m0 + OA::group_row(tid, 0);
    const int pix = div(r, p.dN), n = r - pix * N, yy = div(pix, p.dH), y = yy - p.pad0, x = pix - yy * H - p.pad0;
#pragma unroll
    for (int u = 0; u < OA::NG; ++u) {
      oa.off[u] = 4u * (unsigned)(n + N * (y * Mx + x + p.M * (g * p.Fg + OA::group_k(tid, u) % 4)));
      oa.mask[u] = ring_bits(y - Mx + 1, y + 1 < k ? y + 1 : k) | ring_bits(x - Mx + 1, x + 1 < k ? x + 1 : k) << RING_MAX_SIDE;
    }
    oa.tab = table;
    ob.tab1 = tab1;
    ob.rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p.b, 0, (int)p.b_bytes, 0x00020000);
#pragma unroll
    for (int u = 0; u < OB::NG; ++u) ob.off[u] = 4u * (unsigned)(g * p.Fg + p.F * p.kk2 * (n0 + OB::group_row(tid, u)));
    out += (long long)g * p.Cg * p.ldc + (long long)per * p.rows;
  } else {
    const int cz = div(z, p.dG), chunk = div(cz, p.dsplits), k_beg = (cz - chunk * p.splits) * p.split_stages * BK;
    g = z - cz * p.G;
    const int count = p.K - k_beg < p.split_stages * BK ? p.K - k_beg : p.split_stages * BK, first = chunk * p.m_count * N + k_beg;
    nst = (count + BK - 1) / BK;
    for (int e = tid; e < nst * (BK / 4); e += RING_THREADS) {
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

  float sum[EPL];
  Shape::template run<false>(lds, oa, ob, nst, 0, sum, [] {});
  const int em = m0 + tid % BM, en0 = n0 + tid / BM;
#pragma unroll
  for (int u = 0; u < EPL; ++u) {
    const int en = en0 + u * (RING_THREADS / BM);
    if (em >= m_lo && en >= n_lo) {
      out[(long long)en * p.ldc + em] = sum[u];
    }
  }
}

// The tiles and what they cost: us per stage and per tile of a round (a tile on every CU).  Fitted to 233 measured
// passes (rms 3 to 5 %); behind a product's 0.43 us a stage are the lanes' offsets, and what a tile costs besides its
// stages is its table and its first trip to memory.
static const struct { int bm, bn, bk; double stage, tile; } g_conv_ring_cfgs[] = {
    {64, 64, 32, 0.53, 1.62}, {64, 32, 64, 0.60, 1.61}, {32, 64, 64, 0.59, 1.55},
    {32, 32, 64, 0.344, 1.21}, {32, 16, 128, 0.414, 1.27}, {16, 32, 128, 0.41, 1.25}};
#define RING_TABLE_BYTES 26624      // what a workgroup's LDS holds besides the tiles (64 KB in all)

struct ConvRingPlan { int cfg, splits, split_stages; double us; };

// The tile that is expected to be fastest, cfg < 0: none fits.  rows x cols outputs per period, `jobs` periods x groups x
// chunks, K terms each, of which a tile has the share `used` on average; split_us: what adding up one more
// partial output costs (Outp).
static ConvRingPlan conv_ring_plan(int mode, long long rows, int cols, long long jobs, int K, double used, bool can_split, double split_us) {
  ConvRingPlan best = {-1, 1, 0, 0.};
  const int cus = dn_num_cus();
  for (int c = 0; c < 6; ++c) {
    const auto& f = g_conv_ring_cfgs[c];
    if (rows < f.bm || cols < f.bn) continue;
    const long long tiles = (rows + f.bm - 1) / f.bm * ((cols + f.bn - 1) / f.bn) * jobs;
    const int nst = (K + f.bk - 1) / f.bk;
    const int entry = mode == CONV_UP ? 8 * f.bk : mode == CONV_DOWN ? 3 * f.bk : 2 * f.bk;   // table bytes per stage
    const int most = RING_TABLE_BYTES / entry;
    const int lo = (nst + most - 1) / most, hi = can_split ? (nst / 4 < 512 ? nst / 4 : 512) : 1;
    if (lo > 1 && (!can_split || lo > hi)) continue;
    // the fewest splits, and the most that fill 1 .. 8 rounds of the CUs
    for (int r = 0; r <= (can_split ? 8 : 0); ++r) {
      int s = r == 0 ? lo : (int)((long long)r * cus / tiles);
      if (s > hi) s = hi;
      if (s < lo || s < 1) s = lo;
      const int per = (nst + s - 1) / s, real = (nst + per - 1) / per;
      const long long all = tiles * real;
      if (all >= 1ll << 28) continue;
      const double rounds = all <= 4 * cus ? (double)((all + cus - 1) / cus) : 0.5 + (double)all / cus;
      const double us = 2.7 + rounds * (used * per * f.stage + f.tile) + (real > 1 ? 2.5 + real * split_us : 0.);
      if (best.cfg < 0 || us < best.us) best = {c, real, per, us};
    }
  }
  return best;
}

template <int MODE>
static void conv_ring_launch(const ConvRingPlan& plan, ConvRingArgs p) {
  const auto& f = g_conv_ring_cfgs[plan.cfg];
  p.gx = (p.rows + f.bm - 1) / f.bm; p.gy = (p.cols + f.bn - 1) / f.bn;
  const long long tiles = (long long)p.periods * p.gx * p.gy * p.gz;
  const dim3 grid((unsigned)(8 * ((tiles + 7) / 8)));
  const int stages = MODE == CONV_OUTP ? plan.split_stages : (p.K + f.bk - 1) / f.bk;
  p.dN = make_fastdiv(p.N); p.dMx = make_fastdiv(p.Mx); p.dk = make_fastdiv(p.k); p.dkk2 = make_fastdiv(p.kk2); p.dH = make_fastdiv(p.H);
  p.dFg = make_fastdiv(p.Fg); p.dgx = make_fastdiv(p.gx); p.dgy = make_fastdiv(p.gy); p.dper = make_fastdiv(p.periods);
  p.dsplits = make_fastdiv(p.splits); p.dG = make_fastdiv(p.G);
  const size_t tab = (size_t)(stages < 1 ? 1 : stages) * f.bk * (MODE == CONV_UP ? 8 : MODE == CONV_DOWN ? 3 : 2);
#define CONV_RING(TB, BM, BN, BK) hipLaunchKernelGGL((k_conv_ring<MODE, TB, BM, BN, BK>), grid, dim3(RING_THREADS), tab, dn_stream(), p)
  switch (plan.cfg) {
    case 0: CONV_RING(32, 64, 64, 32); break;
    case 1: CONV_RING(32, 64, 32, 64); break;
    case 2: CONV_RING(32, 32, 64, 64); break;
    case 3: CONV_RING(16, 32, 32, 64); break;
    case 4: CONV_RING(16, 32, 16, 128); break;
    default: CONV_RING(16, 16, 32, 128); break;
  }
#undef CONV_RING
}
