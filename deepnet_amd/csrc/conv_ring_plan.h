// Which convolution passes run on k_conv_ring, and on which of its tiles (host code without HIP; the tests build it by
// itself).  Args: ConvArgs or anything with its sizes.
#pragma once

// CONV_DOWNM: convDown of few colours, the pixels of a block (of the stride's side, on ring tiles of a multiple of it)
// merged into the columns of one product (uniform-row kernels and ring tiles of one block each).
// CONV_DOWNS: convDown of any stride on ring tiles of one pixel (CONV_DOWN there: of stride 1).
// CONV_DOWNO: convDown of filters that are no whole fours, on ring tiles over any run of pixels.
enum { CONV_UP = 0, CONV_DOWN = 1, CONV_OUTP = 2, CONV_DOWNM = 3, CONV_DOWNS = 4, CONV_DOWNO = 5 };

#define RING_MAX_SIDE 15   // filter rows and columns that a mask has room for
#define RING_AHEAD 7       // stages that the table of a tile of one module or pixel reaches beyond its last one

// Bits lo .. hi - 1 of a mask, hi <= RING_MAX_SIDE.  lo grows with the padding, and with the image beyond the modules' reach
// (host and device).
static constexpr unsigned ring_bits(int lo, int hi) {
  lo = lo < 0 ? 0 : lo > RING_MAX_SIDE ? RING_MAX_SIDE : lo;
  hi = hi < lo ? lo : hi;
  return ((1u << hi) - 1u) & ~((1u << lo) - 1u);
}

// The batch that a pass is copied to when it is no multiple of 16 images (see PaddedBatch).
static inline int padded_batch(int N) {
  if (N <= 16 || N % 16 == 0) return N;
  const int n128 = (N + 127) / 128 * 128;
  return (n128 - N) * 10 <= 3 * N ? n128 : (N + 31) / 32 * 32;
}

// The batch of a locally connected layer, whose uniform-row kernels need a multiple of 128.
static inline int local_batch(int N) { return N >= 32 ? (N + 127) / 128 * 128 : N <= 16 || N % 16 == 0 ? N : 32; }

// The filter count that a bank is copied to (see conv_up_filters).
static inline int padded_filters(int F, int numGroups) {
  return numGroups == 1 && F > 0 && F % 16 != 0 ? (F + 15) / 16 * 16 : F;
}

// The tiles and what they cost: us per stage and per tile of a round (a tile on every CU).  Fitted to 500 measured
// passes (rms 4 to 8 %; masks or none, no difference); what a tile costs besides its stages is its table and its first
// trip to memory.
struct ConvRingTile { int bm, bn, bk; double stage, tile; };
#define CONV_RING_CFGS 6                 // the fp32 tiles
#define CONV_CFGS 11
static constexpr ConvRingTile g_conv_ring_cfgs[CONV_CFGS] = {
    {64, 64, 32, 0.545, 1.45}, {64, 32, 64, 0.574, 1.46}, {32, 64, 64, 0.58, 1.45},
    {32, 32, 64, 0.322, 1.0}, {32, 16, 128, 0.372, 1.2}, {16, 32, 128, 0.372, 1.17},
    // on the bf16 matrix cores (split_tile.h), fitted to 280 passes (of 1161 others they miss by 5 to 8 % rms, tile by tile)
    {128, 128, 32, 1.12, 5.}, {128, 96, 32, 1.08, 4.5}, {128, 64, 32, 0.8, 3.5}, {64, 64, 32, 0.53, 1.}, {128, 48, 64, 1.2, 4.}};
// (of Outp the rows are the filters, and there is no tile of 48)
static constexpr ConvRingTile conv_ring_cfg(int mode, int c) {
  ConvRingTile f = g_conv_ring_cfgs[c];
  if (mode == CONV_OUTP && (c == 7 || c == 8)) { f.bm = f.bn; f.bn = 128; }
  if (c == 10 && (mode == CONV_UP || mode == CONV_OUTP)) f.bm = 0;
  return f;
}
// What a workgroup's LDS holds besides the two stages of its tile, which take 36 to 57 KB in fp32.  Two workgroups share a CU
// while they take half of its 160 KB each; with a full table convUp on 32 x 16 and 16 x 32 tiles takes 82 KB and is alone.  On the
// bf16 matrix cores two stages take 48 (64 x 64) to 132 KB (128 x 48, 158 of the 160 with a full table): up to three workgroups of
// 64 x 64 tiles share a CU while their tables are short, of the others one takes half of its registers or more and is alone.
// The table also bounds the reduction of a convUp, with 8 bytes a term: 3328 terms on tiles over several modules, 3104 to
// 2432 on those of one.  Longer ones (7 x 7 filters on 68 colours or more) stay on the other kernels.
#define RING_TABLE_BYTES 26624
#define RING_CU_LDS (160 << 10)

// LDS of the two stages of a tile in bytes (k_conv_ring checks that it is what its tile loop takes).
static constexpr int conv_ring_lds(int mode, int bm, int bn, int bk) {
  const int a = mode == CONV_OUTP ? bm * (bk + 4) : bk * (bm + 4), b = mode == CONV_UP ? bk * (bn + 4) : bn * (bk + 4);
  return 8 * (a + b);
}

// The same on the bf16 matrix cores: two stages of three planes each, or the sums.
static constexpr int conv_split_lds(int bm, int bn, int bk) {
  return 12 * bk * (bm + bn) > 4 * bm * bn ? 12 * bk * (bm + bn) : 4 * bm * bn;
}
static inline int conv_tile_lds(int mode, int c) {
  const ConvRingTile f = conv_ring_cfg(mode, c);
  return c < CONV_RING_CFGS ? conv_ring_lds(mode, f.bm, f.bn, f.bk) : conv_split_lds(f.bm, f.bn, f.bk);
}

struct ConvRingPlan { int cfg, splits, split_stages; bool single; double us; int blocks; };   // blocks: conv_pixels_plan's

static inline int conv_ring_entry(int mode, bool single, int bk) {      // table bytes per stage
  return mode == CONV_UP ? 8 * bk : mode == CONV_DOWNM || mode == CONV_DOWNO || (mode == CONV_DOWN && !single) ? 3 * bk : 2 * bk;
}
static inline int conv_ring_table(int mode, bool single, int bk, int stages) {      // table bytes of a workgroup
  return ((stages < 1 ? 1 : stages) + (single ? RING_AHEAD : 0)) * conv_ring_entry(mode, single, bk);
}

// Whether a tile may be larger than all of a period (see k_conv_ring).
static constexpr bool conv_may_be_loose(int mode, bool bf16) { return !bf16 || mode == CONV_DOWNM; }

// The tile (of the fp32 ones, or of those on the bf16 matrix cores) that is expected to be fastest, cfg < 0: none fits.
// rows x cols outputs per period, `jobs` periods x groups x chunks, K terms each, of which a tile has the share `used` on
// average; split_us: what adding up one more partial output costs (Outp).  loose: tiles may be larger than all of a period.
static inline ConvRingPlan conv_ring_plan(int mode, bool single, long long rows, int cols, long long jobs, int K, double used,
                                          bool can_split, double split_us, int cus, bool bf16 = false, bool uneven = false, bool loose = false) {
  ConvRingPlan best = {-1, 1, 0, false, 0.};
  for (int c = bf16 ? CONV_RING_CFGS : 0; c < (bf16 ? CONV_CFGS : CONV_RING_CFGS); ++c) {
    const ConvRingTile f = conv_ring_cfg(mode, c);
    if (f.bm == 0 || ((rows < f.bm || cols < f.bn) && !(loose && conv_may_be_loose(mode, c >= CONV_RING_CFGS)))) continue;
    const long long tiles = (rows + f.bm - 1) / f.bm * ((cols + f.bn - 1) / f.bn) * jobs;
    const int nst = (K + f.bk - 1) / f.bk;
    const int most = RING_TABLE_BYTES / conv_ring_entry(mode, single, f.bk) - (single ? RING_AHEAD : 0);
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
      double rounds = all <= 4 * cus ? (double)((all + cus - 1) / cus) : 0.5 + (double)all / cus;
      // alone on its CU a workgroup shows its waits (122 -> 126 colours of 5 x 5 on 16 filters, 24 x 24, batch 100: 66 -> 77 us)
      if (rounds > 1. && c < CONV_RING_CFGS && 2 * (conv_tile_lds(mode, c) + conv_ring_table(mode, single, f.bk, per)) > RING_CU_LDS) rounds *= 1.16;
      double share = used;
      // where there are few rounds, the tiles in the middle of a map, which have all taps, end the last one
      if (c >= CONV_RING_CFGS || uneven) share += (1. - used) / (rounds > 1. ? rounds : 1.);
      if (c >= CONV_RING_CFGS) {
        // Few of the smallest per CU show their waits.  Measured on two cards, against the fp32 tiles: convUp and convDown take
        // 1.10 and 1.08 times as long with one, 1.02 and 0.97 with two, 0.84 and 0.80 with more; Outp, of short reductions,
        // 1.05 and 1.01 with one or two, 0.95 and 0.90 with three or four, 0.88 and 0.83 with more.
        if (f.bm == 64 && f.bn == 64 && all <= (mode == CONV_OUTP ? 2 : 1) * cus) continue;
        rounds *= 1.08;                               // (what the estimates miss: they are to win by that much)
      }
      const double us = 3. + rounds * (share * per * f.stage + f.tile) + (real > 1 ? 2.5 + real * split_us : 0.);
      if (best.cfg < 0 || us < best.us) best = {c, real, per, single, us, 0};
    }
  }
  return best;
}

// Every pass first asks what the fastest ring tile would take (conv_ring_plan) and what the other kernels would
// (conv_other_us), and runs on the ring when that is less.  Both estimates are held against passes over random layers: of
// 3900, those so chosen were 1.4 to 1.5 (any), 2.0 (at most 24 images) and 4 times (two groups; locally connected) as fast on
// average as before the ring, and about one in a hundred more than 5 % slower, by 14 % at most.

// What all three passes need: offsets of 31 bits, masks of RING_MAX_SIDE filter rows.
template <class Args>
static inline bool ring_ok(const Args& a, long long bank_cols) {
  return a.k <= RING_MAX_SIDE && (long long)a.N * a.M * a.F * 4 < (1ll << 31) &&
         (long long)a.N * a.HH * a.C * 4 < (1ll << 31) && (long long)a.F * bank_cols * 4 < (1ll << 31);
}

// What a pass takes, in us, on the other matrix-core kernels: operations on whole blocks at the rate that these reach,
// and the copies of a batch or filter count that they do not take; or on the one-lane-per-output kernels.
// rows: positions of the output per image (Up: modules, Down: pixels); maps16, filters16: 16-byte aligned.
template <class Args>
static inline double conv_other_us(const Args& a, int mode, long long rows, bool maps16, bool filters16, int cus) {
  const int Np = !a.local ? padded_batch(a.N) : mode != CONV_OUTP ? local_batch(a.N) : a.N;
  const int Fp = padded_filters(a.F, a.G), Fg = Fp / a.G, K = a.Cg * a.kk2;
  const bool copy_n = Np != a.N, copy_f = Fp != a.F;
  const bool aligned = (copy_n || maps16) && filters16;
  if (Np % 16 != 0 || Fg % 16 != 0 || !aligned || (a.local && (copy_f || (mode != CONV_OUTP && Np % 128 != 0)))) {
    // one lane per output: 1 TFLOP/s, convUp 3, but a chain of K loads (2 groups of 2 -> 24 colours 3 x 3, 38 x 38, batch 128:
    // 101 us against 134 on ring tiles)
    const double all = 2e-6 * a.N * rows * a.F * K;
    return 5. + (mode == CONV_UP && !a.local ? (all / 3. > 0.25 * K ? all / 3. : 0.25 * K) : all);
  }
  auto up = [](long long v, int b) { return (double)((v + b - 1) / b * b); };
  const double maps = 1e-9 * 8. * Np * ((double)a.M * a.F + (double)a.HH * a.C), hid = 1e-9 * 8. * Np * a.M * Fp;   // GB of a copy
  double flops, rate, copy = 5e-3;                                       // GFLOP, TFLOP/s, GB per us
  if (mode == CONV_UP) {
    flops = 2e-9 * Np * rows * up(Fg, Fg <= 96 ? 32 : 64) * a.G * up(K, 16);
    rate = a.local ? 45. : Np % 128 == 0 && K >= 256 && (Fg <= 64 || Fg > 96) ? 105. : 85.;
    // (few colours: the register-resident bank or 256-row tiles, and maps whose copies mostly stay in the caches)
    if (!a.local && copy_n && K < 256 && Fg <= 64 && a.Cg <= 4) { rate = Fg > 32 && a.pad0 == 0 ? 100. : 90.; copy = 6e-3; }
  } else if (mode == CONV_DOWN && !a.local && a.s == 1 && a.Cg <= 16) {
    // the patch matrix, written by a product and read by a gather
    const double patch = 1e-9 * 8. * Np * a.M * a.Cg * a.kk2 * a.G;       // GB
    return 9. + (2e-9 * Np * a.M * Fp * K / 105. + patch / 5.) * 1e3 + (copy_n ? 5. + maps / copy : 0.) + (copy_f ? 5. + hid / copy : 0.);
  } else if (mode == CONV_DOWN) {
    // (uniform rows: 16-wide blocks for 33 to 48 colours; others: 85 where every CU has two tiles, 97 with reductions of 400
    // terms and more: 96 colours from 48 filters of 3 x 3, 32 x 32, batch 128 128 us on ring tiles, 112 there)
    const bool uniform = a.local || (Np % 128 == 0 && a.kk2 * Fg >= 256 && (a.Cg <= 64 || a.Cg > 96));
    flops = 2e-9 * Np * rows * up(a.Cg, uniform && a.Cg > 32 && a.Cg <= 48 ? 16 : 32) * a.G * a.kk2 * Fg;
    rate = a.local ? 70. : uniform ? 115. : a.Cg > 32 && rows * Np * a.G >= 2ll * 128 * cus ? (a.kk2 * Fg >= 400 ? 97. : 85.) : 65.;
  } else {
    const int BMs = Fg <= 32 ? 32 : Fg <= 64 ? 64 : Fg <= 96 || (Fg > 128 && (Fg + 95) / 96 * 96 < (Fg + 127) / 128 * 128) ? 96 : 128;
    const bool regs = K <= 80 && Fg <= 64;                               // 16 x 16 blocks in registers
    flops = 2e-9 * Np * rows * up(Fg, regs && !a.local && Fg > 32 ? 16 : BMs) * a.G * up(K, regs ? 16 : 128);
    rate = a.local ? 45. : 110.;
  }
  // (a long reduction may be split, and is summed by another launch)
  return (mode == CONV_OUTP || K >= 256 ? 9. : 5.) + flops / rate * 1e3 + (copy_n ? 5. + maps / copy : 0.) + (copy_f ? 5. + hid / copy : 0.);
}

// The share of a layer's taps that lie inside the image (Up) or reach a module (Down), and with it of the reduction that
// tiles of one module or pixel have.
template <class Args>
static inline double ring_used(const Args& a, int mode) {
  const int lines = mode == CONV_UP ? a.Mx : a.H;
  long long taps = 0;                                                    // of a column of modules or pixels
  for (int i = 0; i < lines; ++i) {
    const int v = mode == CONV_UP ? i * a.s + a.pad0 : i - a.pad0;
    const int lo = mode == CONV_UP ? -v : v - a.Mx + 1, hi = mode == CONV_UP ? a.H - v : v + 1;
    const int n = (hi < a.k ? hi : a.k) - (lo > 0 ? lo : 0);
    if (n > 0) taps += n;
  }
  const double one = (double)taps / ((double)lines * a.k);
  return one * one;
}

// How much more of the taps than the average the busiest XCD has: every XCD gets a contiguous eighth of the pixels (one
// group), and the lines in the middle of a map reach more modules than those at its edge.
template <class Args>
static inline double ring_crowd(const Args& a) {
  double all = 0., most = 0.;
  for (int x = 0; x < 8; ++x) {
    double sum = 0.;
    for (int i = x * a.H / 8; i < (x + 1) * a.H / 8 || i == x * a.H / 8; ++i) {
      const int v = i - a.pad0, lo = v - a.Mx + 1 > 0 ? v - a.Mx + 1 : 0, hi = v + 1 < a.k ? v + 1 : a.k;
      sum += hi > lo ? hi - lo : 0;
    }
    const int lines = (x + 1) * a.H / 8 - x * a.H / 8;
    sum /= lines > 0 ? lines : 1;
    all += sum / 8.;
    most = sum > most ? sum : most;
  }
  return all > 0. ? most / all : 1.;
}

static inline ConvRingPlan conv_no_ring() { return {-1, 1, 0, false, 0., 0}; }

// Up and Down: tiles over any run of (module | pixel, image) groups, which needs batches of whole groups of four, or of
// one module or pixel each, which leave out taps beyond the edge and need no masks.  cfg < 0: none fits.
template <class Args>
static inline ConvRingPlan conv_rows_best(const Args& a, int mode, int cus, bool bf16, bool loose = false) {
  const bool up = mode == CONV_UP;
  if (!ring_ok(a, (long long)a.Cg * a.kk2 * (a.local ? a.M : 1)) || (!up && (a.s != 1 || a.Fg % 4 != 0)))
    return conv_no_ring();                                               // (Down: an entry is four filters of a tap)
  const int sites = up ? a.M : a.HH, cols = up ? a.Fg : a.Cg, K = a.kk2 * (up ? a.Cg : a.Fg);
  if (bf16 && K < 9) return conv_no_ring();                              // (a stage of 32 terms is mostly empty)
  ConvRingPlan plan = conv_ring_plan(mode, true, a.N, cols, (long long)sites * a.G, K, ring_used(a, mode), false, 0., cus, bf16, false, loose);
  if (!a.local && a.N % 4 == 0) {
    const ConvRingPlan flat = conv_ring_plan(mode, false, (long long)sites * a.N, cols, a.G, K, 1., false, 0., cus, bf16, false, loose);
    if (flat.cfg >= 0 && (plan.cfg < 0 || flat.us < plan.us)) plan = flat;
  }
  return plan;
}

// How much longer a plan of few colours takes than expected: what it is held against, the patch form, does all pixels at once, so
// there the busiest XCD counts; elsewhere the estimates do not differ by as little.
template <class Args>
static inline double conv_crowd(const Args& a, int mode, const ConvRingPlan& plan) {
  return mode == CONV_DOWN && plan.single && !a.local && a.Cg <= 16 ? ring_crowd(a) : 1.;
}

// The fp32 tile for Up and Down, cfg < 0: another kernel.
template <class Args>
static inline ConvRingPlan conv_rows_plan(const Args& a, int mode, bool maps16, bool filters16, int cus) {
  const ConvRingPlan plan = conv_rows_best(a, mode, cus, false);
  const double other = conv_other_us(a, mode, mode == CONV_UP ? a.M : a.HH, maps16, filters16, cus);
  return plan.cfg < 0 || conv_crowd(a, mode, plan) * plan.us > other ? conv_no_ring() : plan;
}

// The tile for Up and Down, on the bf16 matrix cores where that is expected to be faster.
template <class Args>
static inline ConvRingPlan conv_rows_choice(const Args& a, int mode, bool maps16, bool filters16, int cus) {
  const ConvRingPlan ring = conv_rows_plan(a, mode, maps16, filters16, cus), split = conv_rows_best(a, mode, cus, true);
  const double other = ring.cfg >= 0 ? ring.us : conv_other_us(a, mode, mode == CONV_UP ? a.M : a.HH, maps16, filters16, cus);
  return split.cfg >= 0 && split.us < other ? split : ring;
}

// Strided layers of many colours, whose Down is a product for each of the stride^2 phases of pixels on the other kernels.
template <class Args>
static inline bool conv_phases(const Args& a) { return a.s > 1 && a.Cg > 16; }

// Down of strided layers, of few colours, or of filters that are no multiple of four: on tiles of one pixel (blocks = 0), or
// (DownM) of one block of `blocks` x `blocks` strides of pixels, whose pixels are columns beside the colours: a tile's terms are
// the modules that reach it, of which a pixel of a block has a tap with some only.  blocks < 0: on tiles over any run of (pixel,
// image) groups, of stride 1.  The last entry of a tap may repeat filters where entries have masks (RING_LAST): not of one pixel.
template <class Args>
static inline ConvRingPlan conv_pixels_plan(const Args& a, int blocks, int cus, bool bf16) {
  const int b = blocks > 0 ? blocks : 1, side = blocks > 0 ? b * a.s : 1, taps = b - 1 + (a.k + a.s - 1) / a.s, Fg4 = (a.Fg + 3) / 4 * 4;
  const long long cols = (long long)a.Cg * side * side;
  if (a.local || !ring_ok(a, (long long)a.Cg * a.kk2) || a.Fg < 4 || taps > RING_MAX_SIDE) return conv_no_ring();
  if (blocks < 0) {
    if (a.s != 1 || a.N % 4 != 0) return conv_no_ring();
    ConvRingPlan plan = conv_ring_plan(CONV_DOWN, false, (long long)a.HH * a.N, a.Cg, a.G, a.kk2 * Fg4, 1., false, 0., cus, bf16, false, true);
    plan.blocks = blocks;
    return plan;
  }
  if ((blocks == 0 && a.Fg != Fg4) || cols > 2048) return conv_no_ring();
  const int lines = blocks > 0 ? (a.H - a.pad0 - 1) / side + 1 : a.H;
  long long have = 0;                                                    // modules of a line that the taps of its pixels reach
  for (int i = 0; i < lines; ++i) {
    const int v = blocks > 0 ? i * b : (i - a.pad0) / a.s;               // the last module but b - 1 that reaches the first pixel
    const int top = v + b - 1 < a.Mx - 1 ? v + b - 1 : a.Mx - 1, low = v + b - taps > 0 ? v + b - taps : 0;
    if (top >= low) have += top - low + 1;
  }
  const double one = (double)have / ((double)lines * taps);
  ConvRingPlan plan = conv_ring_plan(blocks > 0 ? CONV_DOWNM : CONV_DOWN, true, a.N, (int)cols, (long long)lines * lines * a.G, taps * taps * Fg4,
                                     one * one, false, 0., cus, bf16, true, true);
  if (blocks > 0 && conv_phases(a)) plan.us = 3. + 1.2 * (plan.us - 3.);
  plan.blocks = blocks;
  return plan;
}

// What Down takes on the other kernels, in us (of layers on these tiles).
template <class Args>
static inline double conv_pixels_other_us(const Args& a, bool maps16, bool filters16, int cus) {
  const double any = conv_other_us(a, CONV_DOWN, a.HH, maps16, filters16, cus);
  if (a.s == 1)      // (k_conv_down_px: pixels in registers)
    return a.Cg <= 4 && (a.k == 3 || a.k == 5) && a.Fg % 8 == 0 && a.Fg <= 128 ? 0.7 * any : any;
  const int Np = padded_batch(a.N), Fp = padded_filters(a.F, a.G), Fg = Fp / a.G;
  if (Np % 16 != 0 || Fg % 16 != 0 || !((Np != a.N || maps16) && filters16)) return any;      // (one lane per output)
  const double maps = 1e-9 * 8. * Np * ((double)a.M * a.F + (double)a.HH * a.C), hid = 1e-9 * 8. * Np * a.M * Fp;   // GB of a copy
  const double copies = (Np != a.N ? 5. + maps / 5e-3 : 0.) + (Fp != a.F ? 5. + hid / 5e-3 : 0.);
  if (conv_phases(a)) {   // a pixel has every s-th tap of a row and column
    // (uniform rows: as in conv_other_us; fewer tiles than CUs: as long as one tile takes, 24 ns a term and 32 columns)
    const bool uniform = Np % 128 == 0 && a.kk2 * Fg >= 256 * a.s * a.s && (a.Cg <= 64 || a.Cg > 96);
    const int wide = uniform && a.Cg > 32 && a.Cg <= 48 ? 16 : 32, taps = (a.k + a.s - 1) / a.s;
    const double flops = 2e-9 * Np * a.HH * ((a.Cg + wide - 1) / wide * wide) * a.G * a.kk2 * Fg / (a.s * a.s);
    const double all = 6. + flops / (uniform ? 95. : 80.) * 1e3, one = 5. + 0.024 * taps * taps * Fg * (a.Cg > 64 ? 3 : a.Cg > 32 ? 2 : 1);
    return (all > one ? all : one) + copies;
  }
  if (Np % 128 == 0) {   // pixels of a block as columns
    const int taps = (a.k + a.s - 1) / a.s, cols = a.Cg * a.s * a.s;
    const double lines = (a.H - 1 - a.pad0) / a.s + 1;
    return 9. + 2e-9 * Np * lines * lines * ((cols + 15) / 16 * 16) * a.G * taps * taps * Fg / (cols <= 16 ? 75. : 110.) * 1e3 + copies;
  }
  // the patch matrix, written by a product and read by a gather
  const double patch = 1e-9 * 8. * Np * a.M * a.Cg * a.kk2 * a.G;
  return 9. + (2e-9 * Np * a.M * Fp * a.Cg * a.kk2 / 105. + patch / 5.) * 1e3 + copies;
}

// The fastest of these tiles, on the bf16 matrix cores or not; cfg < 0: none fits, or another kernel is expected to be faster.
// (0.87: of layers whose estimates are as near as that, measured, half lose, by 20 % at most: 3 -> 208 colours of 7 x 7, stride 4, 200 x
// 200, batch 80, 190 -> 237 us; 1 -> 48 of 7 x 7, 26 x 26, 80, 14.6 -> 18.1.  Of 410 random layers of few colours that are taken six are
// slower, by 22 % at most.  0.96 of strided layers of many colours, whose estimates are nearer: of 500 that coarser ones gave to these
// tiles 48 were more than 4 % slower, by up to 38 %, and now 13, by up to 17 %; 21 that the others keep would gain 4 to 48 %.)
template <class Args>
static inline ConvRingPlan conv_pixels_choice(const Args& a, bool maps16, bool filters16, int cus) {
  ConvRingPlan best = conv_no_ring();
  if (a.s == 1 && a.Cg > 16 && a.Fg % 4 == 0) return best;
  for (int blocks = -1; blocks <= 4; blocks = blocks > 0 ? 2 * blocks : blocks + 1)
    for (int bf16 = 0; bf16 < 2; ++bf16) {
      const ConvRingPlan plan = conv_pixels_plan(a, blocks, cus, bf16 != 0);
      if (plan.cfg >= 0 && (best.cfg < 0 || plan.us < best.us)) best = plan;
    }
  return best.cfg >= 0 && best.us < (conv_phases(a) ? 0.96 : 0.87) * conv_pixels_other_us(a, maps16, filters16, cus) ? best : conv_no_ring();
}

// Outp of `a`, whose batch the ring takes in whole groups of four images: others are copied with up to three images of zeros.
template <class Args>
static inline ConvRingPlan conv_outp_best(const Args& a, int cus, bool bf16, bool loose = false) {
  Args r = a;
  r.N = (a.N + 3) / 4 * 4;
  const int cols = a.Cg * a.kk2;
  if (!ring_ok(r, (long long)cols * a.chunks) || a.chunks > 32767) return conv_no_ring();
  ConvRingPlan plan = conv_ring_plan(CONV_OUTP, false, a.Fg, cols, (long long)a.G * a.chunks, a.m_count * r.N, 1., true,
                                     2e-6 * a.chunks * a.F * cols, cus, bf16, false, loose);
  const double maps = 1e-9 * 8. * r.N * ((double)a.M * a.F + (double)a.HH * a.C);
  // (1.12: what a layer's sums over many splits take beyond the plan's estimate)
  plan.us = 1.12 * plan.us + (r.N != a.N ? 5. + maps / 5e-3 : 0.);
  return plan;
}
template <class Args>
static inline ConvRingPlan conv_outp_plan(const Args& a, bool maps16, bool filters16, int cus) {
  const ConvRingPlan plan = conv_outp_best(a, cus, false);
  return plan.cfg < 0 || plan.us > conv_other_us(a, CONV_OUTP, a.M, maps16, filters16, cus) ? conv_no_ring() : plan;
}
template <class Args>
static inline ConvRingPlan conv_outp_choice(const Args& a, bool maps16, bool filters16, int cus) {
  const ConvRingPlan ring = conv_outp_plan(a, maps16, filters16, cus), split = conv_outp_best(a, cus, true);
  const double other = ring.cfg >= 0 ? ring.us : conv_other_us(a, CONV_OUTP, a.M, maps16, filters16, cus);
  return split.cfg >= 0 && split.us < other ? split : ring;
}

// What a pass runs on, where its tile may be larger than all the filters, colours or taps there are (conv_ring_plan: loose): the choice
// of the tiles that are not, unless such a one is expected to be faster.
template <class Args>
static inline ConvRingPlan conv_loose_choice(const Args& a, int mode, bool maps16, bool filters16, int cus) {
  const ConvRingPlan tight = mode == CONV_OUTP ? conv_outp_choice(a, maps16, filters16, cus) : conv_rows_choice(a, mode, maps16, filters16, cus);
  const double other = tight.cfg >= 0 ? tight.us : conv_other_us(a, mode, mode == CONV_DOWN ? a.HH : a.M, maps16, filters16, cus);
  ConvRingPlan best = tight;
  double us = 0.87 * other;
  for (int bf16 = 0; bf16 < 2; ++bf16) {
    const ConvRingPlan plan = mode == CONV_OUTP ? conv_outp_best(a, cus, bf16 != 0, true) : conv_rows_best(a, mode, cus, bf16 != 0, true);
    if (plan.cfg < 0 || plan.us >= us) continue;
    // (the busiest XCD of few colours, on all but the 6 us that a short pass takes anyway.  Of 230 such layers 26 were up to 66 % slower
    // without it: 13 -> 244 colours 7 x 7, 15 x 15, batch 173 86 us on the patch form, 142 on ring tiles; with it 2, by up to 19 %.)
    if (6. + conv_crowd(a, mode, plan) * (plan.us - 6.) >= other) continue;
    best = plan;
    us = plan.us;
  }
  return best;
}

// What a pass runs on: `pixels` says that `plan` is conv_pixels_plan's.  cfg < 0: another kernel.
struct ConvChoice { ConvRingPlan plan; bool pixels; };
template <class Args>
static inline ConvChoice conv_choice(const Args& a, int mode, bool maps16, bool filters16, int cus) {
  const ConvRingPlan rows = conv_loose_choice(a, mode, maps16, filters16, cus);
  if (mode == CONV_DOWN) {
    const ConvRingPlan pixels = conv_pixels_choice(a, maps16, filters16, cus);
    if (pixels.cfg >= 0 && (rows.cfg < 0 || pixels.us < rows.us)) return {pixels, true};
  }
  return {rows, false};
}

// All that conv_choice depends on.
struct ConvKey { int v[15]; };
template <class Args>
static inline ConvKey conv_key(const Args& a, int mode, bool maps16, bool filters16, int cus) {
  return {{mode, a.N, a.C, a.H, a.F, a.k, a.Mx, a.s, a.pad0, a.G, a.local, a.m_count, a.chunks, (maps16 ? 2 : 0) + (filters16 ? 1 : 0), cus}};
}
