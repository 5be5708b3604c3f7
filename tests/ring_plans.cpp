// The host's choice of ring tiles for the tests, as the libraries make it (tests/test_ring_plans.py builds and loads this).
#include "../deepnet_amd/csrc/gemm_ring_plan.h"
#include "../deepnet_amd/csrc/conv_ring_plan.h"

// (a shift by 32 or more does not compile here)
static_assert(ring_bits(2, 5) == 0x1c && ring_bits(-3, 4) == 0xf && ring_bits(0, RING_MAX_SIDE) == 0x7fff && ring_bits(4, 4) == 0, "");
static_assert(ring_bits(5, 3) == 0 && ring_bits(14, -2) == 0 && ring_bits(33, 7) == 0 && ring_bits(400, 15) == 0, "");

struct Sizes { int N, C, Cg, H, HH, F, Fg, k, kk2, Mx, M, s, pad0, G, local, m_count, chunks; };

extern "C" {

// Tile number (the order of g_ring_cfgs) of an M x N x K product of whole matrices; -1: not on k_gemm_ring.  vec: as there.
int gemm_tile(int M, int N, int K, int cus, int vec) {
  return K > 128 ? gemm_ring_plan(M, N, K, (size_t)M * K * 4, (size_t)N * K * 4, cus, vec != 0).cfg : -1;
}

// Whether the product is k_gemm_split's (of a target that is not read).
int gemm_split(int M, int N, int K, int cus, int vec) {
  const size_t a = (size_t)M * K * 4, b = (size_t)N * K * 4;
  return gemm_split_wins(M, N, K, false, a, b, K > 128 ? gemm_ring_plan(M, N, K, a, b, cus, vec != 0) : RingPlan{-1, 0.}, cus);
}

// The side of k_gemm's tiles, 128 or 64, for a product of more than 128 terms; 0: another kernel's.
int gemm_slab(int M, int N, int K, int cus, int vec) {
  const long long tiles32 = (long long)((M + 31) / 32) * ((N + 31) / 32);
  if (gemm_tile(M, N, K, cus, vec) >= 0 || gemm_split(M, N, K, cus, vec) || tiles32 <= 2ll * cus) return 0;
  return gemm_slab_big(M, N, K, false, cus) ? 128 : 64;
}

// The fp32 tile of a pass, or with mode + 4 the tile of all: out = {tile number or -1, one module or pixel per tile, splits, LDS bytes of a workgroup, us}
void conv_tile(int mode, int N, int C, int H, int F, int k, int Mx, int s, int pad0, int G, int local, int partial_sum, int cus, double* out) {
  const int m = partial_sum ? partial_sum : Mx * Mx;
  const Sizes a = {N, C, C / G, H, H * H, F, F / G, k, k * k, Mx, Mx * Mx, s, pad0, G, local, m, Mx * Mx / m};
  const bool all = mode >= 4;          // 4 + mode: of all tiles
  mode &= 3;
  const bool maps16 = N % 4 == 0;
  const ConvRingPlan p = mode == CONV_OUTP ? (all ? conv_outp_choice(a, maps16, true, cus) : conv_outp_plan(a, maps16, true, cus))
                                           : (all ? conv_rows_choice(a, mode, maps16, true, cus) : conv_rows_plan(a, mode, maps16, true, cus));
  out[0] = p.cfg; out[1] = p.single; out[2] = p.splits;
  const int K = mode == CONV_OUTP ? 0 : a.kk2 * (mode == CONV_UP ? a.Cg : a.Fg);
  if (p.cfg < 0) return;
  const ConvRingTile f = conv_ring_cfg(mode, p.cfg);
  out[3] = conv_tile_lds(mode, p.cfg) + conv_ring_table(mode, p.single, f.bk, mode == CONV_OUTP ? p.split_stages : (K + f.bk - 1) / f.bk);
  out[4] = p.us;
}

// Whether a pass runs on a tile that is larger than all its rows or columns (of one module or pixel, where the tile lies in one).
int conv_tile_is_loose(int mode, int N, int C, int H, int F, int k, int Mx, int s, int pad0, int G, int cus) {
  const Sizes a = {N, C, C / G, H, H * H, F, F / G, k, k * k, Mx, Mx * Mx, s, pad0, G, 0, Mx * Mx, 1};
  const ConvChoice c = conv_choice(a, mode, N % 4 == 0, true, cus);
  if (c.plan.cfg < 0 || c.pixels) return 0;
  const ConvRingTile f = conv_ring_cfg(mode, c.plan.cfg);
  const int cols = mode == CONV_UP ? a.Fg : mode == CONV_DOWN ? a.Cg : a.Cg * a.kk2;
  return (mode == CONV_OUTP ? a.Fg : c.plan.single ? N : 1 << 30) < f.bm || cols < f.bn;
}

// What a pass runs on: out = {tile number or -1, one module or pixel per tile, from conv_pixels_plan, us, us on the other kernels, how much
// longer the busiest XCD takes}
void conv_route(int mode, int N, int C, int H, int F, int k, int Mx, int s, int pad0, int G, int cus, double* out) {
  const Sizes a = {N, C, C / G, H, H * H, F, F / G, k, k * k, Mx, Mx * Mx, s, pad0, G, 0, Mx * Mx, 1};
  const ConvChoice c = conv_choice(a, mode, N % 4 == 0, true, cus);
  out[0] = c.plan.cfg; out[1] = c.plan.single; out[2] = c.pixels; out[3] = c.plan.us;
  out[4] = conv_other_us(a, mode, mode == CONV_DOWN ? a.HH : a.M, N % 4 == 0, true, cus); out[5] = ring_crowd(a);
}

// What a layer's choice is kept by; in: mode, the sizes from N to chunks but for those that follow from others, both alignments, CUs.
int conv_key_of(const int* in, int* out) {
  const Sizes a = {in[1], in[2], in[2] / in[9], in[3], in[3] * in[3], in[4], in[4] / in[9], in[5], in[5] * in[5], in[6], in[6] * in[6], in[7], in[8],
                   in[9], in[10], in[11], in[12]};
  const ConvKey key = conv_key(a, in[0], in[13] != 0, in[14] != 0, in[15]);
  for (int v : key.v) *out++ = v;
  return sizeof key / sizeof(int);
}

// convDown of strided layers, few colours or filters that are no whole fours: out = {tile number or -1, side of a block in strides, 0 a
// pixel or -1 any run, stages of the table, LDS bytes of a workgroup}
void conv_pixels_tile(int N, int C, int H, int F, int k, int Mx, int s, int pad0, int G, int cus, double* out) {
  const Sizes a = {N, C, C / G, H, H * H, F, F / G, k, k * k, Mx, Mx * Mx, s, pad0, G, 0, Mx * Mx, 1};
  const ConvRingPlan p = conv_pixels_choice(a, N % 4 == 0, true, cus);
  out[0] = p.cfg; out[1] = p.blocks;
  if (p.cfg < 0) return;
  const int mode = p.blocks > 0 ? CONV_DOWNM : CONV_DOWN, b = p.blocks > 0 ? p.blocks : 1, taps = b - 1 + (k + s - 1) / s;
  const ConvRingTile f = conv_ring_cfg(mode, p.cfg);
  const int terms = (p.blocks < 0 ? k * k : taps * taps) * ((a.Fg + 3) / 4 * 4), stages = (terms + f.bk - 1) / f.bk;
  out[2] = stages;
  out[3] = conv_tile_lds(mode, p.cfg) + conv_ring_table(mode, p.blocks >= 0, f.bk, stages);
}

}  // extern "C"
