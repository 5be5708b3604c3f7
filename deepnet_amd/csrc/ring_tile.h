// The tile loop of the mid-sized products (gemm_ring.h) and of the convolutions (conv_ring.h).
#pragma once
#include <type_traits>

#define RING_THREADS 512
#define RING_SETS 4        // register sets: the stages on their way from global memory

typedef float ring_f32x16 __attribute__((ext_vector_type(16)));
typedef float ring_f32x4 __attribute__((ext_vector_type(4)));

// The lane's number.  OPAQUE: in a kernel that holds several tile loops, so that what each makes of it is not kept in registers
// for all of them from the start (the eight loops of k_gemm_group<3, 4>: 109 -> 107 registers, of <1, 2> 128 -> 125).
template <bool OPAQUE>
__device__ __forceinline__ int ring_tid() {
  unsigned t = threadIdx.x;
  if (OPAQUE) {
    asm volatile("" : "+v"(t));
    __builtin_assume(t < RING_THREADS);
  }
  return (int)t;
}

// One operand of a stage in LDS: [row][BK + 4] when it is K-contiguous in memory (KC), [k][rows + 4] otherwise, both free
// of bank conflicts for the order of terms that `frag` reads (pitch 4 mod 8).  A stage is NG 16-byte groups per lane.
template <int ROWS, int BK_, bool KC_>
struct RingTile {
  static constexpr int BK = BK_;
  static constexpr bool KC = KC_;
  static constexpr int KPACK = KC ? 4 : 1;                 // consecutive terms of a lane's groups
  static constexpr int REACH = 1;                          // stages that the lanes' first terms lie in
  static constexpr int NG = ROWS * BK / 4 / RING_THREADS;
  static_assert(NG * RING_THREADS * 4 == ROWS * BK, "whole groups per lane");
  static constexpr int PITCH = KC ? BK + 4 : ROWS + 4;
  static constexpr int FLOATS = KC ? ROWS * PITCH : BK * PITCH;
  // group u of lane `tid`: its (first) term of the stage and its (first) row
  __device__ __forceinline__ static int group_k(int tid, int u) {
    const int f = tid + u * RING_THREADS;
    return KC ? 4 * (f % (BK / 4)) : f / (ROWS / 4);
  }
  __device__ __forceinline__ static int group_row(int tid, int u) {
    const int f = tid + u * RING_THREADS;
    return KC ? f / (BK / 4) : 4 * (f % (ROWS / 4));
  }
  __device__ __forceinline__ static void stash(float* S, int tid, const ring_f32x4 (&r)[NG]) {
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      float* d = KC ? S + group_row(tid, u) * PITCH + group_k(tid, u) : S + group_k(tid, u) * PITCH + group_row(tid, u);
      *reinterpret_cast<ring_f32x4*>(d) = r[u];
    }
  }
  // v[4 u + j] = operand(row, k0 + u * KU + j), u < 2, j < 4
  template <int KU>
  __device__ __forceinline__ static void frag(const float* S, int row, int k0, float (&v)[8]) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (KC) {
        const ring_f32x4 x = *reinterpret_cast<const ring_f32x4*>(S + row * PITCH + k0 + KU * u);
        v[4 * u] = x.x; v[4 * u + 1] = x.y; v[4 * u + 2] = x.z; v[4 * u + 3] = x.w;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[4 * u + j] = S[(k0 + KU * u + j) * PITCH + row];
      }
    }
  }
};

__device__ __forceinline__ ring_f32x16 ring_mfma(float b, float a, ring_f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(b, a, c, 0, 0, 0); }
__device__ __forceinline__ ring_f32x4 ring_mfma(float b, float a, ring_f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(b, a, c, 0, 0, 0); }

// 8 wavefronts on a BM x BN tile: WM x WN blocks of TB x TB outputs, the wavefronts that are left over split a stage's
// terms KS ways.  OA / OB: RingTile plus fetch(t, nst, registers), called for t = 0, 1, 2 ... in order.
template <int TB, int BM, int BN, int BK, typename OA, typename OB>
struct RingShape {
  static constexpr int WM = BM / TB, WN = BN / TB, KS = 8 / (WM * WN), KW = BK / KS;
  static_assert(KW == 512 / TB, "eight MFMAs per wavefront and stage");
  using acc_t = std::conditional_t<TB == 32, ring_f32x16, ring_f32x4>;
  static constexpr int NACC = TB * TB / 64, KU = TB == 32 ? 4 : 16;
  static constexpr int STAGE = OA::FLOATS + OB::FLOATS, RED = KS * BM * BN;
  static constexpr int LDS = 2 * STAGE > RED ? 2 * STAGE : RED;
  static constexpr int EPL = BM * BN / RING_THREADS;       // outputs per lane: (tid % BM, tid / BM + u * RING_THREADS / BM)

  // The tile's sums over nst >= 1 stages, lane by lane in sum[EPL].  kskip terms of the last stage are left out.
  // early(): called while the first loads are on their way.
  template <bool SKIP, bool OPAQUE, typename F>
  __device__ __forceinline__ static void run(float* lds, OA& oa, OB& ob, int nst, int kskip, float (&sum)[EPL], F early) {
    const int tid = ring_tid<OPAQUE>(), lane = tid & 63, li = lane % TB, lk = lane / TB;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wv % WM, wn = (wv / WM) % WN, ks = wv / (WM * WN);
    ring_f32x4 ra[RING_SETS][OA::NG], rb[RING_SETS][OB::NG];
#define RING_FETCH(SET, T) do { oa.fetch(T, nst, ra[SET]); ob.fetch(T, nst, rb[SET]); } while (0)
#define RING_STASH(BUF, SET) do { OA::stash(lds + (BUF) * STAGE, tid, ra[SET]); OB::stash(lds + (BUF) * STAGE + OA::FLOATS, tid, rb[SET]); } while (0)
    const int arow = wm * TB + li, brow = wn * TB + li, fk = ks * KW + (TB == 32 ? 8 : 4) * lk;
#define RING_FRAG(BUF, AV, BV) do { OA::template frag<KU>(lds + (BUF) * STAGE, arow, fk, AV); OB::template frag<KU>(lds + (BUF) * STAGE + OA::FLOATS, brow, fk, BV); } while (0)
    // stage s sits in register set (s + 2) % 4 until it is written to LDS[s & 1]
    RING_FETCH(2, 0); RING_FETCH(3, 1); RING_FETCH(0, 2); RING_FETCH(1, 3);
    early();
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
    // the last one to four stages
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (s + q < nst) {
        const int kmin = SKIP && s + q == nst - 1 ? kskip : 0;
        if (s + q + 1 < nst) RING_FRAG((q + 1) & 1, fa[(q + 1) & 1], fb[(q + 1) & 1]);
        if (s + q + 2 < nst) RING_STASH(q & 1, q);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const bool in = !SKIP || fk + KU * (j >> 2) + (j & 3) >= kmin;
          acc = ring_mfma(in ? fb[q & 1][j] : 0.f, in ? fa[q & 1][j] : 0.f, acc);
        }
        __syncthreads();
      }
    }
#undef RING_FETCH
#undef RING_STASH
#undef RING_FRAG
    // acc[v] is the tile's (m, n) = (32 wm + li, 32 wn + 8 (v / 4) + 4 lk + v % 4); partial tiles are [n][m]
    float* part = lds + ks * (BM * BN);
#pragma unroll
    for (int v = 0; v < NACC; ++v) part[(wn * TB + 8 * (v >> 2) + 4 * lk + (v & 3)) * BM + wm * TB + li] = acc[v];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < EPL; ++u) {
      const int e = tid + RING_THREADS * u;
      sum[u] = lds[e];
#pragma unroll
      for (int w = 1; w < KS; ++w) sum[u] += lds[w * (BM * BN) + e];
    }
  }
};
