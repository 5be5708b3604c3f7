// fp32 products on the bf16 matrix cores: the tile loop of the larger products (gemm_split.h) and convolutions (conv_ring.h).
#pragma once
#include "ring_tile.h"

// Every operand is taken apart into three bf16 numbers h + m + l, each the nearest one to what is left: 8 + 8 + 8 bits of
// mantissa, so the sum is the fp32 number itself.  A product a b is the six products hh, hm, mh, mm, hl, lh; ml, lm and ll are
// left out, 2^-24 of it at most.  hh has an accumulator of its own and the others, 2^-8 of it and less, share another, which
// are added at the end.  Six v_mfma_f32_16x16x32_bf16 take 96 cycles where eight v_mfma_f32_16x16x4_f32 take 256.
// Against sums in 64 bits the results are nearer than those of the fp32 instructions, which round an accumulator for
// every second term: the error is 0.3 to 0.4 times theirs for dense operands of 64 to 8192 terms, of both signs, of one
// sign or rectified, 0.05 to 0.4 for samples of zeros and ones; from 0.65 to 1.0 at 64 terms of which few are not zero.  It is
// larger where only one term of a sum is not zero and neither factor is short (0, 1, or 16 bits against 8, which are
// exact): there they round once, by half an ulp at most and 0.2885 rms, and what is left out here makes it 0.954 and 0.297.  From
// two terms on the rms error is the smaller one (ulp here / there: two terms 0.297 / 0.369, three 0.298 / 0.414, 705 2.01 / 3.12), the
// largest up to four or so is not (two 1.7 / 1.25).  With ml and lm too, eight products, one term is as there (0.51, 0.2885)
// and dense sums are no nearer, for 1.17 times the time (three products of a 4096 x 4096 layer 2081 -> 2432 us, convolutions of 96
// -> 256 colours 1002 -> 1146): not done.
// Numbers are scaled by 2^24 on the way in and results by 2^-48 on the way out: what is left of an fp32 number of any size,
// denormals too, is then an ordinary bf16 number.  A tile whose sums are not all finite (an operand that is infinite,
// not a number or beyond 2^104, a result beyond 2^80) is computed again on the fp32 instructions, and takes 2.4 times as long as
// on those alone (4096 x 4096 x 4096 with NaN in every tile 951 -> 2250 us, in one row 1057 -> 1080).  Loads ahead and unrolled
// products there gave 5 to 7 % of it back and cost ordinary tiles 1 % (registers).
#define SPLIT_IN 0x1p24f
#define SPLIT_OUT 0x1p-48f

typedef __bf16 split_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 split_bf16x2 __attribute__((ext_vector_type(2)));
typedef unsigned split_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned split_u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ unsigned split_round2(float x, float y) {
  const split_bf16x2 r = {(__bf16)x, (__bf16)y};
  return __builtin_bit_cast(unsigned, r);
}
__device__ __forceinline__ void split_pair(float x, float y, unsigned (&p)[3]) {
  x *= SPLIT_IN; y *= SPLIT_IN;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    p[q] = split_round2(x, y);
    x -= __builtin_bit_cast(float, p[q] << 16);
    y -= __builtin_bit_cast(float, p[q] & 0xffff0000u);
  }
  p[2] = split_round2(x, y);
}

// One operand of a stage: three planes of [k / 8][slot] groups of eight terms, 16 bytes each.  A lane takes NG 16-byte groups
// from global memory: of a K-contiguous operand (KC) four terms of NG rows, else NG consecutive terms of four rows, of
// which it packs NG terms a row.  There a slot is not its row: the rows 4 q + j of a block of 4 Q rows sit in slots Q j + q, and
// eight lanes with consecutive q fill 128 bytes together with those that have the other terms.  Slots are exchanged
// within their sixteen (swap) against bank conflicts: a read takes sixteen slots of two k / 8 at once, a store of 128 bytes
// has all k / 8 of a row of a KC operand.  Neither has conflicts.
template <int ROWS_, int BK_, bool KC_, int NT_>
struct SplitTile {
  static constexpr int ROWS = ROWS_, BK = BK_, NT = NT_;
  static constexpr bool KC = KC_;
  static constexpr int GROUPS = ROWS * BK / 4, NGS = (GROUPS + NT - 1) / NT, NG = KC || NGS > 1 ? NGS : 2, PACKS = KC ? 2 : 8 / NG;
  static constexpr int KPACK = KC ? 4 : NG;                // consecutive terms of a lane's groups
  static_assert(GROUPS % 64 == 0 && ROWS % 16 == 0 && BK % 32 == 0 && NT % (BK / 4) == 0, "whole wavefronts and blocks");
  static_assert(KC || ((NG == 2 || NG == 4) && ROWS % 32 == 0 && GROUPS / NG % 64 == 0), "whole packs of terms");
  // stages that the lanes' first terms lie in: lanes that are left over have theirs behind the stage, and store nothing
  static constexpr int REACH = KC ? 1 : 8 * ((NT - 1) / (8 * PACKS * (ROWS / 32))) / BK + 1;
  static constexpr int Q = ROWS % 64 == 0 ? 16 : 8;
  static constexpr int PLANE = BK * ROWS * 2, BYTES = 3 * PLANE;
  // group u of lane `tid`: its (first) term of the stage and its (first) row (beyond the stage for lanes that are left over)
  __device__ __forceinline__ static int group_k(int tid, int u) {
    return KC ? 4 * (tid % (BK / 4)) : 8 * (tid / (8 * PACKS * (ROWS / 32))) + NG * (tid / 8 % PACKS) + u;
  }
  __device__ __forceinline__ static int group_row(int tid, int u) {
    return KC ? (tid + u * NT) / (BK / 4) : 32 * (tid / (8 * PACKS) % (ROWS / 32)) + 4 * (tid % 8);
  }
  __device__ __forceinline__ static int slot_of(int row) {
    return KC ? row : row / (4 * Q) * (4 * Q) + Q * (row % 4) + row % (4 * Q) / 4;
  }
  __device__ __forceinline__ static int row_of(int slot) {
    return KC ? slot : slot / (4 * Q) * (4 * Q) + 4 * (slot % Q) + slot % (4 * Q) / Q;
  }
  __device__ __forceinline__ static int swap(int kg) { return BK == 32 ? 2 * kg : kg & 7; }
  // (terms below kmin of a last stage were taken by the one before)
  template <bool SKIP>
  __device__ __forceinline__ static void stash(char* S, int tid, ring_f32x4 (&r)[NG], int kmin) {
    const int k = group_k(tid, 0), kg = k / 8;
    if (SKIP) {
#pragma unroll
      for (int u = 0; u < NG; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) r[u][j] = k + (KC ? j : u) >= kmin ? r[u][j] : 0.f;
    }
    char* D = S + kg * (ROWS * 16) + k % 8 * 2;
    if (KC) {
#pragma unroll
      for (int u = 0; u < NG; ++u) {
        unsigned a[3], b[3];
        split_pair(r[u][0], r[u][1], a);
        split_pair(r[u][2], r[u][3], b);
        if (GROUPS == NG * NT || tid + u * NT < GROUPS) {
#pragma unroll
          for (int p = 0; p < 3; ++p)
            *reinterpret_cast<split_u32x2*>(D + p * PLANE + (group_row(tid, u) ^ swap(kg)) * 16) = split_u32x2{a[p], b[p]};
        }
      }
    } else if (GROUPS == NG * NT || tid < GROUPS / NG) {
      const int slot = slot_of(group_row(tid, 0)) ^ swap(kg);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        unsigned a[3], b[3];
        split_pair(r[0][j], r[1][j], a);
        if (NG == 4) split_pair(r[NG - 2][j], r[NG - 1][j], b);
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          char* d = D + p * PLANE + (slot + Q * j) * 16;
          if (NG == 4) *reinterpret_cast<split_u32x2*>(d) = split_u32x2{a[p], b[p]};
          else *reinterpret_cast<unsigned*>(d) = a[p];
        }
      }
    }
  }
  // plane p, terms 32 c + 8 lk .. + 7 of a slot
  __device__ __forceinline__ static split_bf16x8 frag(const char* S, int p, int c, int lk, int slot) {
    const int kg = 4 * c + lk;
    return __builtin_bit_cast(split_bf16x8, *reinterpret_cast<const split_u32x4*>(S + p * PLANE + kg * (ROWS * 16) + (slot ^ swap(kg)) * 16));
  }
  // the stage as it is, [k][ROWS]
  __device__ __forceinline__ static void stash32(float* S, int tid, const ring_f32x4 (&r)[NG], int kmin) {
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      if (GROUPS == NG * NT || (KC ? tid + u * NT < GROUPS : tid < GROUPS / NG)) {
        const int k = group_k(tid, u), row = group_row(tid, u);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          S[(KC ? k + j : k) * ROWS + (KC ? row : row + j)] = k + (KC ? j : 0) >= kmin ? r[u][j] : 0.f;
      }
    }
  }
};

__device__ __forceinline__ ring_f32x4 split_mfma(split_bf16x8 b, split_bf16x8 a, ring_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, c, 0, 0, 0);
}

// NT / 64 wavefronts on a BM x BN tile, WM x WN of them next to each other, each with (BM / WM) x (BN / WN) outputs in
// blocks of 16 x 16; KS of them share a block's outputs and split a stage's terms in chunks of 32.
// OA / OB: SplitTile plus fetch(t, nst, registers), called for t = 0, 1, 2 ... in order, and perhaps again from 0.
// A trip of the loop is one barrier: LDS holds the stage that is multiplied and the next one, registers (SETS sets) those on
// their way from global memory.  The products run plane by plane, so that every read of LDS has the products of another
// plane to hide behind, those of the first plane after the barrier what the stage before has left; taking the next stage
// apart is spread over all of them, three vector instructions behind every MFMA (two or four: 3 to 6 % slower), a store
// behind every third (at the end, behind the last MFMA: 5 %).
template <int BM, int BN, int BK, int WM, int WN, int KS, int SETS, typename OA, typename OB>
struct SplitShape {
  static constexpr int NT = 64 * WM * WN * KS, TM = BM / WM / 16, TN = BN / WN / 16, U = SETS > 2 ? SETS : 2;
  static_assert(OA::NT == NT && OB::NT == NT && OA::ROWS == BM && OB::ROWS == BN && OA::BK == BK && OB::BK == BK, "one shape");
  static_assert(TM * WM * 16 == BM && TN * WN * 16 == BN && KS * 32 == BK && U % 2 == 0 && U % SETS == 0, "whole blocks");
  static constexpr int STAGE = OA::BYTES + OB::BYTES, RED = 4 * KS * BM * BN;
  static constexpr int LDS = 2 * STAGE > RED ? 2 * STAGE : RED;
  static_assert(LDS >= 4 * BK * (BM + BN), "a stage in fp32");
  static constexpr int EPL = BM * BN / NT;                 // outputs per lane: e = tid + u * NT is (e % BM, e / BM)
  static_assert(EPL * NT == BM * BN, "whole tiles");

  static constexpr int AHEAD = SETS - 1;                   // run() fetches stages up to nst + AHEAD

  struct Acc { ring_f32x4 main[TN][TM], small[TN][TM]; };
  struct Frags { split_bf16x8 a[TM], b[TN]; };             // of one plane

  __device__ __forceinline__ static void read_a(Frags& f, const char* S, int plane, int wm, int wn, int ks, int li, int lk) {
#pragma unroll
    for (int i = 0; i < TM; ++i) f.a[i] = OA::frag(S, plane, ks, lk, (wm * TM + i) * 16 + li);
  }
  __device__ __forceinline__ static void read_b(Frags& f, const char* S, int plane, int wm, int wn, int ks, int li, int lk) {
#pragma unroll
    for (int j = 0; j < TN; ++j) f.b[j] = OB::frag(S + OA::BYTES, plane, ks, lk, (wn * TN + j) * 16 + li);
  }
  __device__ __forceinline__ static void multiply(const Frags& fb, const Frags& fa, ring_f32x4 (&acc)[TN][TM]) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[j][i] = split_mfma(fb.b[j], fa.a[i], acc[j][i]);
  }

  // The tile's sums over nst >= 1 stages, which sum() reads.  kskip terms of the last stage are left out.
  // early(): called while the first loads are on their way.
  template <bool SKIP, typename F>
  __device__ __forceinline__ static void run(char* lds, OA& oa, OB& ob, int nst, int kskip, F early) {
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wv % WM, wn = (wv / WM) % WN, ks = KS > 1 ? wv / (WM * WN) : 0;
    ring_f32x4 ra[SETS][OA::NG], rb[SETS][OB::NG];
#define SPLIT_FETCH(SET, T) do { oa.fetch(T, nst, ra[SET]); ob.fetch(T, nst, rb[SET]); } while (0)
#define SPLIT_STASH(BUF, SET, SK, KMIN)                                         \
  do {                                                                          \
    OA::template stash<SK>(lds + (BUF) * STAGE, tid, ra[SET], KMIN);              \
    OB::template stash<SK>(lds + (BUF) * STAGE + OA::BYTES, tid, rb[SET], KMIN);  \
  } while (0)
    Acc acc;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) acc.main[j][i] = acc.small[j][i] = ring_f32x4{0.f, 0.f, 0.f, 0.f};
    Frags f0[2], f1, f2;                                   // f0: of two stages in turn
#pragma unroll
    for (int i = 0; i < TM; ++i) f0[1].a[i] = f2.a[i] = split_bf16x8{};
#pragma unroll
    for (int j = 0; j < TN; ++j) f0[1].b[j] = f2.b[j] = split_bf16x8{};
    // stage s sits in register set s % SETS until it is written to LDS[s & 1]
#pragma unroll
    for (int q = 0; q < SETS; ++q) SPLIT_FETCH(q, q);
    early();
    SPLIT_STASH(0, 0, SKIP, nst == 1 ? kskip : 0);
    SPLIT_FETCH(0, SETS);
    __syncthreads();
    // A trip: the products of a stage that its last plane takes part in run while the next stage's first plane is read, those
    // of the first plane while the second is, those of the second while the third is.
#define SPLIT_READ(F, P, Q) do { read_b(F, lds + ((Q) & 1) * STAGE, P, wm, wn, ks, li, lk); read_a(F, lds + ((Q) & 1) * STAGE, P, wm, wn, ks, li, lk); } while (0)
#define SPLIT_LAST(Q) do { multiply(f0[(Q) & 1], f2, acc.small); multiply(f2, f0[(Q) & 1], acc.small); } while (0)
#define SPLIT_STAGE(Q)                            \
  do {                                            \
    SPLIT_READ(f0[(Q) & 1], 0, Q);                \
    SPLIT_LAST((Q) + 1);                          \
    SPLIT_READ(f1, 1, Q);                         \
    multiply(f0[(Q) & 1], f0[(Q) & 1], acc.main); \
    SPLIT_READ(f2, 2, Q);                         \
    multiply(f0[(Q) & 1], f1, acc.small);         \
    multiply(f1, f0[(Q) & 1], acc.small);         \
    multiply(f1, f1, acc.small);                  \
  } while (0)
    int s = 0;
    // The code ahead of it decides where the loop falls in the 32 bytes that a fetch of instructions takes, and on 128 x 48 tiles that
    // is up to 3 % of the time: convDown of 96 -> 256 colours 5 x 5, 2 groups, 27 x 27, batch 128 takes 399 us with the loop's head 8 bytes
    // behind a multiple of 32, 402 with 16 or 20, 407 to 411 elsewhere; 84 -> 256 of 9 x 9, stride 2, 15 x 15, 128 233 and 239.  So the
    // place is fixed, 8 bytes in front of the head (4 more where offsets have masks, which make no difference there).  Other tiles
    // differ by 0.5 %.
    if (BN == 48 && U + 1 < nst) asm volatile(".p2align 5\n\ts_nop 0\n\ts_nop 0");
    for (; s + U + 1 < nst; s += U) {
#pragma unroll
      for (int q = 0; q < U; ++q) {
        SPLIT_STAGE(q);
        SPLIT_STASH((q + 1) & 1, (q + 1) % SETS, false, 0);
        SPLIT_FETCH((q + 1) % SETS, s + q + 1 + SETS);
        constexpr int P = TM * TN;
        __builtin_amdgcn_sched_group_barrier(0x100, TM + TN, 0);
#pragma unroll
        for (int g = 0; g < 6 * P; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (g < TM + TN || (g >= 2 * P && g < 2 * P + TM + TN)) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          if (g % 3 == 2) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // the last one to U + 1 stages
#pragma unroll
    for (int q = 0; q <= U; ++q) {
      if (s + q < nst) {
        if (s + q + 1 < nst) SPLIT_STASH((q + 1) & 1, (q + 1) % SETS, SKIP, s + q + 2 == nst ? kskip : 0);
        if (SETS < U && s + q + 1 + SETS < nst) SPLIT_FETCH((q + 1) % SETS, s + q + 1 + SETS);
        SPLIT_STAGE(q);
        if (s + q + 1 == nst) SPLIT_LAST(q);
        __syncthreads();
      }
    }
#undef SPLIT_STASH
#undef SPLIT_READ
#undef SPLIT_STAGE
#undef SPLIT_LAST
    int bad = 0;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float x = acc.main[j][i][v] + acc.small[j][i][v];
          bad |= !(__builtin_fabsf(x) < __builtin_inff());
          acc.main[j][i][v] = x * SPLIT_OUT;
        }
    int* vote = reinterpret_cast<int*>(lds);
    if (tid == 0) *vote = 0;
    __syncthreads();
    if (bad) *vote = 1;
    __syncthreads();
    bad = *vote;
    __syncthreads();
    if (bad) {
      float *SA = reinterpret_cast<float*>(lds), *SB = SA + BK * BM;
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) acc.main[j][i] = ring_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
      for (int t = 0; t < nst; ++t) {
        SPLIT_FETCH(0, t);
        const int kmin = SKIP && t == nst - 1 ? kskip : 0;
        OA::stash32(SA, tid, ra[0], kmin);
        OB::stash32(SB, tid, rb[0], kmin);
        __syncthreads();
#pragma unroll 1
        for (int k = ks * (BK / KS) + lk; k < (ks + 1) * (BK / KS); k += 4) {
          float a[TM], b[TN];
#pragma unroll
          for (int i = 0; i < TM; ++i) a[i] = SA[k * BM + OA::row_of((wm * TM + i) * 16 + li)];
#pragma unroll
          for (int j = 0; j < TN; ++j) b[j] = SB[k * BN + OB::row_of((wn * TN + j) * 16 + li)];
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int i = 0; i < TM; ++i) acc.main[j][i] = ring_mfma(b[j], a[i], acc.main[j][i]);
        }
        __syncthreads();
      }
    }
#undef SPLIT_FETCH
    // acc[j][i][v] is the tile's (m, n) = rows (16 (wm TM + i) + li, 16 (wn TN + j) + 4 lk + v) as slots; partial tiles are [n][m]
    float* part = reinterpret_cast<float*>(lds) + ks * (BM * BN);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float* col = part + OB::row_of((wn * TN + j) * 16 + 4 * lk + v) * BM;
#pragma unroll
        for (int i = 0; i < TM; ++i) col[OA::row_of((wm * TM + i) * 16 + li)] = acc.main[j][i][v];
      }
    __syncthreads();
  }
  // output u of lane `tid`, behind run()
  __device__ __forceinline__ static float sum(const char* lds, int tid, int u) {
    const float* part = reinterpret_cast<const float*>(lds) + tid + NT * u;
    float x = part[0];
#pragma unroll
    for (int w = 1; w < KS; ++w) x += part[w * (BM * BN)];
    return x;
  }
};
