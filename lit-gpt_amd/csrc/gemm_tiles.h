// A tile of a product of two bf16 matrices, C = A B^T, sums in fp32, in the registers of one workgroup: the part that the
// layered models' products (seq_gemm.hip) and the GPT models' (gemm_bf16.hip) share.
//
// A tile of BM x BN outputs belongs to one workgroup of WM x WN waves; a wave holds FM x FN accumulators of
// v_mfma_f32_32x32x16_bf16. A and B reach LDS by LDS-DMA (global_load_lds, 16 bytes a lane, whole 128-byte lines of a row,
// source-swizzled so that fragments are read without bank conflicts) in steps of 64 values of K, A's rows into a ring of RA
// buffers, B's into one of RB: three and two of a 256 x 256 tile fill the 160 KB. Per 16 values of K a wave reads FM + FN
// fragments for FM * FN matrix instructions; the fragments of the next 16 are read while these run, across the steps
// too: the one barrier of a step stands before its last 16 values' matrix instructions, whose operands are in registers by
// then, and the buffers that it frees are refilled between the matrix instructions that follow. Where reads and DMAs stand
// among the matrix instructions is written out (sched_barrier), not left to the scheduler, which bunches the DMAs.
//
// What bounds it: LDS has 128 bytes a clock for the fragments and the DMAs. Four waves of 128 x 128 read 1024 clocks' worth
// per step of 64 and the DMAs write 512, for 2048 clocks of matrix instructions; eight waves of 128 x 64 would read 1536.
// Measured 2340 clocks a step, 1.48 us at the 1.6 GHz that a full chip of matrix instructions is left with (power), where
// stages of 32 values (half lines) in one ring took 3230 clocks, 1.8 us: 2048 x 22016 x 4096 355 -> 296 us, 8192 x 8192 x
// 8192 950 -> 804. Both give the same bits.
#pragma once

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"

namespace lga {

typedef __bf16 gemm_bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

__device__ __forceinline__ void gemm_dma16(const void* src, unsigned char* lds) {
  __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}
template <int N>  // until at most N of this wave's DMAs are in flight (the count is a field of the instruction)
__device__ __forceinline__ void gemm_wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <int WM, int WN, int FM, int FN, int RA, int RB>
struct GemmTile {
  static constexpr int BM = WM * FM * 32, BN = WN * FN * 32, NW = WM * WN, NT = NW * 64;
  static constexpr int A_BYTES = BM * 128, B_BYTES = BN * 128, LDS = RA * A_BYTES + RB * B_BYTES;
  static constexpr int PA = BM / 8 / NW, PB = BN / 8 / NW;  // DMAs (8 rows, 1 KB) per wave and step
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "every wave issues the same number of DMAs");
  static_assert(RA >= 2 && (RB == RA || RB == RA - 1), "one buffer in use, the others on their way");
  static_assert((RA - 1) * (PA + PB) <= 63, "DMAs in flight are counted in six bits");
  static_assert(LDS <= 163840, "LDS");
};

// which row and 16-byte chunk of a step's 128 bytes lane `lane` of piece `piece` (8 rows) fetches
__device__ __forceinline__ void gemm_dma_at(int piece, int lane, int* row, int* chunk) {
  *row = piece * 8 + (lane >> 3);
  *chunk = (lane & 7) ^ (*row & 7);
}

// acc = the products of nk steps. a[i], b[i]: where lane's 16 bytes of DMA i of its wave begin (pieces wave * PA + i of A's
// rows, wave * PB + i of B's). Accumulator [i][j] of wave (wave % WM, wave / WM): a lane holds row l31 of B's fragment j
// and rows 8 (e / 4) + 4 hi + e % 4 of A's fragment i.
template <int WM, int WN, int FM, int FN, int RA, int RB, int PA, int PB>
__device__ __forceinline__ void gemm_tile(unsigned char* lds, const unsigned char* const (&a)[PA],
                                          const unsigned char* const (&b)[PB], int nk, int wave, int lane,
                                          f32x16_t (&acc)[FM][FN]) {
  using T = GemmTile<WM, WN, FM, FN, RA, RB>;
  static_assert(PA == T::PA && PB == T::PB, "DMAs per wave and step");
  // Past the last step the last one is fetched again into a buffer that nobody reads: the count of DMAs in flight is
  // the same at every barrier, and no branch stands around them.
  auto dma_a = [&](int i, int k, int slot) {
    gemm_dma16(a[i] + (size_t)min(k, nk - 1) * 128, lds + slot * T::A_BYTES + (wave * PA + i) * 1024);
  };
  auto dma_b = [&](int i, int k, int slot) {
    gemm_dma16(b[i] + (size_t)min(k, nk - 1) * 128, lds + RA * T::A_BYTES + slot * T::B_BYTES + (wave * PB + i) * 1024);
  };
  // row l31 of a fragment, chunk hi, swizzled; chunk 2 s + hi lies at that address ^ 32 s
  const int wm = wave % WM, wn = wave / WM, l31 = lane & 31, hi = lane >> 5;
  const int sw = l31 * 128 + 16 * (hi ^ (l31 & 7));
  const int a_at = wm * FM * 4096 + sw, b_at = RA * T::A_BYTES + wn * FN * 4096 + sw;
  struct Frags {
    gemm_bf16x8 a[FM], b[FN];
  };
  // fragment number n in the order of use: a0, b0, b1, .. , a1, a2, ..
  auto read = [&](Frags& f, int n, int sa, int sb, int s) {
    if (n >= 1 && n <= FN) {
      f.b[n - 1] = *(const gemm_bf16x8*)(lds + sb * T::B_BYTES + (b_at ^ (32 * s)) + (n - 1) * 4096);
    } else {
      const int i = n == 0 ? 0 : n - FN;
      f.a[i] = *(const gemm_bf16x8*)(lds + sa * T::A_BYTES + (a_at ^ (32 * s)) + i * 4096);
    }
  };
  // the matrix instructions of 16 values of K, and among them the reads of the next 16 and ND DMAs
  auto mma = [&](const Frags& f, Frags& g, int sa, int sb, int s, auto nd, auto&& dma) {
    constexpr int ND = decltype(nd)::value, E = FM * FN, READS = (FM + FN + E - 1) / E;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      acc[e / FN][e % FN] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[e / FN], f.b[e % FN], acc[e / FN][e % FN], 0, 0, 0);
#pragma unroll
      for (int n = e * READS; n < (e + 1) * READS && n < FM + FN; ++n) read(g, n, sa, sb, s);
#pragma unroll
      for (int q = ND * e / E; q < ND * (e + 1) / E; ++q) dma(q);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  constexpr std::integral_constant<int, PA> all_a{};
  constexpr std::integral_constant<int, PB> all_b{};
  constexpr std::integral_constant<int, 0> none{};
  auto no_dma = [](int) {};
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
#pragma unroll
  for (int s = 0; s < RA - 1; ++s) {
#pragma unroll
    for (int i = 0; i < PA; ++i) dma_a(i, s, s);
#pragma unroll
    for (int i = 0; i < PB; ++i) dma_b(i, s, s);
  }
  gemm_wait_vm<(RA - 2) * (PA + PB)>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  Frags f0, f1;
#pragma unroll
  for (int n = 0; n < FM + FN; ++n) read(f0, n, 0, 0, 0);
  // buffers: sa, sb of this step; free_a, free_b those that the last barrier freed (at first the ones never filled)
  int sa = 0, sb = 0, free_a = RA - 1, free_b = RB - 1;
  for (int k = 0; k < nk; ++k) {
    const int na = sa + 1 == RA ? 0 : sa + 1, nb = sb + 1 == RB ? 0 : sb + 1;
    __builtin_amdgcn_sched_barrier(0);
    mma(f0, f1, sa, sb, 1, all_a, [&](int i) { dma_a(i, k + RA - 1, free_a); });
    if constexpr (RB == RA) mma(f1, f0, sa, sb, 2, all_b, [&](int i) { dma_b(i, k + RB - 1, free_b); });
    else mma(f1, f0, sa, sb, 2, none, no_dma);
    mma(f0, f1, sa, sb, 3, none, no_dma);
    // this wave's part of step k + 1 has landed (what it issued later may still be on its way), ...
    gemm_wait_vm<RB == RA ? (RA - 2) * (PA + PB) : (RA - 2) * PA + (RB - 2) * PB>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // ... and it has read all that it reads of step k
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    // (past the last step: the repeated one, never used)
    if constexpr (RB == RA) mma(f1, f0, na, nb, 0, none, no_dma);
    else mma(f1, f0, na, nb, 0, all_b, [&](int i) { dma_b(i, k + RB, sb); });
    free_a = sa, free_b = sb;
    sa = na, sb = nb;
  }
  gemm_wait_vm<0>();  // no DMA may outlive the workgroup's LDS
}

// The rows past the last whole tile get a tile of their own with fewer fragments along them: the same columns, waves and
// sums, in the LDS that the whole tile leaves, so a matrix instruction works on at most STEP - 1 rows that are not there. The
// short tiles stand last in the grid and fill the whole ones' last round.
template <int WM, int WN, int FM, int FN, int MOST>
struct GemmShort {
  static constexpr int A = WM * FM * 4096, B = WN * FN * 4096, FIT = MOST / (A + B), R = FIT < 6 ? FIT : 6;
  static constexpr int RA = R < 3 && (R + 1) * A + R * B <= MOST ? R + 1 : R, RB = R;
  using T = GemmTile<WM, WN, FM, FN, RA, RB>;
};
template <class T>
constexpr int kGemmLds = T::LDS > 81920 ? 163840 : 81920;  // (two workgroups on a CU or one)

// rows: whole tiles of ROWS, a short one behind them that leaves STEP rows out at least
template <int ROWS, int STEP>
__host__ __device__ constexpr int gemm_whole(int rows) {
  return rows / ROWS + (rows % ROWS > ROWS - STEP ? 1 : 0);
}
// Workgroup b runs on XCD b % 8, and an XCD takes neighbouring tiles, whose rows and columns its L2 then holds: of `whole` ones, then
// of `last` ones, as many as any other XCD or one less (an XCD with a tile more than it has compute units makes them in two rounds).
// Its place in the first list, or else (false) in the second; -1: none is left.
__device__ __forceinline__ bool gemm_xcd(int whole, int last, int* t) {
  const int x = blockIdx.x & 7, at = blockIdx.x >> 3, q = whole / 8, r = whole % 8, own = q + (x < r ? 1 : 0);
  if (at < own) {
    *t = x * q + min(x, r) + at;
    return true;
  }
  const int ql = last / 8, rl = last % 8, more = x - (8 - rl);  // (the odd ones to the XCDs at the other end)
  *t = at - own < ql + (more >= 0 ? 1 : 0) ? x * ql + max(more, 0) + at - own : -1;
  return false;
}
inline unsigned gemm_grid(long tiles) { return (unsigned)((tiles + 7) / 8 * 8); }
// Where a workgroup's tile lies among those of `count` products (batches or ranges of K), the short tiles behind all whole ones
struct GemmAt {
  int which, m, n;
};
template <int ROWS, int STEP>
__device__ __forceinline__ bool gemm_at(int rows, int nt, int count, GemmAt* o) {
  const int all = (rows + ROWS - 1) / ROWS, mt = gemm_whole<ROWS, STEP>(rows), per = mt * nt;
  int t;
  if (gemm_xcd(count * per, count * (all - mt) * nt, &t)) {
    o->which = t / per;
    t -= o->which * per;
    const int g = t / (8 * nt), gm = min(8, mt - g * 8);  // groups of up to 8 row tiles
    t -= g * 8 * nt;
    o->m = g * 8 + t % gm, o->n = t / gm;
    return true;
  }
  if (t < 0) return false;
  o->which = t / nt, o->m = mt, o->n = t % nt;
  return true;
}
// The tile forms: what a step of 64 values of K costs a full chip of their workgroups, and what it would cost at the 2.4 GHz
// that a chip with few of them runs at; start, end and fp32 results of a round of them. Measured on 256 tiles (512 of the
// form of which a compute unit holds two) and K 1024 and 4096. The larger tile moves fewer bytes per product (256 x 256:
// 1450 TFLOP/s, 256 x 128 1290, 128 x 128 1190, 64 x 128 940), the smaller ones fill the chip when rows or columns are few.
// X(index, workgroups of the whole chip at a time, us of a step, us of it at 2.4 GHz, us of a round, waves WM x WN,
//   fragments FM x FN, rings RA, RB)
#define LGA_GEMM_FORMS(X)                                 \
  X(0, 256, 1.48f, 0.98f, 15.5f, 2, 2, 4, 4, 3, 2)        \
  X(1, 256, 1.165f, 0.745f, 10.6f, 2, 2, 4, 3, 3, 2)      \
  X(2, 256, 0.835f, 0.547f, 8.0f, 2, 2, 4, 2, 3, 3)       \
  X(3, 256, 0.833f, 0.544f, 7.4f, 2, 2, 2, 4, 3, 3)       \
  X(4, 256, 0.65f, 0.439f, 5.9f, 2, 2, 2, 3, 4, 4)        \
  X(5, 512, 0.898f, 0.593f, 7.1f, 2, 2, 2, 2, 2, 2)       \
  X(6, 256, 0.45f, 0.38f, 5.5f, 2, 4, 2, 1, 5, 5)         \
  X(7, 256, 0.285f, 0.275f, 4.9f, 1, 4, 2, 1, 6, 6)       \
  X(8, 256, 1.163f, 0.745f, 10.3f, 2, 2, 3, 4, 3, 2)
struct GemmForm {
  int bm, bn, fm, fn, slots;
  float step_us, fast_us, round_us;
};
#define LGA_GEMM_FORM(I, SLOTS, US, FAST, ROUND, WM, WN, FM, FN, ...) {WM * FM * 32, WN * FN * 32, FM, FN, SLOTS, US, FAST, ROUND},
constexpr GemmForm kGemmForms[] = {LGA_GEMM_FORMS(LGA_GEMM_FORM)};
#undef LGA_GEMM_FORM
constexpr int kGemmFormCount = sizeof(kGemmForms) / sizeof(kGemmForms[0]);

// Which form, and how many ranges of K (ksplit 0: the plan's own choice); tile -1: K is no multiple of 64.
struct GemmPlan {
  int tile, ksplit;
};
enum {
  kGemmRowsB = 1,  // the rows are the tile's B, the columns its A
  kGemmPairs = 2,  // A's fragments are those of two matrices in turn: forms with an even number of them
  kGemmActs = 4,   // forms whose code holds activations
  kGemmSums = 8    // results go into sums
};
inline bool gemm_form_fits(const GemmForm& t, int flags) {
  return !((flags & kGemmActs && t.bm * t.bn > 256 * 128) || (flags & kGemmPairs && t.fm % 2));
}
// (a plan is made at every launch: no library call for a rounding, nothing of the ranges for each form anew. us a plan, mean of 66 sizes,
// with both / here: ranges to choose 2.34 / 0.85, given 0.45 / 0.14)
// (of 0 to 2^63)
inline float gemm_floor(float v) { return (float)(long)v; }
inline float gemm_ceil(float v) { return gemm_floor(v) + (gemm_floor(v) < v ? 1.0f : 0.0f); }
// Counted in whole tiles: rounds of workgroups times what one takes; several ranges of K cost a second launch that reads them all.
// Against all forms and ranges on 24 products of 64 to 4096 rows, weights from memory, the choice was the fastest or within 7 % of it
// before there were short tiles. It still says the ranges, and with them the order of a product's sums, and the forms of grouped products.
inline GemmPlan gemm_whole_plan(int M, int N, int K, int batch, bool grouped, int ksplit, int flags) {
  GemmPlan best{-1, 1};
  if (K % 64 != 0 || M <= 0) return best;
  constexpr int kMost = 16;
  const int steps = K / 64, s_lo = ksplit > 0 ? ksplit : 1, s_hi = ksplit > 0 ? ksplit : (batch > 1 || grouped ? 1 : kMost);
  int each[kMost], count = 0;  // steps of a range, by the number of ranges asked for
  float made[kMost];           // ranges that there are
  for (int s = s_lo; s <= s_hi && (s == s_lo || steps / s >= 4); ++s, ++count) {
    each[count] = (steps + s - 1) / s;
    made[count] = (float)((steps + each[count] - 1) / each[count]);
  }
  float best_us = 0.0f;
#pragma unroll
  for (int f = 0; f < kGemmFormCount; ++f) {
    const GemmForm& t = kGemmForms[f];
    if (!gemm_form_fits(t, flags)) continue;
    const int rows = flags & kGemmRowsB ? t.bn : t.bm, cols = flags & kGemmRowsB ? t.bm : t.bn;
    const float nt = (float)((N + cols - 1) / cols);
    // a range of the list ends somewhere in its last tile, and has one
    const float mt = grouped ? std::max((float)M / rows + 0.5f * batch, (float)std::min(batch, M)) : (float)((M + rows - 1) / rows) * batch;
    for (int i = 0; i < count; ++i) {
      const int s = s_lo + i, per = each[i];
      const float rounds = mt * nt * made[i] / (float)t.slots, whole = gemm_floor(rounds);
      float us = (grouped && rounds > 1.0f ? rounds + 0.5f : whole) * (per * t.step_us + t.round_us);
      if (grouped ? rounds <= 1.0f : rounds > whole) {
        // few workgroups have a higher clock: 160 of 256 x 256 take 0.74 of 256's time; smaller tiles, which draw less, 0.82
        const float most = t.bm * t.bn > 128 * 192 ? 0.7f : 0.5f;
        us += per * std::max(t.fast_us, t.step_us * (1.0f - most * (1.0f - (rounds - whole)))) + t.round_us;
      }
      if (s > 1) us += 2.0f + (float)M * N * 4.0f * (s + 1) / 5.5e6f;
      if (best.tile < 0 || us < best_us) best_us = us, best.tile = f, best.ksplit = s;
    }
  }
  return best;
}

// The form of a plain product for these ranges: whole tiles' rounds, the short ones among the last of them or behind, where they fill
// the chip's idle part. Of 1491 products of 33 to 2600 rows, weights from memory, it is 1.1 % from the fastest form in the mean, and
// the form that counts whole tiles 2.0 %. us of whole tiles alone / here: 2407 x 20608 x 4096 448 / 381, 517 x 11008 x 4096 with SwiGLU
// 109 / 101, 40 rows of it 37 / 33.
// Rows as the tile's B: at least nine steps, and a fortieth gained, or else the form that counts whole tiles. (Ends of tiles are most
// of shorter products, and of 64 x 128 they are less than the sums here say: 990 products for which the two choose otherwise, the sums' choice
// alone 1.04 times the time of whole tiles' for plain ones, 1.06 for gated units, with the line 0.99 and 0.99; 120 x 768 x 3072 10.8 / 12.1, 2849
// x twice 5524 x 512 53 / 62. Rows as A 0.93, at every length; but activations into sums, where ends of tiles are the most work, need nine
// steps too: 2084 x 3159 x 256 24.1 / 33.8, 291 x 17493 x 192 22.6 / 30.2.)
// A grouped product's short tiles stand beside the whole ones of their columns, whose weights they would otherwise fetch anew (16 groups of
// 278 rows of twice 2752 x 4096 302 behind, 260 beside): 480 products of 8 to 18 groups, 144 to 16384 rows in all, weights from memory,
// take 0.93 of the time that whole tiles took (gated units 0.98), none more than 3 % more. (Weights that stay in the last cache from
// call to call gain less, up to 6 % lost.)
inline GemmPlan gemm_tile_plan(int M, int N, int K, int batch, bool grouped, int ksplit, int flags) {
  GemmPlan best{-1, 1};
  if (grouped) return gemm_whole_plan(M, N, K, batch, true, ksplit, flags);
  if (K % 64 != 0 || M <= 0) return best;
  const bool rows_b = flags & kGemmRowsB, acts_sums = flags & kGemmActs && flags & kGemmSums;
  if (rows_b || acts_sums || (ksplit <= 0 && batch == 1)) best = gemm_whole_plan(M, N, K, batch, false, ksplit, flags);
  else best.ksplit = ksplit > 0 ? ksplit : 1;
  const int steps = K / 64, per = (steps + best.ksplit - 1) / best.ksplit, count = batch * ((steps + per - 1) / per);
  if ((rows_b || acts_sums) && per < 9) return best;
  const int kept = best.tile;
  float best_us = 0.0f, kept_us = 0.0f;
#pragma unroll
  for (int f = 0; f < kGemmFormCount; ++f) {
    const GemmForm& t = kGemmForms[f];
    if (!gemm_form_fits(t, flags)) continue;
    const int rows = rows_b ? t.bn : t.bm, cols = rows_b ? t.bm : t.bn, frags = rows_b ? t.fn : t.fm, step = rows / frags;
    // (of what fewer workgroups gain: 0.7 and 0.5 above, fitted anew on these products)
    const float most = t.bm * t.bn > 128 * 192 ? 0.69f : 0.46f;
    auto round = [&](float load) { return per * std::max(t.fast_us, t.step_us * (1.0f - most * (1.0f - load))) + t.round_us; };
    const int pieces = (M + step - 1) / step, mt = pieces / frags, left = pieces % frags;
    const float nt = (float)((N + cols - 1) / cols), slots = (float)t.slots;
    const float whole = mt * nt * count, full = gemm_floor(whole / slots), over = whole - full * slots;
    // a short tile's time of a whole one's; alone on the chip it is mostly latency
    const float each = left == 0 ? 1.0f : std::max(0.3f + 0.7f * left / frags, mt > 0 ? 0.0f : 0.75f);
    float shorts = left ? nt * count : 0.0f, us;
    us = full * round(1.0f);
    if (over > 0.0f) {
      const float beside = std::min(shorts, (slots - over) * gemm_floor(1.0f / each));
      us += round((over + beside * each) / slots);
      shorts -= beside;
    }
    if (shorts > 0.0f) us += each * gemm_ceil(shorts / slots) * round(std::min(shorts / slots, 1.0f) * each);
    if (best_us == 0.0f || us < best_us) best_us = us, best.tile = f;
    if (f == kept) kept_us = us;
  }
  if (rows_b && best_us > 0.975f * kept_us) best.tile = kept;
  return best;
}

}  // namespace lga
