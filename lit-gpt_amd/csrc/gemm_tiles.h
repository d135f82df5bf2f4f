// A tile of a product of two bf16 matrices, C = A B^T, sums in fp32, in the registers of one workgroup: the part that the
// layered models' products (seq_gemm.hip) and the GPT models' (gemm_bf16.hip) share.
//
// A tile of BM x BN outputs belongs to one workgroup of WM x WN waves; a wave holds FM x FN accumulators of
// v_mfma_f32_32x32x16_bf16. A and B reach LDS by LDS-DMA (global_load_lds, 16 bytes a lane, source-swizzled so that
// fragments are read without bank conflicts) in ST stages of BK values of K. Per 16 values of K a wave reads FM + FN
// fragments for FM * FN matrix instructions; the fragments of the next 16 are read while these run, across the stages
// too: the one barrier of a stage stands before its last 16 values' matrix instructions, whose operands are in
// registers by then, and the buffer that it frees is refilled between the matrix instructions that follow.
#pragma once

#include <cmath>

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

template <int WM, int WN, int FM, int FN, int BK, int ST>
struct GemmTile {
  static_assert(BK == 32 || BK == 64, "a row of a stage is half or all of a 128-byte LDS row");
  static constexpr int BM = WM * FM * 32, BN = WN * FN * 32, NW = WM * WN, NT = NW * 64;
  static constexpr int RPL = 64 / BK;                     // matrix rows per LDS row
  static constexpr int STAGE = (BM + BN) / RPL * 128;     // bytes
  static constexpr int ROWS = 8 * RPL;                    // matrix rows per DMA of a wave (1 KB)
  static constexpr int P = (BM + BN) / ROWS / NW;         // DMAs per wave and stage
  static constexpr int H = (P + 1) / 2;                   // ... of these ahead of the next barrier but one
  static_assert((BM + BN) % (ROWS * NW) == 0 && BM % ROWS == 0 && ST >= 2, "every wave issues the same number of DMAs");
  static_assert((ST - 1) * P <= 63, "DMAs in flight are counted in six bits");
  static_assert(ST * STAGE <= 163840, "LDS");
};

// acc = the products of nk stages. src[i]: where lane's 16 bytes of DMA i of its wave begin (piece wave * P + i: eight LDS
// rows, A's first). Accumulator [i][j] of wave (wave % WM, wave / WM): a lane holds row l31 of B's fragment j and rows
// 8 (e / 4) + 4 hi + e % 4 of A's fragment i.
template <int WM, int WN, int FM, int FN, int BK, int ST, int P>
__device__ __forceinline__ void gemm_tile(unsigned char* lds, const unsigned char* const (&src)[P], int nk, int wave,
                                          int lane, f32x16_t (&acc)[FM][FN]) {
  using T = GemmTile<WM, WN, FM, FN, BK, ST>;
  static_assert(P == T::P, "DMAs per wave and stage");
  constexpr int H = T::H;
  // Past the last stage the last one is fetched again into a buffer that nobody reads: the count of DMAs in flight is
  // the same at every barrier, and no branch stands around them.
  auto stage = [&](int k, int buf, int from, int to) {
    const size_t at = (size_t)min(k, nk - 1) * (BK * 2);
#pragma unroll
    for (int i = 0; i < P; ++i)
      if (i >= from && i < to) gemm_dma16(src[i] + at, lds + buf * T::STAGE + (wave * P + i) * 1024);
  };
  const int wm = wave % WM, wn = wave / WM;
  const int l31 = lane & 31, hi = lane >> 5;
  // row l31 of a fragment, chunk hi: its LDS row and swizzled chunk; chunk 2 s + hi lies at that address ^ 32 s
  const int lrow = l31 / T::RPL;
  const int sw = lrow * 128 + 16 * (((l31 % T::RPL) * 4 + hi) ^ (lrow & 7));
  const int abase = wm * FM * 32 / T::RPL * 128 + sw, bbase = (T::BM + wn * FN * 32) / T::RPL * 128 + sw;
  struct Frags {
    gemm_bf16x8 a[FM], b[FN];
  };
  auto read = [&](int buf, int s, Frags& f) {
    const unsigned char* A = lds + buf * T::STAGE + (abase ^ (32 * s));
    const unsigned char* B = lds + buf * T::STAGE + (bbase ^ (32 * s));
#pragma unroll
    for (int j = 0; j < FN; ++j) f.b[j] = *(const gemm_bf16x8*)(B + j * (4096 / T::RPL));
#pragma unroll
    for (int i = 0; i < FM; ++i) f.a[i] = *(const gemm_bf16x8*)(A + i * (4096 / T::RPL));
  };
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  auto mma = [&](const Frags& f) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[i], f.b[j], acc[i][j], 0, 0, 0);
  };
  // after every matrix instruction two reads of the next fragments, after every second a DMA
#define LGS_WEAVE(DMAS)                                                \
  do {                                                                 \
    int rd_ = 0, dma_ = 0;                                             \
    _Pragma("unroll") for (int e_ = 0; e_ < FM * FN; ++e_) {           \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);               \
      _Pragma("unroll") for (int q_ = 0; q_ < 2; ++q_)                 \
        if (rd_ < FM + FN) {                                           \
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);           \
          ++rd_;                                                       \
        }                                                              \
      if (e_ % 2 == 1 && dma_ < (DMAS)) {                              \
        __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);             \
        ++dma_;                                                        \
      }                                                                \
    }                                                                  \
  } while (0)
#pragma unroll
  for (int s = 0; s < ST; ++s) stage(s, s, 0, P);
  gemm_wait_vm<(ST - 1) * P>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  Frags f0, f1;
  read(0, 0, f0);
  int buf = 0, last = ST - 1;  // the buffers of stages k and k - 1
  for (int k = 0; k < nk; ++k) {
    __builtin_amdgcn_sched_barrier(0);
    read(buf, 1, f1);
    stage(k - 1 + ST, last, H, P);  // (first pass: the second half of the last stage of the lead once more)
    mma(f0);
    LGS_WEAVE(P - H);
    if constexpr (BK == 64) {
      __builtin_amdgcn_sched_barrier(0);
      read(buf, 2, f0);
      mma(f1);
      LGS_WEAVE(0);
      __builtin_amdgcn_sched_barrier(0);
      read(buf, 3, f1);
      mma(f0);
      LGS_WEAVE(0);
    }
    __builtin_amdgcn_sched_barrier(0);
    const int next = buf + 1 == ST ? 0 : buf + 1;
    gemm_wait_vm<(ST - 2) * P>();                       // this wave's part of stage k + 1 has landed,
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // and it has read all that it reads of stage k
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    read(next, 0, f0);  // (past the last stage: the repeated one, never used)
    stage(k + ST, buf, 0, H);
    mma(f1);
    LGS_WEAVE(H);
    last = buf;
    buf = next;
  }
#undef LGS_WEAVE
  gemm_wait_vm<0>();  // no DMA may outlive the workgroup's LDS
}

// which row and 16-byte chunk of a stage's BK values lane `lane` of piece row R8 (LDS row) holds
template <int BK>
__device__ __forceinline__ void gemm_dma_at(int R, int lane, int* row, int* chunk) {
  const int lc = (lane & 7) ^ (R & 7);
  *row = BK == 64 ? R : 2 * R + (lc >> 2);
  *chunk = BK == 64 ? lc : lc & 3;
}
// The tile forms, and what a stage of 64 values of K costs a full chip of their workgroups, measured on products of
// 2048 x 2048 x 2048 to 2407 x 22016 x 4096: a tile of 256 x 256 runs 1.80 us per 64 values (1190 TFLOP/s, 0.79 of
// what a large matrix product reaches on this card), of 256 x 128 1.02, of 128 x 128 0.63 alone on a compute unit and
// 1.14 for two, of 64 x 128 0.43. The larger tile moves fewer bytes per product, the smaller ones fill the chip when
// rows or columns are few. A workgroup's start and end cost about 3 us.
// X(index, workgroups of the whole chip at a time, us, waves WM x WN, fragments FM x FN, BK, stages)
#define LGA_GEMM_FORMS(X)                  \
  X(0, 256, 1.80f, 2, 4, 4, 2, 32, 5)      \
  X(1, 256, 1.02f, 4, 2, 2, 2, 64, 3)      \
  X(2, 512, 1.14f, 2, 2, 2, 2, 64, 2)      \
  X(3, 256, 0.63f, 2, 4, 2, 1, 64, 4)      \
  X(4, 256, 0.43f, 1, 4, 2, 1, 64, 4)
struct GemmForm {
  int bm, bn, slots;
  float step_us;
};
#define LGA_GEMM_FORM(I, SLOTS, US, ...) {GemmTile<__VA_ARGS__>::BM, GemmTile<__VA_ARGS__>::BN, SLOTS, US},
constexpr GemmForm kGemmForms[] = {LGA_GEMM_FORMS(LGA_GEMM_FORM)};
#undef LGA_GEMM_FORM

// Which form, and how many ranges of K (ksplit 0: the plan's own choice); tile -1: K is no multiple of 64.
struct GemmPlan {
  int tile, ksplit;
};
// Rounds of workgroups times what one takes; several ranges of K cost a second launch that reads them all. E.g.
// 2048 x 2048 x 5632: 256 tiles of 128 x 128 in one round, 55 us (64 of 256 x 256: 131); 128 x 4096 x 4096: 64 tiles of
// 64 x 128 in four ranges of K, 16 us (whole: 41); before these tiles 126 and 86 us.
// rows_b: the rows are the tile's B, the columns its A.
inline GemmPlan gemm_tile_plan(int M, int N, int K, int batch, bool grouped, int ksplit, bool rows_b = false) {
  GemmPlan best{-1, 1};
  if (K % 64 != 0 || M <= 0) return best;
  const int steps = K / 64;
  float best_us = 0.0f;
  for (int f = 0; f < (int)(sizeof(kGemmForms) / sizeof(kGemmForms[0])); ++f) {
    const GemmForm& t = kGemmForms[f];
    const int rows = rows_b ? t.bn : t.bm, cols = rows_b ? t.bm : t.bn;
    const float nt = (float)((N + cols - 1) / cols);
    // a range of the list ends somewhere in its last tile
    const float mt = grouped ? (float)M / rows + 0.5f * batch : (float)((M + rows - 1) / rows) * batch;
    const int s_lo = ksplit > 0 ? ksplit : 1, s_hi = ksplit > 0 ? ksplit : (batch > 1 || grouped ? 1 : 16);
    for (int s = s_lo; s <= s_hi && (s == s_lo || steps / s >= 4); ++s) {
      const int per = (steps + s - 1) / s;
      const float rounds = ceilf(mt * nt * (float)((steps + per - 1) / per) / (float)t.slots);
      float us = rounds * (per * t.step_us + 3.0f);
      if (s > 1) us += 5.0f + (float)M * N * 4.0f * (2 * s + 1) / 3.0e6f;
      if (best.tile < 0 || us < best_us) {
        best_us = us;
        best = GemmPlan{f, s};
      }
    }
  }
  return best;
}


}  // namespace lga
