// The operands of lgs_linear and its large-tile form (seq_gemm.hip).
#pragma once

#include "gemm_tiles.h"
#include "seq_common.h"

namespace lgs {

struct LinArgs {
  const float* a;
  long lda, sa;
  const void* w;
  long sw;
  float* y;
  long ldy, sy;
  int M, N, K;
  int accumulate, act;
  const int* a_rows;   // row r of the list reads A row a_rows[r] (null: r)
  const int* z_start;  // batch z owns list rows [z_start[z], z_start[z + 1]) (null: rows [0, M) in every batch)
  const uint16_t* a16;  // MFMA tiles only: A as bf16 (a producer's rounded copy) instead of fp32 `a`
  uint16_t* y16;        // MFMA tiles only: Y written as bf16 (the operand of a following bf16 product), no accumulate
  const float* bias;    // [N] added to the product ahead of the activation (null: none)
  float* part;          // MFMA tiles only: partial sums [ksplit][M][N] of equal ranges of K, summed by lin_sum_kernel
  int ksplit, kper;     // (ksplit 1: none); kper: BK-deep steps per range
};

// Which tile form and how many ranges of K a product of bf16 A and W takes on the pipelined tiles (seq_gemm.hip); tile
// -1: not one of theirs (K is no multiple of 64). Rows of A and W start on 16 bytes. ksplit 0: the plan's own choice.
using lga::GemmPlan;
GemmPlan gemm_plan(int M, int N, int K, int batch, bool grouped, int ksplit, int act = kActNone, bool sums = false);
GemmPlan gemm_glu_plan(int M, int n, int K, int batch, bool grouped);
int gemm_launch(const LinArgs& p, const GemmPlan& plan, int batch, hipStream_t stream);

// Up to 32 columns on a kernel of their own: false where it does not take the product (nothing is launched)
bool gemm_narrow(const LinArgs& p, int batch, hipStream_t stream);

// A grouped product whose list is one tile of lgs_linear's older kernel and whose groups have two rows or less: that kernel
// finds a group's rows by its place in the grid, where every workgroup here looks the list's groups through and most have
// nothing to do. us there / here of top-4 routed tokens, up and down products: 64 experts of 512 x 2048, 13 tokens 45 + 30 / 60
// + 34, 32 tokens 50 + 34 / 71 + 37, 33 tokens 92 + 57 / 68 + 36; 128 of 256 x 1024, 13 tokens 27 + 11 / 36 + 25; 40 of 1024 x
// 4096, 13 tokens 124 + 51 / 136 + 67, 26 tokens 222 + 93 / 155 + 72; 24 of 512 x 2048, 13 tokens 41 + 19 / 32 + 16
inline bool gemm_few_rows(int M, int groups) { return M <= 128 && M <= 2 * groups; }

// the gated unit on two products: act(gate) * up, or clamped: g sigmoid(alpha g) (u + shift) with g = min(gate, limit),
// u = clamp(up, -limit, limit) (limit <= 0: no clamps)
struct GluForm {
  int clamped, act;
  float alpha, limit, shift;
  size_t up;  // where the up rows begin in W, from the gate rows (elements)
};
template <bool CLAMPED>
__device__ __forceinline__ float glu_f(const GluForm& f, float g, float u) {
  if (!CLAMPED) return act_f(f.act, g) * u;
  if (f.limit > 0.0f) {
    g = fminf(g, f.limit);
    u = fminf(fmaxf(u, -f.limit), f.limit);
  }
  return g * sigmoid_f(f.alpha * g) * (u + f.shift);
}
int gemm_glu_launch(const LinArgs& p, const GluForm& f, int batch, hipStream_t stream);

}  // namespace lgs
