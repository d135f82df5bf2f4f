// The register-dequantizing prefill GEMM (gemm_q4d.hip) and the bf16 weights' tiles (gemm_bf16.hip), called by the fused
// GEMM's entry points (gemm_q4f.hip).
#pragma once

#include "gemm_tiles.h"

namespace lga {

struct Q4dArgs {
  const uint16_t* x;  // [M][K]
  const void *w, *sc, *w2, *sc2;  // as the fused GEMM's; w2 / sc2: fc_2 of the SwiGLU form
  const uint16_t* bias;
  const uint16_t* residual;  // [M][N]
  uint16_t* y;
  int M, N, K, G, ldy, cb;
  float* slabs;  // [splits][1 or 2][M][N] partial sums
};

// mf: 16-row pieces of X per tile (0: not one of its products), mt / nt: tiles over rows and columns, splits ranges of K
// of `per` blocks of 128
struct Q4dPlan {
  int mf, mt, nt, splits, per;
};
Q4dPlan q4d_plan(int M, int N, int K, bool dual);
size_t q4d_workspace(const Q4dPlan& p, int M, int N, bool dual);
int q4d_run(const Q4dArgs& a, const Q4dPlan& p, int kernel_fmt, bool dual, hipStream_t stream);
// the partial sums of `splits` ranges of K in order, then the epilogue
void q4d_sum(const Q4dArgs& a, int splits, bool dual, hipStream_t stream);
int preload_gemm_q4d();

GemmPlan bf16_plan(int M, int N, int K, bool dual);
size_t bf16_workspace(const GemmPlan& p, int M, int N, bool dual);
int bf16_run(const Q4dArgs& a, const GemmPlan& p, bool dual, hipStream_t stream);
int preload_gemm_bf16();

typedef float q4d_f32x4 __attribute__((ext_vector_type(4)));

// bf16(bf16(silu(bf16 h1)) * bf16 h2) of four columns
__device__ __forceinline__ uint2 q4d_swiglu(q4d_f32x4 h1, q4d_f32x4 h2) {
  float g[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) g[e] = __fmul_rn(round_bf(silu_f(round_bf(h1[e]))), round_bf(h2[e]));
  return make_uint2(pack2(g[0], g[1]), pack2(g[2], g[3]));
}
// bf16(h + bias), then bf16 of its sum with the residual
__device__ __forceinline__ void q4d_store(const Q4dArgs& a, int m, int n, size_t ldy, q4d_f32x4 h) {
  float v[4] = {h[0], h[1], h[2], h[3]};
  if (a.bias) {
    const uint2 b = *(const uint2*)(a.bias + n);
    v[0] += bflo(b.x), v[1] += bfhi(b.x), v[2] += bflo(b.y), v[3] += bfhi(b.y);
  }
  if (a.residual) {
    const uint2 r = *(const uint2*)(a.residual + m * ldy + n);
    v[0] = round_bf(v[0]) + bflo(r.x), v[1] = round_bf(v[1]) + bfhi(r.x);
    v[2] = round_bf(v[2]) + bflo(r.y), v[3] = round_bf(v[3]) + bfhi(r.y);
  }
  *(uint2*)(a.y + m * ldy + n) = make_uint2(pack2(v[0], v[1]), pack2(v[2], v[3]));
}

}  // namespace lga
