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

// long prompts and most short ones (gemm_q4r.hip). fn: 32-row pieces of X per tile (0: not one of its products), per: pairs of steps
// of 64 values
struct Q4rPlan {
  int fn, mt, nt, splits, per;
};
Q4rPlan q4r_plan(int M, int N, int K, bool dual, int kernel_fmt, bool ranges);  // ranges: there is a workspace for the plan's ranges of K
size_t q4r_workspace(const Q4rPlan& p, int M, int N, bool dual);
int q4r_run(const Q4dArgs& a, const Q4rPlan& p, int kernel_fmt, bool dual, hipStream_t stream);
int preload_gemm_q4r();

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

// silu of a bf16 number for a result rounded to bf16, in a third of silu_f's instructions: of all 65536 inputs the same bits as
// round_bf(silu_f(x)). The quarter keeps the reciprocal out of the denormal numbers, which it flushes (-87.5 to -88.5 were 0), the
// bound its correction from an infinity times 0; without the correction 5.9375 fell on the other side of a tie.
__device__ __forceinline__ float silu_bf(float x) {
  const float d = fminf(__builtin_fmaf(__builtin_amdgcn_exp2f(x * -1.44269504f), 0.25f, 0.25f), 3.40282347e38f);
  const float r = __builtin_amdgcn_rcpf(d);
  return (0.25f * x) * __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
}

// A row's 32 columns [n, n + 32) of a product, held by two lanes as an accumulator of v_mfma_f32_32x32x16_bf16 with the weights
// as A has them (lane half hi: columns 8 q + 4 hi + e of register 4 q + e): the halves swap, so that a lane has eight
// neighbouring columns and stores 16 bytes. h2: the second matrix' (SwiGLU).
template <bool DUAL>
__device__ __forceinline__ void q4d_store_fragment(const Q4dArgs& a, const f32x16_t& h1, const f32x16_t& h2, int m, int n,
                                                   int hi, int split, int splits) {
  const size_t ldy = a.ldy ? a.ldy : a.N;
#pragma unroll
  for (int q = 0; q < 4; q += 2) {
    float v[8], u[8];
    auto swap = [&](const f32x16_t& h, float (&o)[8]) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(h[q * 4 + e]), __float_as_uint(h[q * 4 + 4 + e]), false, false);
        o[e] = __uint_as_float(r[0]), o[4 + e] = __uint_as_float(r[1]);
      }
    };
    swap(h1, v);
    if (DUAL) swap(h2, u);
    const int c = n + (q + hi) * 8;
    if (m >= a.M || c >= a.N) continue;
    if (splits > 1) {
      float* o = a.slabs + ((size_t)split * (DUAL ? 2 : 1) * a.M + m) * a.N + c;
      *(q4d_f32x4*)o = q4d_f32x4{v[0], v[1], v[2], v[3]}, *(q4d_f32x4*)(o + 4) = q4d_f32x4{v[4], v[5], v[6], v[7]};
      if (DUAL) {
        o += (size_t)a.M * a.N;
        *(q4d_f32x4*)o = q4d_f32x4{u[0], u[1], u[2], u[3]}, *(q4d_f32x4*)(o + 4) = q4d_f32x4{u[4], u[5], u[6], u[7]};
      }
      continue;
    }
    if (DUAL) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = __fmul_rn(round_bf(silu_bf(round_bf(v[e]))), round_bf(u[e]));
    } else {
      auto eight = [](const uint16_t* p, float (&o)[8]) {
        const uint4 w = *(const uint4*)p;
        o[0] = bflo(w.x), o[1] = bfhi(w.x), o[2] = bflo(w.y), o[3] = bfhi(w.y);
        o[4] = bflo(w.z), o[5] = bfhi(w.z), o[6] = bflo(w.w), o[7] = bfhi(w.w);
      };
      if (a.bias) {
        // (a bias starts where its caller put it)
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
          const uint2 b = *(const uint2*)(a.bias + c + e);
          v[e] += bflo(b.x), v[e + 1] += bfhi(b.x), v[e + 2] += bflo(b.y), v[e + 3] += bfhi(b.y);
        }
      }
      if (a.residual) {
        float r[8];
        eight(a.residual + m * ldy + c, r);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = round_bf(v[e]) + r[e];
      }
    }
    *(uint4*)(a.y + m * ldy + c) = make_uint4(pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7]));
  }
}

}  // namespace lga
