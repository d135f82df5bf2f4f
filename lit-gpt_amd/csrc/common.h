// Shared device helpers for the lit-gpt MI355X (gfx950) decode path.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lga {

constexpr int kWave = 64;  // CDNA wavefront

// 4-bit codebook formats (kernel template FMT 1, weight = code[nibble] * fp32 block absmax, one fp32 multiply):
//   row 0 — bitsandbytes NF4 (LGA_FMT_NF4 = 1), get_4bit_type('nf4');
//   row 1 — bitsandbytes FP4 (LGA_FMT_FP4 = 3), get_4bit_type('fp4') = {0, .0625, 8, 12, 4, 6, 2, 3, -0, -.0625,
//           -8, -12, -4, -6, -2, -3} / 12: the sign-bit / 2-bit exponent / 1-bit mantissa code whose values
//           dDequantizeFP4Tree returns (bnb 0.41.0 csrc/kernels.cu, upstream; reference generate/base.py:105).
// Kernels take the row as a runtime index (`cb`), so FP4 shares every NF4 instantiation.
constexpr int kFmtFP4 = 3;
__host__ __device__ constexpr int codebook_of(int fmt) { return fmt == kFmtFP4 ? 1 : 0; }
__host__ __device__ constexpr int kernel_fmt(int fmt) { return fmt == kFmtFP4 ? 1 : fmt; }
static __constant__ float kCode4[2][16] = {
    {-1.0f, -0.6961928009986877f, -0.5250730514526367f, -0.39491748809814453f, -0.28444138169288635f,
     -0.18477343022823334f, -0.09105003625154495f, 0.0f, 0.07958029955625534f, 0.16093020141124725f,
     0.24611230194568634f, 0.33791524171829224f, 0.44070982933044434f, 0.5626170039176941f,
     0.7229568362236023f, 1.0f},
    {0.0f, 0.005208333333333333f, 0.6666666666666666f, 1.0f, 0.3333333333333333f, 0.5f, 0.16666666666666666f,
     0.25f, -0.0f, -0.005208333333333333f, -0.6666666666666666f, -1.0f, -0.3333333333333333f, -0.5f,
     -0.16666666666666666f, -0.25f}};

// ---- bf16 <-> f32 (bf16 stored as raw uint16_t; RNE on the way down, NaN kept a NaN) ----
__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float(((uint32_t)b) << 16); }
__device__ __forceinline__ float bflo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bfhi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }
// fp32 -> bf16 round-to-nearest-even in hardware (v_cvt_pk_bf16_f32: one instruction per PAIR, NaN stays NaN), by way of a vector that
// hipcc converts as one. Not in asm: hipcc keeps two wait states between an instruction that writes a matrix instruction's operand and
// that one, but not of an asm block, and the operand was then read as it was before.
typedef float lga_f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 lga_bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((lga_f32x2{lo, hi}), lga_bf16x2));
}
__device__ __forceinline__ uint16_t f2bf(float f) {
  return __builtin_bit_cast(unsigned short, static_cast<__bf16>(f));
}
__device__ __forceinline__ float round_bf(float f) { return bf2f(f2bf(f)); }

// Ahead of stores that stand under conditions of their own. Where a register that they use or write may be a load's for all that hipcc
// knows, on any way that leads there, it waits for everything in flight before each of them, the store before it included; behind a
// wait that it counts it knows better. (The wait is for earlier stores as well: not for between stores.)
__device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0F70); }
// The same for values of their own, whose loads then cannot move behind the wait
template <int N>
__device__ __forceinline__ void wait_loads(float (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(v[i]));
  wait_loads();
}

// ---- wave-level reductions (64 lanes) ----
// Every lane's value and its partner's, lane ^ D away, in either order; in registers, where a shuffle goes through LDS, whose latency
// a wave sum then has six times. All lanes of the wave take part. One-token steps, us by shuffles / here: pythia-160m fp32 303 / 291, 8
// sequences of the 2048-wide delta-rule model 545 / 532, one of the state-space one 286 / 277, Llama-2-7B int4 1288 / 1270.
struct LanePair {
  float a, b;
};
template <int CTRL, int BANKS = 0xf>
__device__ __forceinline__ float lane_dpp(float old, float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v), CTRL, 0xf, BANKS, false));
}
template <int D>
__device__ __forceinline__ LanePair lane_pair(float v) {
  static_assert(D == 32 || D == 16 || D == 8 || D == 4 || D == 2 || D == 1, "a power of two");
  if constexpr (D == 32) {
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return {__uint_as_float(h[0]), __uint_as_float(h[1])};
  } else if constexpr (D == 16) {
    const auto h = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return {__uint_as_float(h[0]), __uint_as_float(h[1])};
  } else if constexpr (D == 8) {
    return {v, lane_dpp<0x128>(v, v)};  // row_ror:8
  } else if constexpr (D == 4) {  // row_shl:4 in the even groups of four, row_shr:4 in the odd ones
    return {v, lane_dpp<0x114, 0xa>(lane_dpp<0x104, 0x5>(v, v), v)};
  } else {
    return {v, lane_dpp<D == 2 ? 0x4E : 0xB1>(v, v)};  // quad_perm
  }
}
// of two values at once: lanes with bit D clear get x's pair, the others y's
template <int D>
__device__ __forceinline__ LanePair lane_swap(float x, float y) {
  static_assert(D == 32 || D == 16, "whole rows of 16 lanes");
  if constexpr (D == 32) {
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return {__uint_as_float(h[0]), __uint_as_float(h[1])};
  } else {
    const auto h = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return {__uint_as_float(h[0]), __uint_as_float(h[1])};
  }
}
// f over aligned groups of W lanes, the partners W / 2, ..., 2, 1 away: the same bits as by shuffles (f is commutative)
template <int W, class F>
__device__ __forceinline__ float lanes_fold(float v, F&& f) {
  static_assert(W == 64 || W == 32 || W == 16 || W == 8 || W == 4 || W == 2, "a power of two");
  auto step = [&](LanePair p) { return f(p.a, p.b); };
  if constexpr (W >= 64) v = step(lane_pair<32>(v));
  if constexpr (W >= 32) v = step(lane_pair<16>(v));
  if constexpr (W >= 16) v = step(lane_pair<8>(v));
  if constexpr (W >= 16) v = f(v, lane_dpp<0x124>(v, v));  // (row_ror:4: lanes 8 apart are equal by now)
  else if constexpr (W >= 8) v = step(lane_pair<4>(v));
  if constexpr (W >= 4) v = step(lane_pair<2>(v));
  return step(lane_pair<1>(v));
}
// f over the lanes that share the bits below FROM, nearest first; f(a, b) of lanes without the bit: their own value, then the other's
template <int FROM, class F>
__device__ __forceinline__ float lanes_join(float v, F&& f) {
  auto step = [&](LanePair p) { return f(p.a, p.b); };
  if constexpr (FROM <= 1) v = step(lane_pair<1>(v));
  if constexpr (FROM <= 2) v = step(lane_pair<2>(v));
  if constexpr (FROM <= 4) v = step(lane_pair<4>(v));
  if constexpr (FROM <= 8) v = step(lane_pair<8>(v));
  if constexpr (FROM <= 16) v = step(lane_pair<16>(v));
  if constexpr (FROM <= 32) v = step(lane_pair<32>(v));
  return v;
}
template <int FROM>
__device__ __forceinline__ float lanes_join_sum(float v) {
  return lanes_join<FROM>(v, [](float a, float b) { return a + b; });
}
// the largest value of the wave and its place (the lowest among equals), in every lane
__device__ __forceinline__ void wave_best(float& v, int& i) {
  auto step = [&](LanePair p, LanePair q) {
    const int x = __float_as_int(q.a), y = __float_as_int(q.b);
    const bool second = p.b > p.a || (p.b == p.a && y < x);
    v = second ? p.b : p.a, i = second ? y : x;
  };
  step(lane_pair<32>(v), lane_pair<32>(__int_as_float(i)));
  step(lane_pair<16>(v), lane_pair<16>(__int_as_float(i)));
  step(lane_pair<8>(v), lane_pair<8>(__int_as_float(i)));
  step(lane_pair<4>(v), lane_pair<4>(__int_as_float(i)));
  step(lane_pair<2>(v), lane_pair<2>(__int_as_float(i)));
  step(lane_pair<1>(v), lane_pair<1>(__int_as_float(i)));
}
__device__ __forceinline__ float wave_sum(float v) {
  return lanes_fold<64>(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ float wave_max(float v) {
  return lanes_fold<64>(v, [](float a, float b) { return fmaxf(a, b); });
}
// sum over aligned groups of `W` lanes (W power of two <= 64)
template <int W>
__device__ __forceinline__ float group_sum(float v) {
  return lanes_fold<W>(v, [](float a, float b) { return a + b; });
}

// exact-order (no FMA contraction) helpers used where the reference's CPU math does mul then add. HIP's
// __fmul_rn / __fadd_rn are plain `a * b` / `a + b` (clang __clang_hip_math.h) and -ffp-contract may fuse them;
// the pragma drops the `contract` flag from these ops, which survives inlining.
__device__ __forceinline__ float mul_rn(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}
__device__ __forceinline__ float add_rn(float a, float b) {
#pragma clang fp contract(off)
  return a + b;
}

__device__ __forceinline__ float silu_f(float x) { return x / (1.0f + expf(-x)); }

// The runtime builds a kernel's device-side object at the kernel's first launch (about 0.5 ms each on ROCm 7.2,
// profiles/r03c_cold_prefill.txt); hipFuncGetAttributes builds it ahead of time. Each file lists the kernels of the
// prefill path it owns; lga_preload_kernels (capi.hip) runs them all at model load.
template <class F>
inline int preload(F* f) {
  hipFuncAttributes a;
  return hipFuncGetAttributes(&a, (const void*)f) == hipSuccess ? 0 : 1;
}
// compute units of the current device (cached; 256 if the query fails)
inline int num_cu() {
  static int n = 0;
  if (n == 0) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) !=
                                                 hipSuccess || n <= 0)
      n = 256;
  }
  return n;
}
int preload_gemm_q4f();
int preload_attention();
int preload_norm_rope();
int preload_sample();
int preload_gemv();
int preload_moe();

}  // namespace lga

// error plumbing shared by every C entry point
extern "C" void lga_set_error(const char* msg);

#define LGA_CHECK_ARG(cond, msg)    \
  do {                              \
    if (!(cond)) {                  \
      lga_set_error(msg);           \
      return (int)hipErrorInvalidValue; \
    }                               \
  } while (0)

#define LGA_LAUNCH_RETURN()                          \
  do {                                               \
    hipError_t e_ = hipGetLastError();               \
    if (e_ != hipSuccess) {                          \
      lga_set_error(hipGetErrorString(e_));          \
      return (int)e_;                                \
    }                                                \
    return 0;                                        \
  } while (0)
