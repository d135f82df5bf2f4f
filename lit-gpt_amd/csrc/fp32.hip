// fp32 forward path: the reference's `--precision 32-true` (generate/base.py:132, Fabric precision "32-true":
// weights and activations in float32). BASELINE config 1 is quoted in it (pythia-160m fp32, greedy 128 tokens);
// the bf16 kernels round every activation to bf16, which the fp32 fixture (tests/golden/g1) does not.
//
// A step of a 160M model is launches and their latency: what runs on one row is fused into three launches a block (both norms,
// the attention's input product and the MLP's with gelu; RoPE, cache append and attention; both output products with the
// residual adds), 38 a token.
// Per-op arithmetic is the reference's: fp32 products and sums, no bf16 rounding anywhere:
//   lga_f32_linear          F.linear (lit_gpt/model.py:619, 656, 699-702, 519): y = x W^T (+ b) (+ residual)
//   lga_f32_layernorm       torch.nn.LayerNorm (GPT-NeoX norm_class, config.py:137-144): two-pass mean / biased var
//                           (lga_f32_linear_act: with gelu and a second residual, lga_f32_layernorm_pair: two norms of a row)
//   lga_f32_norm_linears    one row's norms and the products that read them (the next two lines' numbers)
//   lga_f32_linears_sum     one row: two products and the residual adds of a parallel-residual block
//   lga_f32_gelu            F.gelu exact (erf) or tanh (GptNeoxMLP, model.py:699-702)
//   lga_f32_add             the Block's residual adds (model.py:584-593)
//   lga_f32_rope_kv_append  apply_rope (model.py:767-773, partial rotary) + KVCache.forward (:788-795)
//   lga_f32_attention       SDPA over the cache with the input_pos mask rows (model.py:651, 658-665)
//   lga_f32_attention_decode  the two above for one token in one launch
// (the token-embedding gather is lga_embedding over the fp32 rows as pairs of 16-bit words — a byte copy; greedy
// sampling is lga_argmax_f32 in sample.hip)
#include <type_traits>

#include "gemm_tiles.h"

namespace lga {

__device__ __forceinline__ float gelu_f32(float v, bool approximate_tanh) {
  if (approximate_tanh) {
    const float inner = 0.7978845608028654f * (v + 0.044715f * v * v * v);
    return 0.5f * v * (1.0f + tanhf(inner));
  }
  return 0.5f * v * (1.0f + erff(v * 0.7071067811865476f));
}

__device__ __forceinline__ void f32_fma4(const float4& x, const float4& w, float4& acc) {
  acc.x = fmaf(x.x, w.x, acc.x), acc.y = fmaf(x.y, w.y, acc.y), acc.z = fmaf(x.z, w.z, acc.z), acc.w = fmaf(x.w, w.w, acc.w);
}

// act: 0 none, 1 exact gelu, 2 tanh gelu, on the product + bias; then the residuals, one after the other
// one wave per output (m, n): lanes stride over K (16-B loads when K % 4 == 0), then a wave sum
__global__ void __launch_bounds__(256) f32_linear_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                         const float* __restrict__ b, int act,
                                                         const float* __restrict__ res, const float* __restrict__ res2,
                                                         float* __restrict__ y, int N, int K) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int n = blockIdx.x * 4 + wave, m = blockIdx.y;
  if (n >= N) return;
  const float* xr = x + (size_t)m * K;
  const float* wr = w + (size_t)n * K;
  float acc = 0.0f;
  if ((K & 3) == 0) {
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);  // (four sums of a lane are nearer to the exact one than one)
    for (int k = lane * 4; k < K; k += 256) f32_fma4(*(const float4*)(xr + k), *(const float4*)(wr + k), a);
    acc = (a.x + a.y) + (a.z + a.w);
  } else {
    for (int k = lane; k < K; k += 64) acc = fmaf(xr[k], wr[k], acc);
  }
  acc = wave_sum(acc);
  if (lane == 0) {
    if (b) acc += b[n];
    if (act) acc = gelu_f32(acc, act == 2);
    if (res) acc += res[(size_t)m * N + n];
    if (res2) acc += res2[(size_t)m * N + n];
    y[(size_t)m * N + n] = acc;
  }
}

// Prompts of other K % 4 == 0: the same sums for eight rows and two outputs a wave. A wave per output read the matrix once a row from L2 and
// a kilobyte of x for every four products of its lanes; here ten loads stand beside 64. Lane 2 r + o finishes row r of output o.
// us, a wave per output / here: 300 rows of 3072 x 768 204 / 92, of 768 x 3072 158 / 90, 40 rows 30 / 18, 26 / 17
__global__ void __launch_bounds__(256) f32_linear_rows_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                              const float* __restrict__ b, int act,
                                                              const float* __restrict__ res, const float* __restrict__ res2,
                                                              float* __restrict__ y, int M, int N, int K) {
  constexpr int R = 8, O = 2;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int n0 = (blockIdx.x * 4 + wave) * O, m0 = blockIdx.y * R;
  if (n0 >= N) return;
  const float* wr[O];
  const float* xr[R];
#pragma unroll
  for (int o = 0; o < O; ++o) wr[o] = w + (size_t)min(n0 + o, N - 1) * K;
#pragma unroll
  for (int r = 0; r < R; ++r) xr[r] = x + (size_t)min(m0 + r, M - 1) * K;  // (rows past the end repeat the last one, never stored)
  float4 a[R][O];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int o = 0; o < O; ++o) a[r][o] = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int k = lane * 4; k < K; k += 256) {
    float4 wv[O], xv[R];
#pragma unroll
    for (int o = 0; o < O; ++o) wv[o] = *(const float4*)(wr[o] + k);
#pragma unroll
    for (int r = 0; r < R; ++r) xv[r] = *(const float4*)(xr[r] + k);
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int o = 0; o < O; ++o) f32_fma4(xv[r], wv[o], a[r][o]);
  }
  float acc = 0.0f;
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int o = 0; o < O; ++o) {
      const float s = wave_sum((a[r][o].x + a[r][o].y) + (a[r][o].z + a[r][o].w));
      if (lane == r * O + o) acc = s;
    }
  const int m = m0 + lane / O, n = n0 + lane % O;
  if (lane >= R * O || m >= M || n >= N) return;
  if (b) acc += b[n];
  if (act) acc = gelu_f32(acc, act == 2);
  if (res) acc += res[(size_t)m * N + n];
  if (res2) acc += res2[(size_t)m * N + n];
  y[(size_t)m * N + n] = acc;
}

typedef float f32x32_t __attribute__((ext_vector_type(32)));
typedef float f32q_t __attribute__((ext_vector_type(4)));

// Prompts of K % 256 == 0, two rows and more: the same sums once more, on the fp32 matrix cores. f32_linear_kernel's sum is 256 chains
// (k modulo 256) and a tree over them; a matrix instruction of one k (32x32x1, 16x16x1: 2 or 4 products' blocks side by side)
// extends one chain of T x T outputs by an fma, so the blocks take the chains that the tree joins first, the four values of a lane's 16
// bytes four accumulators, and a wave the chains of one 16-byte chunk of every 128-byte line: its part of the tree lies in its own
// registers, and the last three levels join the eight waves. Rounding, denormals and infinities are fmaf's: the bits of one row alone.
// A step is 16 KB of x and W by LDS-DMA (whole lines, chunks source-swizzled so that 16 lanes of a fragment read all banks), four on
// their way, and four instructions a wave. The fragments are read as vectors of the compiler's own: reads of HIP's float4 may alias the
// DMAs for it, and it waits for all of them before each (T 32: 300 x 768 x 3072 26.5 us so, 20.6 as it is).
// Bound by the matrix cores (a step without its DMAs takes 0.9 of the time, without its instructions 0.55) and the tree's 256 adds an
// output; at few rows by one workgroup's chain of steps. us, f32_linear_kernel or f32_linear_rows_kernel / here: 300 rows of 3072 x 768 88 / 31, of
// 768 x 3072 89 / 21, of 768 x 768 25 / 9.0; 40 rows 16.8 / 9.0, 15.9 / 8.7, 7.6 / 4.6; 16 rows 9.7 / 4.9, 14.3 / 8.3, 5.4 / 4.6; 16 of 50304
// x 768 100 / 42; 8 of 4096 x 1024 10.9 / 6.3.
template <int T, int RING>
__global__ void __launch_bounds__(512, T == 32 ? 2 : 4) f32_linear_tiles_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                 const float* __restrict__ b, int act,
                                                                 const float* __restrict__ res, const float* __restrict__ res2,
                                                                 float* __restrict__ y, int M, int N, int K) {
  constexpr int BLK = 64 / T, SETS = 8 / BLK, REG = T * T / 64, STEP = 16384;
  using Acc = std::conditional_t<T == 32, f32x32_t, f32x16_t>;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[RING * STEP];
  static_assert(RING >= 3 && T * T * 32 <= RING * STEP, "one step in use, others on their way; the waves' sums in their place");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tm = (M + T - 1) / T, tn = (N + T - 1) / T, per = (tm * tn + 7) / 8;
  const int at = (blockIdx.x % 8) * per + blockIdx.x / 8;  // (an XCD's workgroups: neighbouring columns, all rows)
  if (at >= tm * tn) return;
  const int m0 = at % tm * T, n0 = at / tm * T;
  const unsigned char* src[2];
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const int q = (wave * 2 + d) * 8 + (lane >> 3), blk = q / (2 * T), r = q % (2 * T), line = T == 32 ? 4 * blk : 4 * (blk & 1) + 2 * (blk >> 1);
    const float* row = r < T ? x + (size_t)min(m0 + r, M - 1) * K : w + (size_t)min(n0 + r - T, N - 1) * K;
    src[d] = (const unsigned char*)row + 128 * line + 16 * ((lane & 7) ^ ((q >> 1) & 7));
  }
  const int n = K / 256, last = SETS * n - 1;
  int set = 0, i = 0;  // of the next step to fetch (past the last: that one again, never used)
  auto dma = [&](int buffer) {
    const int at = 128 * (T == 32 ? (set & 1) * 2 + (set >> 1) : set) + 1024 * i;
#pragma unroll
    for (int d = 0; d < 2; ++d) gemm_dma16(src[d] + at, lds + buffer * STEP + (wave * 2 + d) * 1024);
    if (set * n + i < last && ++i == n) i = 0, ++set;
  };
  const int row = lane % T, chunk = 16 * (wave ^ ((row >> 1) & 7));
  const int a_at = (lane / T * 2 * T + row) * 128 + chunk, b_at = a_at + T * 128;
#pragma unroll
  for (int s = 0; s < RING; ++s) dma(s);
  gemm_wait_vm<2 * (RING - 1)>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  f32q_t a = *(const f32q_t*)(lds + a_at), c = *(const f32q_t*)(lds + b_at);
  int buffer = 0;
  float t[2][REG];
#pragma unroll
  for (int s = 0; s < SETS; ++s) {
    Acc acc[4];
    auto step = [&](auto first) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this step's values are in registers, its buffer is free, ...
      gemm_wait_vm<2 * (RING - 2)>();                      // ... and the next step's have landed
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      const int freed = buffer;
      buffer = buffer + 1 == RING ? 0 : buffer + 1;
      const f32q_t a1 = *(const f32q_t*)(lds + buffer * STEP + a_at), c1 = *(const f32q_t*)(lds + buffer * STEP + b_at);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (T == 32) acc[e] = __builtin_amdgcn_mfma_f32_32x32x1f32(a[e], c[e], first ? Acc(0.0f) : acc[e], 0, 0, 0);
        else acc[e] = __builtin_amdgcn_mfma_f32_16x16x1f32(a[e], c[e], first ? Acc(0.0f) : acc[e], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (e == 0) dma(freed);
        __builtin_amdgcn_sched_barrier(0);
      }
      a = a1, c = c1;
    };
    step(std::true_type{});
#pragma nounroll
    for (int k = 1; k < n; ++k) step(std::false_type{});
#pragma unroll
    for (int r = 0; r < REG; ++r) {
      float v[BLK];
#pragma unroll
      for (int k = 0; k < BLK; ++k) v[k] = (acc[0][k * REG + r] + acc[1][k * REG + r]) + (acc[2][k * REG + r] + acc[3][k * REG + r]);
      float sum = v[0] + v[1];
      if constexpr (BLK == 4) sum += v[2] + v[3];
      if constexpr (T == 32) t[s >> 1][r] = s & 1 ? t[s >> 1][r] + sum : sum;
      else t[s][r] = sum;
      asm volatile("" : "+v"(t[T == 32 ? s >> 1 : s][r]));  // (or the sums sink to the end and every set's products stay in registers)
    }
  }
  gemm_wait_vm<0>();  // no DMA may outlive its buffer
  __syncthreads();
  float* part = (float*)lds;
#pragma unroll
  for (int r = 0; r < REG; ++r) part[(wave * T + (T == 32 ? 8 * (r / 4) : 0) + lane / T * 4 + r % 4) * T + row] = t[0][r] + t[1][r];
  __syncthreads();
#pragma unroll
  for (int e = tid; e < T * T; e += 512) {
    float p[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) p[k] = part[k * T * T + e];
    float v = ((p[0] + p[4]) + (p[2] + p[6])) + ((p[1] + p[5]) + (p[3] + p[7]));
    const int m = m0 + e / T, o = n0 + e % T;
    if (m >= M || o >= N) continue;
    if (b) v += b[o];
    if (act) v = gelu_f32(v, act == 2);
    if (res) v += res[(size_t)m * N + o];
    if (res2) v += res2[(size_t)m * N + o];
    y[(size_t)m * N + o] = v;
  }
}

// From eight rows and some eight waves a CU on, where few of the rows computed are repeated ones or the chip is full several times
// over. us, a wave per output / here: 8 rows of 4096 x 768 9.3 / 8.3, of 3072 x 768 (1536 waves) 7.6 / 7.9, of 3072 x 3072 21.1 / 23.6; 9
// rows of 2304 x 256 4.4 / 6.4, of 4096 x 768 10.5 / 11.5, of 8192 x 768 21.1 / 19.1; 12 rows of 2304 x 768 8.2 / 9.2, of 3072 x 768
// 10.0 / 9.6; 16 rows of 2304 x 768 10.0 / 9.2; 17 of 4096 x 768 17.2 / 14.6, of 2304 x 256 6.5 / 7.5
static bool f32_linear_in_rows(int M, int N, int K) {
  const long live = (long)M * N / 16, padded = (long)((N + 1) / 2) * ((M + 7) / 8);  // waves' worth of rows, and waves
  return K % 4 == 0 && M >= 8 && live >= 2000 && (live * 10 >= padded * 7 || live >= 4500);
}

template <int T>
static long f32_tiles(int M, int N) { return (long)((M + T - 1) / T) * ((N + T - 1) / T); }
// Whether the matrix cores serve: from some 9000 outputs on they do at every K, below a wave per output ends sooner. us, a wave per output /
// T 16: 8 x 1024 x 256 3.0 / 3.3, 9 rows 3.3 / 3.2; 5 x 1536 x 512 3.6 / 4.1, 6 rows 4.2 / 4.1; 3 x 2304 x 768 4.0 / 4.7, 4 rows 4.9 / 4.7; 3 x
// 3072 x 768 5.0 / 4.9; 8 x 1024 x 4096 11.7 / 11.0; 4 x 2048 x 8192 19.5 / 18.2; 2 x 50304 x 768 44 / 36.
// (2^23 workgroups of 512: as many work-items as a launch holds)
static bool f32_linear_in_tiles(int M, int N, int K) {
  return K % 256 == 0 && M > 1 && (long)M * N >= 9000 && f32_tiles<16>(M, N) < (1 << 23) - 8;
}
// Tiles of 16 x 16 (two workgroups a CU) or of 32 x 32 (one, four times the outputs in 1.7 times the time): by rounds of the chip, and 16
// where one of those tiles a CU is enough. us of 16 / 32: 40 x 768 x 3072 8.8 / 20.4, 64 x 3072 x 768 9.0 / 9.2, 96 x 3072 x 768 12.8 / 16.1,
// 300 x 3072 x 768 32.4 / 30.5, 300 x 768 x 3072 25.7 / 20.6, 64 x 4096 x 1024 14.8 / 11.6.
static bool f32_tiles_of_16(int M, int N) {
  const long t16 = f32_tiles<16>(M, N), t32 = f32_tiles<32>(M, N);
  return t16 <= 256 || (t16 + 511) / 512 * 3 <= (t32 + 255) / 256 * 5;
}
template <int T>
static void f32_linear_tiles(const float* x, const float* w, const float* bias, int act, const float* residual, const float* residual2, float* y,
                             int M, int N, int K, hipStream_t stream) {
  const unsigned blocks = 8 * (unsigned)((f32_tiles<T>(M, N) + 7) / 8);
  f32_linear_tiles_kernel<T, 4><<<blocks, 512, 0, stream>>>(x, w, bias, act, residual, residual2, y, M, N, K);
}

// Mean and biased variance of a row by a workgroup of 256, the first 256 CPT columns left in r
template <int CPT>
__device__ __forceinline__ void f32_row_stats(const float* __restrict__ xr, int n, float (&r)[CPT], float (&red)[4],
                                              float& mean, float& var) {
  const int at = threadIdx.x;
  float s = 0.0f;
#pragma unroll
  for (int e = 0; e < CPT; ++e) {
    const int i = at + 256 * e;
    r[e] = i < n ? xr[i] : 0.0f;
  }
#pragma unroll
  for (int e = 0; e < CPT; ++e) s += r[e];
  for (int i = at + 256 * CPT; i < n; i += 256) s += xr[i];
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  mean = ((red[0] + red[1]) + (red[2] + red[3])) / (float)n;
  __syncthreads();
  float ss = 0.0f;
#pragma unroll
  for (int e = 0; e < CPT; ++e) {
    const float d = at + 256 * e < n ? r[e] - mean : 0.0f;
    ss = fmaf(d, d, ss);
  }
  for (int i = at + 256 * CPT; i < n; i += 256) {
    const float d = xr[i] - mean;
    ss = fmaf(d, d, ss);
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  var = ((red[0] + red[1]) + (red[2] + red[3])) / (float)n;
}
__device__ __forceinline__ float f32_normed(float v, float mean, float rstd, float w, bool biased, float b) {
  const float o = mul_rn(mul_rn(v - mean, rstd), w);
  return biased ? add_rn(o, b) : o;
}

// two norms of one row where w2 is given (a block whose attention and MLP read the same residual): the row stays in
// registers (up to 256 CPT columns), mean and variance are made once per eps
template <int CPT>
__global__ void __launch_bounds__(256) f32_layernorm_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                            const float* __restrict__ b, float* __restrict__ y, int n,
                                                            float eps, const float* __restrict__ w2,
                                                            const float* __restrict__ b2, float* __restrict__ y2, float eps2) {
  const size_t row = blockIdx.x;
  const float* xr = x + row * n;
  __shared__ float red[4];
  float r[CPT];
  float mean, var;
  f32_row_stats<CPT>(xr, n, r, red, mean, var);
  auto put = [&](const float* w_, const float* b_, float rstd, float* y_, int i, float v) {
    y_[row * n + i] = f32_normed(v, mean, rstd, w_[i], b_, b_ ? b_[i] : 0.0f);
  };
  const float rstd = 1.0f / sqrtf(var + eps), rstd2 = w2 ? 1.0f / sqrtf(var + eps2) : 0.0f;
#pragma unroll
  for (int e = 0; e < CPT; ++e) {
    const int i = threadIdx.x + 256 * e;
    if (i < n) {
      put(w, b, rstd, y, i, r[e]);
      if (w2) put(w2, b2, rstd2, y2, i, r[e]);
    }
  }
  for (int i = threadIdx.x + 256 * CPT; i < n; i += 256) {
    put(w, b, rstd, y, i, xr[i]);
    if (w2) put(w2, b2, rstd2, y2, i, xr[i]);
  }
}

// One row, K a multiple of 4: up to two products of a norm of the row each (f32_linear_kernel of f32_layernorm_kernel's row, to
// the bit). A workgroup makes its norm anew, in LDS, a wave then one output after the other. The first weights are loaded ahead of the
// row, and loads return in order: the statistics wait for both, the sums for nothing more. pythia-160m (768 -> 2304 and 3072):
// norms and products in three launches 16.2 us, in this one 7.0. With a norm of each wave's own in registers, and no barrier, 8.1: four times
// the loads of the row and its weights (weights from memory, LDS / registers: 512 -> 8192 6.9 / 8.8, 1024 -> 3072 and 4096 8.8 / 10.1, 256 ->
// 50304 14.0 / 19.7; a token behind 300 keys of pythia-160m 268 / 279, of pythia-410m 582 / 613).
struct F32NormLinear {
  const float *nw, *nb;
  float eps;
  const float *w, *b;
  int act;
  float* y;
  int N, blocks;
};
struct F32NormLinears {
  const float* x;
  int K;
  F32NormLinear p[2];
};
constexpr int kF32Chunks = 4;  // 256 columns each: a wave's loads in flight
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef f32x4_t f32x4_any_t __attribute__((aligned(4)));
typedef float f32x2_any_t __attribute__((ext_vector_type(2), aligned(4)));
// 16 bytes of a row, or of a vector, whose address (of any float) is the same for the wave; k: a lane's columns, those past the last four
// are theirs
__device__ __forceinline__ f32x4_t f32_load4(const float* row, int k, int K) {
  return *(const f32x4_any_t*)((const char*)row + (unsigned)min(k, K - 4) * 4u);
}
__device__ __forceinline__ void f32_load_chunks(const float* row, int c0, int K, int lane, f32x4_t (&v)[kF32Chunks]) {
#pragma unroll
  for (int c = 0; c < kF32Chunks; ++c)
    if ((c0 + c) * 256 < K) v[c] = f32_load4(row, (c0 + c) * 256 + lane * 4, K);
}
__device__ __forceinline__ void f32_fma4(const f32x4_t& x, const f32x4_t& w, f32x4_t& acc) {
  acc.x = fmaf(x.x, w.x, acc.x), acc.y = fmaf(x.y, w.y, acc.y), acc.z = fmaf(x.z, w.z, acc.z), acc.w = fmaf(x.w, w.w, acc.w);
}
__device__ __forceinline__ void f32_dot_chunks(const float* xr, int c0, int K, int lane, const f32x4_t (&w)[kF32Chunks], f32x4_t& acc) {
#pragma unroll
  for (int c = 0; c < kF32Chunks; ++c) {
    const int k = (c0 + c) * 256 + lane * 4;
    if (k < K) f32_fma4(*(const f32x4_t*)(xr + k), w[c], acc);
  }
}
__device__ __forceinline__ float f32_dot_end(const f32x4_t& a) { return wave_sum((a.x + a.y) + (a.z + a.w)); }
template <int CPT>
__global__ void __launch_bounds__(256) f32_norm_linears_kernel(F32NormLinears a) {
  extern __shared__ __attribute__((aligned(16))) float xn[];  // [K]
  __shared__ float red[4];
  const bool second = (int)blockIdx.x >= a.p[0].blocks;
  const F32NormLinear p = second ? a.p[1] : a.p[0];
  const int block = (int)blockIdx.x - (second ? a.p[0].blocks : 0), K = a.K;
  const float* x = a.x;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  int n = block * 4 + wave;
  f32x4_t w[kF32Chunks];
  if (n < p.N) f32_load_chunks(p.w + (size_t)n * K, 0, K, lane, w);
  float bias = n < p.N && p.b ? p.b[n] : 0.0f;
  const int at = threadIdx.x;
  float r[CPT], nw[CPT], nb[CPT], mean, var;
#pragma unroll
  for (int e = 0; e < CPT; ++e) {
    const int i = at + 256 * e;
    nw[e] = i < K ? p.nw[i] : 0.0f;
    nb[e] = i < K && p.nb ? p.nb[i] : 0.0f;
  }
  f32_row_stats<CPT>(x, K, r, red, mean, var);
  const float rstd = 1.0f / sqrtf(var + p.eps);
#pragma unroll
  for (int e = 0; e < CPT; ++e) {
    const int i = at + 256 * e;
    if (i < K) xn[i] = f32_normed(r[e], mean, rstd, nw[e], p.nb, nb[e]);
  }
  for (int i = at + 256 * CPT; i < K; i += 256) xn[i] = f32_normed(x[i], mean, rstd, p.nw[i], p.nb, p.nb ? p.nb[i] : 0.0f);
  __syncthreads();
  for (const int step = p.blocks * 4; n < p.N; n += step) {
    f32x4_t a4 = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int c0 = 0; c0 * 256 < K; c0 += kF32Chunks) {
      f32_dot_chunks(xn, c0, K, lane, w, a4);
      const bool more = (c0 + kF32Chunks) * 256 < K;
      if (more || n + step < p.N) f32_load_chunks(p.w + (size_t)(more ? n : n + step) * K, more ? c0 + kF32Chunks : 0, K, lane, w);
    }
    float acc = f32_dot_end(a4);
    if (lane == 0) {
      if (p.b) acc += bias;
      if (p.act) acc = gelu_f32(acc, p.act == 2);
      p.y[n] = acc;
    }
    bias = n + step < p.N && p.b ? p.b[n + step] : 0.0f;
  }
}

// One row: y = ((x2 W2^T + b2) + (x1 W1^T + b1)) + res, a wave per output, both products in f32_linear_kernel's order. Bound by
// latency: the weights of a block of 768 columns beside 3072 are in flight at once. E2 > 0: x2 (of up to 1024 E2 values) and an
// attention's ranges come ahead of the weights, so that the join waits for nothing else, and x2 is read once for a workgroup's four
// outputs (kept in registers until LDS has them: as an array of HIP's float4 they went through scratch memory, a trip of their own
// ahead of all weights). Weights from memory, an attention in five ranges, us without / with: 768 columns beside 3072 9.4 / 9.5, 1024
// beside 4096 10.2 / 9.6, 1600 beside 6400 24.2 / 18.1, 2048 beside 8192 30.0 / 24.3, in one range 23.3 / 18.2; a token behind 300 keys:
// pythia-160m 292 / 267, pythia-410m 652 / 581, pythia-1b 1109 / 1013. Not where x1 is longer than half of x2: 4096 beside 4096 in
// five ranges 47.8 / 66.4, 2240 beside 1280 9.8 / 10.3.
struct F32LinearsSum {
  const float *x1, *w1, *b1, *x2, *w2, *b2, *res;
  float* y;
  int N, K1, K2;
  // parts > 1: x1 is [parts][K1], an attention's sums over ranges of its keys, ml [parts][K1 / hs][2] (f32_attention_vec_kernel)
  const float* ml;
  int parts, hs;
};
// x1 of ranges of keys, joined in LDS: the ranges' sums weighted by exp(their largest score - the largest of all)
struct F32Parts {
  static constexpr int E = 4, P = 8;
  float o[E][P], m[P], l[P];  // (of the thread's first columns, and of head threadIdx.x)
};
__device__ __forceinline__ void f32_load_parts(const F32LinearsSum& a, F32Parts& p) {
  const int H = a.K1 / a.hs;
  const unsigned h = (unsigned)min((int)threadIdx.x, H - 1) * 8u;
  unsigned at[F32Parts::E];  // (columns past the last one are its)
#pragma unroll
  for (int e = 0; e < F32Parts::E; ++e) at[e] = (unsigned)min((int)threadIdx.x + 256 * e, a.K1 - 1) * 4u;
#pragma unroll
  for (int s = 0; s < F32Parts::P; ++s) {
    p.m[s] = -INFINITY, p.l[s] = -1.0f;
    if (s >= a.parts) continue;
    const f32x2_any_t ml = *(const f32x2_any_t*)((const char*)(a.ml + (size_t)s * H * 2) + h);
    p.m[s] = ml.x, p.l[s] = ml.y;
#pragma unroll
    for (int e = 0; e < F32Parts::E; ++e) p.o[e][s] = *(const float*)((const char*)(a.x1 + (size_t)s * a.K1) + at[e]);
  }
}
__device__ __forceinline__ void f32_join_parts(const F32LinearsSum& a, const F32Parts& p, float* xs, float* wt) {
  constexpr int E = F32Parts::E, P = F32Parts::P;
  const int H = a.K1 / a.hs;
  if ((int)threadIdx.x < H) {  // (up to 256 heads)
    const int h = threadIdx.x;
    float most = -INFINITY, sum = 0.0f;
#pragma unroll
    for (int s = 0; s < P; ++s) most = fmaxf(most, p.m[s]);
#pragma unroll
    for (int s = 0; s < P; ++s) {
      const bool empty = p.l[s] < 0.0f;
      const float w = empty ? -1.0f : (p.m[s] == -INFINITY ? 0.0f : expf(p.m[s] - most));
      if (!empty) sum = fmaf(w, p.l[s], sum);
      wt[h * (P + 1) + s] = w;
    }
    wt[h * (P + 1) + P] = sum;
  }
  __syncthreads();
  auto join = [&](int i, auto&& at) {
    const float* w = wt + i / a.hs * (P + 1);
    float acc = 0.0f;
#pragma unroll
    for (int s = 0; s < P; ++s)
      if (!(w[s] < 0.0f)) acc = fmaf(w[s], at(s), acc);
    xs[i] = acc / w[P];
  };
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = threadIdx.x + 256 * e;
    if (i < a.K1) join(i, [&](int s) { return p.o[e][s]; });
  }
  for (int i = threadIdx.x + 256 * E; i < a.K1; i += 256) join(i, [&](int s) { return a.x1[(size_t)s * a.K1 + i]; });
  __syncthreads();
}
template <bool PARTS, int E2>
__global__ void __launch_bounds__(256) f32_linears_sum_kernel(F32LinearsSum a) {
  extern __shared__ __attribute__((aligned(16))) float xs[];  // [K1] the joined row, then the ranges' weights; or [K1]; x2
  const int lane = threadIdx.x & 63, row = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = min(row, a.N - 1);
  const float *r1 = a.w1 + (size_t)n * a.K1, *r2 = a.w2 + (size_t)n * a.K2;
  constexpr bool AHEAD = E2 > 0;
  f32x4_t x2[E2 > 0 ? E2 : 1];
#pragma unroll
  for (int e = 0; e < E2; ++e) x2[e] = f32_load4(a.x2, (threadIdx.x + 256 * e) * 4, a.K2);
  F32Parts parts;
  if (PARTS && AHEAD) f32_load_parts(a, parts);
  __builtin_amdgcn_sched_barrier(0);
  f32x4_t w1[kF32Chunks], w2[3][kF32Chunks];
  f32_load_chunks(r1, 0, a.K1, lane, w1);
#pragma unroll
  for (int u = 0; u < 3; ++u) f32_load_chunks(r2, u * kF32Chunks, a.K2, lane, w2[u]);
  const float b1 = a.b1 ? a.b1[n] : 0.0f, b2 = a.b2 ? a.b2[n] : 0.0f, res = a.res[n];
  __builtin_amdgcn_sched_barrier(0);
  if (PARTS && !AHEAD) f32_load_parts(a, parts);
  const float *px1 = a.x1, *px2 = a.x2;
  if (AHEAD) {
    float* to = xs + (PARTS ? a.K1 + (a.K1 / a.hs * 9 + 3) / 4 * 4 : 0);
#pragma unroll
    for (int e = 0; e < E2; ++e) {
      const int k = (threadIdx.x + 256 * e) * 4;
      if (k < a.K2) *(f32x4_t*)(to + k) = x2[e];
    }
    px2 = to;
  }
  if (PARTS) {
    f32_join_parts(a, parts, xs, xs + a.K1);
    px1 = xs;
  } else if (AHEAD) {
    __syncthreads();
  }
  f32x4_t h4 = {0.0f, 0.0f, 0.0f, 0.0f}, m4 = h4;
  for (int c0 = 0; c0 * 256 < a.K1; c0 += kF32Chunks) {
    if (c0 > 0) f32_load_chunks(r1, c0, a.K1, lane, w1);
    f32_dot_chunks(px1, c0, a.K1, lane, w1, h4);
  }
  for (int c0 = 0; c0 * 256 < a.K2; c0 += 3 * kF32Chunks) {
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      if (c0 > 0) f32_load_chunks(r2, c0 + u * kF32Chunks, a.K2, lane, w2[u]);
    }
#pragma unroll
    for (int u = 0; u < 3; ++u) f32_dot_chunks(px2, c0 + u * kF32Chunks, a.K2, lane, w2[u], m4);
  }
  float h = f32_dot_end(h4), m = f32_dot_end(m4);
  if (lane == 0 && row < a.N) {
    if (a.b1) h += b1;
    if (a.b2) m += b2;
    m += h;
    a.y[n] = m + res;
  }
}

static void f32_layernorm_go(const float* x, const float* w, const float* b, float* y, const float* w2, const float* b2,
                             float* y2, int rows, int n, float eps, float eps2, hipStream_t stream) {
  if (n <= 256) f32_layernorm_kernel<1><<<rows, 256, 0, stream>>>(x, w, b, y, n, eps, w2, b2, y2, eps2);
  else if (n <= 1024) f32_layernorm_kernel<4><<<rows, 256, 0, stream>>>(x, w, b, y, n, eps, w2, b2, y2, eps2);
  else f32_layernorm_kernel<16><<<rows, 256, 0, stream>>>(x, w, b, y, n, eps, w2, b2, y2, eps2);
}

__global__ void __launch_bounds__(256) f32_gelu_kernel(const float* __restrict__ a, float* __restrict__ y, size_t n,
                                                       int approximate_tanh) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    y[i] = gelu_f32(a[i], approximate_tanh != 0);
  }
}

__global__ void __launch_bounds__(256) f32_add_kernel(const float* __restrict__ a, const float* __restrict__ b,
                                                      float* __restrict__ y, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) y[i] = a[i] + b[i];
}

// grid (T, G): the q heads, k and v of query group g for token t (qkv row layout per group [q_0..q_{qpk-1}, k, v],
// scripts/convert_hf_checkpoint.py:174-188); x * cos + rotate_half(x) * sin on the first n_elem dims, two roundings
__global__ void __launch_bounds__(256) f32_rope_kv_kernel(const float* __restrict__ qkv, float* __restrict__ q_out,
                                                          float* __restrict__ k_cache, float* __restrict__ v_cache,
                                                          const int64_t* __restrict__ cache_pos,
                                                          const int64_t* __restrict__ rope_pos,
                                                          const float* __restrict__ cos, const float* __restrict__ sin,
                                                          int n_head, int n_groups, int hs, int n_elem, int max_seq,
                                                          int rope_rows) {
  const int t = blockIdx.x, g = blockIdx.y;
  const int qpk = n_head / n_groups;
  const long p = cache_pos[t];
  const long rp = rope_pos[t];
  if (p < 0 || p >= max_seq || rp < 0 || rp >= rope_rows) return;  // host validates; never go out of bounds
  const float* src = qkv + ((size_t)t * (n_head + 2 * n_groups) + (size_t)g * (qpk + 2)) * hs;
  const float* cr = cos + (size_t)rp * n_elem;
  const float* sr = sin + (size_t)rp * n_elem;
  const int half = n_elem / 2;
  for (int it = threadIdx.x; it < (qpk + 2) * hs; it += blockDim.x) {
    const int slot = it / hs, d = it % hs;
    const float* xs = src + (size_t)slot * hs;
    float out = xs[d];
    if (slot <= qpk && d < n_elem) {
      const float r = d < half ? -xs[d + half] : xs[d - half];
      out = add_rn(mul_rn(xs[d], cr[d]), mul_rn(r, sr[d]));
    }
    if (slot < qpk) q_out[((size_t)t * n_head + (size_t)g * qpk + slot) * hs + d] = out;
    else if (slot == qpk) k_cache[((size_t)g * max_seq + p) * hs + d] = out;
    else v_cache[((size_t)g * max_seq + p) * hs + d] = out;
  }
}

struct F32AttnArgs {
  const float* q;  // [T][H][hs] roped; fused: the token's projection, per group [q_0 .. q_{qpk-1}, k, v]
  float *kc, *vc;  // [G][max_seq][hs] (written by the fused form only)
  const int64_t* pos;
  float* y;
  int H, G, hs, max_seq;
  float scale;
  const int64_t* rope_pos;  // fused only
  const float *cos, *sin;
  int n_elem, rope_rows;
  int parts;  // ranges of the keys (fused only), beyond one:
  float* ml;  // [parts][H][2] the largest score and the sum of the weights; y holds [parts][H * hs] sums of weighted values
};

// Keys of a range, whole steps of the 32 keys of the narrowest rows: 64 at least, so that with lga_f32_attention_parts' number of
// ranges they follow from the keys alone, and a token's bits not from the size of its cache
__host__ __device__ inline int f32_attention_chunk(int keys, int parts) {
  const int chunk = ((keys + parts - 1) / parts + 31) / 32 * 32;
  return chunk < 64 ? 64 : chunk;
}

// grid (T, H): softmax(q . K^T * scale) . V over keys 0..pos[t] of the query's group; scores kept in LDS, exact max, fp32
// exp and sums. LPK adjacent lanes hold a key's or value's row in pieces of four (hs <= 4 LPK), the other lanes of the 8
// waves other keys, four rows of each in flight. FUSED (one token): RoPE on q and on the group's k, which go with v to the
// caches at position pos[0] and into LDS, in the same launch. Latency-bound at decode sizes (300 keys of 64 per head are
// 150 KB): one key per wave at a time took 80 us, this form 9 beside the rotation and the append. A workgroup's loads bring some
// 20 GB/s, so that the fused form takes the keys in ranges side by side (grid (parts, H)), whose sums f32_linears_sum_kernel
// joins; pythia-160m at 301 keys 12.2 us in one range, 7.7 in five, 6.8 with its
// first rows loaded beside q and the angles.
template <int LPK, bool FUSED>
__global__ void __launch_bounds__(512) f32_attention_vec_kernel(F32AttnArgs a) {
  extern __shared__ float sc[];  // [max_seq] scores, then [8][hs] partial sums
  __shared__ float red[8];
  __shared__ __attribute__((aligned(16))) float qs[256], ks[256], vs[256];
  constexpr int KPW = 64 / LPK, STEP = 8 * KPW;
  const int t = FUSED ? 0 : blockIdx.x, range = FUSED ? blockIdx.x : 0, h = blockIdx.y, qpk = a.H / a.G, g = h / qpk, hs = a.hs;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, sub = lane % LPK, first = wave * KPW + lane / LPK;
  const long p = a.pos[t];
  float* kb = a.kc + (size_t)g * a.max_seq * hs;
  float* vb = a.vc + (size_t)g * a.max_seq * hs;
  const int L = (int)min(max(p + 1, 1L), (long)a.max_seq);
  // this workgroup's keys, of as many ranges as there are keys for
  const int chunk = FUSED && a.parts > 1 ? f32_attention_chunk(L, a.parts) : L, lo = range * chunk, hi = min(lo + chunk, L);
  const bool mine = sub * 4 < hs;
  // (the last columns again for a lane past them, its values cleared: a choice of addresses, one of them a constant's, makes the compiler load
  // through the generic aperture, in two pieces; pythia-160m at 301 keys 6.7 us so, 5.3 as it is)
  const int at = mine ? sub * 4 : hs - 4;
  auto kept = [&](float4 v) { return make_float4(mine ? v.x : 0.0f, mine ? v.y : 0.0f, mine ? v.z : 0.0f, mine ? v.w : 0.0f); };
  auto row = [&](const float* base, int j) { return kept(*(const float4*)(base + (size_t)min(j, L - 1) * hs + at)); };
  // the token's q, k, v and angles, and behind them the first keys and values (of a fused range all of them), on their way
  // together. (The fused form's own row is read here before it is written, and not used.)
  float4 k[4], v[4];
  float x[5], cs = 1.0f, sn = 0.0f;
  const int d0 = min((int)threadIdx.x, hs - 1), half = a.n_elem / 2, d1 = d0 < half ? d0 + half : d0 < a.n_elem ? d0 - half : d0;
  if (FUSED) {
    const long rp = a.rope_pos[0];
    if (p < 0 || p >= a.max_seq || rp < 0 || rp >= a.rope_rows) return;  // host validates; never go out of bounds
    if (lo >= L) {  // (an empty range: a sum below zero)
      if (threadIdx.x == 0) a.ml[((size_t)range * a.H + h) * 2] = -INFINITY, a.ml[((size_t)range * a.H + h) * 2 + 1] = -1.0f;
      return;
    }
    const float *src = a.q + (size_t)g * (qpk + 2) * hs, *sq = src + (size_t)(h % qpk) * hs, *sk = src + (size_t)qpk * hs;
    if ((int)threadIdx.x < hs) {
      x[0] = sq[d0], x[1] = sq[d1], x[2] = sk[d0], x[3] = sk[d1], x[4] = sk[hs + d0];
      if (d0 < a.n_elem) cs = a.cos[(size_t)rp * a.n_elem + d0], sn = a.sin[(size_t)rp * a.n_elem + d0];
    }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) k[u] = row(kb, lo + first + u * STEP);
  if (FUSED) {
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = row(vb, lo + first + u * STEP);
    __builtin_amdgcn_sched_barrier(0);
    if ((int)threadIdx.x < hs) {
      // x * cos + rotate_half(x) * sin on the first n_elem dims, two roundings
      auto turned = [&](float own, float mate) {
        return d0 < a.n_elem ? add_rn(mul_rn(own, cs), mul_rn(d0 < half ? -mate : mate, sn)) : own;
      };
      const float kd = turned(x[2], x[3]);
      qs[d0] = turned(x[0], x[1]);
      ks[d0] = kd;
      vs[d0] = x[4];
      if (h % qpk == 0 && hi == L) {
        kb[(size_t)p * hs + d0] = kd;
        vb[(size_t)p * hs + d0] = x[4];
      }
    }
  } else {
    const float* qr = a.q + ((size_t)t * a.H + h) * hs;
    for (int d = threadIdx.x; d < hs; d += 512) qs[d] = qr[d];
  }
  __syncthreads();
  const float4 q4 = kept(*(const float4*)(qs + at));
  auto own = [&](float4 (&x)[4], const float* row, int j0) {
    if (!FUSED || !mine) return;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (j0 + u * STEP == L - 1) x[u] = kept(*(const float4*)(row + at));
  };
  float mx = -INFINITY;
  for (int j0 = lo + first; j0 < hi; j0 += 4 * STEP) {
    if (j0 != lo + first) {
#pragma unroll
      for (int u = 0; u < 4; ++u) k[u] = row(kb, j0 + u * STEP);
    }
    own(k, ks, j0);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      float d = fmaf(q4.w, k[u].w, fmaf(q4.z, k[u].z, fmaf(q4.y, k[u].y, q4.x * k[u].x)));
      d = group_sum<LPK>(d) * a.scale;
      const int j = j0 + u * STEP;
      if (j < hi) {
        mx = fmaxf(mx, d);
        if (sub == 0) sc[j - lo] = d;
      }
    }
  }
  mx = wave_max(mx);
  if (lane == 0) red[wave] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 8; ++w) mx = fmaxf(mx, red[w]);
  __syncthreads();
  float sum = 0.0f;
  const float from = FUSED && a.parts > 1 && mx == -INFINITY ? 0.0f : mx;  // (other ranges may have finite scores)
  for (int j = threadIdx.x; j < hi - lo; j += 512) {
    const float e = expf(sc[j] - from);
    sc[j] = e;
    sum += e;
  }
  sum = wave_sum(sum);
  if (lane == 0) red[wave] = sum;
  __syncthreads();
  sum = ((red[0] + red[1]) + (red[2] + red[3])) + ((red[4] + red[5]) + (red[6] + red[7]));
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int j0 = lo + first; j0 < hi; j0 += 4 * STEP) {
    if (!FUSED || j0 != lo + first) {
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = row(vb, j0 + u * STEP);
    }
    own(v, vs, j0);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = j0 + u * STEP;
      const float w = j < hi ? sc[j - lo] : 0.0f;
      if (j < hi) o.x = fmaf(w, v[u].x, o.x), o.y = fmaf(w, v[u].y, o.y), o.z = fmaf(w, v[u].z, o.z), o.w = fmaf(w, v[u].w, o.w);
    }
  }
  auto fold = [&](float v) {  // over the lanes of other keys, the farthest first
    auto add = [](LanePair p) { return p.a + p.b; };
    if constexpr (LPK <= 32) v = add(lane_pair<32>(v));
    if constexpr (LPK <= 16) v = add(lane_pair<16>(v));
    return v;
  };
  static_assert(LPK >= 16, "lanes of a key");
  o = make_float4(fold(o.x), fold(o.y), fold(o.z), fold(o.w));
  __syncthreads();  // the weights are read
  float* part = sc;
  if (lane < LPK && mine) *(float4*)(part + wave * hs + sub * 4) = o;
  __syncthreads();
  for (int d = threadIdx.x; d < hs; d += 512) {
    float acc = 0.0f;
#pragma unroll
    for (int w = 0; w < 8; ++w) acc += part[w * hs + d];
    a.y[((size_t)(t + range) * a.H + h) * hs + d] = FUSED && a.parts > 1 ? acc : acc / sum;
  }
  if (FUSED && a.parts > 1 && threadIdx.x == 0) {
    a.ml[((size_t)range * a.H + h) * 2] = mx;
    a.ml[((size_t)range * a.H + h) * 2 + 1] = sum;
  }
}

template <bool FUSED>
static void f32_attention_go(const F32AttnArgs& a, int T, hipStream_t stream) {
  const int keys = a.parts > 1 ? f32_attention_chunk(a.max_seq, a.parts) : a.max_seq;
  const size_t lds = sizeof(float) * (size_t)std::max(keys, 8 * a.hs);
  const dim3 grid(FUSED ? a.parts : T, a.H);
  if (a.hs <= 64) f32_attention_vec_kernel<16, FUSED><<<grid, 512, lds, stream>>>(a);
  else if (a.hs <= 128) f32_attention_vec_kernel<32, FUSED><<<grid, 512, lds, stream>>>(a);
  else f32_attention_vec_kernel<64, FUSED><<<grid, 512, lds, stream>>>(a);
}

// grid (T, H): the same for head sizes that are no multiple of four (scores in LDS: max_seq floats, then partial sums)
__global__ void __launch_bounds__(256) f32_attention_kernel(const float* __restrict__ q, const float* __restrict__ kc,
                                                            const float* __restrict__ vc,
                                                            const int64_t* __restrict__ input_pos, float* __restrict__ y,
                                                            int n_head, int n_groups, int hs, int max_seq, float scale) {
  extern __shared__ float sc[];  // [max_seq] scores, then [256] partials
  __shared__ float red[4];
  __shared__ float qs[256];
  const int t = blockIdx.x, h = blockIdx.y;
  const int g = h / (n_head / n_groups);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long p = input_pos[t];
  const int L = (int)min(max(p + 1, 1L), (long)max_seq);
  const float* qr = q + ((size_t)t * n_head + h) * hs;
  for (int d = threadIdx.x; d < hs; d += 256) qs[d] = qr[d];
  __syncthreads();
  const float* kb = kc + (size_t)g * max_seq * hs;
  const float* vb = vc + (size_t)g * max_seq * hs;
  float mx = -INFINITY;
  for (int j = wave; j < L; j += 4) {
    float d = 0.0f;
    for (int e = lane; e < hs; e += 64) d = fmaf(qs[e], kb[(size_t)j * hs + e], d);
    d = wave_sum(d) * scale;
    mx = fmaxf(mx, d);
    if (lane == 0) sc[j] = d;
  }
  if (lane == 0) red[wave] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  __syncthreads();
  float sum = 0.0f;
  for (int j = threadIdx.x; j < L; j += 256) {
    const float e = expf(sc[j] - mx);
    sc[j] = e;
    sum += e;
  }
  sum = wave_sum(sum);
  if (lane == 0) red[wave] = sum;
  __syncthreads();
  sum = (red[0] + red[1]) + (red[2] + red[3]);
  // P.V: thread -> (dim d = tid % hs', key phase tid / hs') with hs' = min(hs, 256); partials reduced in LDS
  float* part = sc + max_seq;
  const int HSP = hs < 256 ? hs : 256, phases = 256 / HSP;
  const int ph = threadIdx.x / HSP, dd = threadIdx.x % HSP;
  for (int d0 = 0; d0 < hs; d0 += HSP) {
    float o = 0.0f;
    if (ph < phases)
      for (int j = ph; j < L; j += phases) o = fmaf(sc[j], vb[(size_t)j * hs + d0 + dd], o);
    part[threadIdx.x] = o;
    __syncthreads();
    if (threadIdx.x < HSP) {
      float acc = 0.0f;
      for (int k = 0; k < phases; ++k) acc += part[k * HSP + threadIdx.x];
      y[((size_t)t * n_head + h) * hs + d0 + threadIdx.x] = acc / sum;
    }
    __syncthreads();
  }
}

static unsigned elementwise_blocks(size_t n) { return (unsigned)std::min<size_t>((n + 255) / 256, 65535); }

}  // namespace lga

extern "C" int lga_f32_linear_act(const float* x, const float* w, const float* bias, int act, const float* residual,
                                  const float* residual2, float* y, int M, int N, int K, hipStream_t stream) {
  LGA_CHECK_ARG(x && w && y && M > 0 && N > 0 && K > 0 && M <= 65535 && act >= 0 && act <= 2, "lga_f32_linear: bad arguments");
  LGA_CHECK_ARG(((uintptr_t)x | (uintptr_t)w) % 16 == 0 || K % 4 != 0, "lga_f32_linear: 16-B aligned x, w needed");
  if (lga::f32_linear_in_tiles(M, N, K))
    (lga::f32_tiles_of_16(M, N) ? lga::f32_linear_tiles<16> : lga::f32_linear_tiles<32>)(x, w, bias, act, residual, residual2, y, M, N, K, stream);
  else if (lga::f32_linear_in_rows(M, N, K))
    lga::f32_linear_rows_kernel<<<dim3((N + 7) / 8, (M + 7) / 8), 256, 0, stream>>>(x, w, bias, act, residual, residual2, y, M, N, K);
  else lga::f32_linear_kernel<<<dim3((N + 3) / 4, M), 256, 0, stream>>>(x, w, bias, act, residual, residual2, y, N, K);
  LGA_LAUNCH_RETURN();
}

extern "C" int lga_f32_norm_linears(const float* x, int K, const float* nw1, const float* nb1, float eps1, const float* w1,
                                    const float* b1, int act1, float* y1, int N1, const float* nw2, const float* nb2,
                                    float eps2, const float* w2, const float* b2, int act2, float* y2, int N2,
                                    hipStream_t stream) {
  LGA_CHECK_ARG(x && nw1 && w1 && y1 && K > 0 && N1 > 0 && N2 >= 0 && (N2 == 0 || (nw2 && w2 && y2)) && act1 >= 0 && act1 <= 2 &&
                    act2 >= 0 && act2 <= 2,
                "lga_f32_norm_linears: bad arguments");
  LGA_CHECK_ARG(K % 4 == 0 && K <= 8192 && ((uintptr_t)w1 | (uintptr_t)w2) % 16 == 0,
                "lga_f32_norm_linears: K a multiple of 4 up to 8192 and 16-B aligned weights needed");
  // One output a wave up to 2048 workgroups. Beyond, a wave makes several, in as many workgroups as stand on the chip side by side: rows of
  // 1024 values and more let five (past 7996 values four: a workgroup's LDS comes in pieces of 1280 bytes) stand on a compute unit, and the
  // others of 2048 come behind them; shorter ones are done before that counts. Weights from memory, us in 2048 / 1280 workgroups: 256 values
  // to 14000 and 50304 outputs 6.4 / 7.0, 14.0 / 16.6, 768 to 8500, 20480 and 50304 8.2 / 7.6, 12.1 / 13.1, 27.0 / 28.2, 1024 to those 9.4 / 8.4,
  // 16.0 / 15.7, 36.2 / 35.1, 2048 to 8500 and 50304 18.1 / 16.8, 81 / 70, 4096 to 14000 51 / 44; 8192 to 8500 and 14000 in 2048 / 1280 / 1024
  // 86 / 84 / 73, 108 / 126 / 102, 8188 to 14000 109 / 129 / 104. (As many outputs a wave as any other or one less: 8192 to 14000 in 1167 134.)
  const int most = K < 1024 ? 2048 : (K + 4) * 4 <= 25 * 1280 ? 1280 : 1024;
  auto blocks = [&](int N) {
    const int all = (N + 3) / 4;
    return all > 2048 ? most : all;
  };
  const lga::F32NormLinears a{x, K, {{nw1, nb1, eps1, w1, b1, act1, y1, N1, blocks(N1)}, {nw2, nb2, eps2, w2, b2, act2, y2, N2, blocks(N2)}}};
  const unsigned grid = (unsigned)(blocks(N1) + blocks(N2));
  if (K <= 1024) lga::f32_norm_linears_kernel<4><<<grid, 256, K * sizeof(float), stream>>>(a);
  else lga::f32_norm_linears_kernel<16><<<grid, 256, K * sizeof(float), stream>>>(a);
  LGA_LAUNCH_RETURN();
}

extern "C" int lga_f32_linears_sum(const float* x1, const float* ml, int parts, int hs, const float* w1, const float* b1, int K1,
                                   const float* x2, const float* w2, const float* b2, int K2, const float* residual, float* y,
                                   int N, hipStream_t stream) {
  LGA_CHECK_ARG(x1 && w1 && x2 && w2 && residual && y && N > 0 && K1 > 0 && K2 > 0, "lga_f32_linears_sum: bad arguments");
  LGA_CHECK_ARG(K1 % 4 == 0 && K2 % 4 == 0 && ((uintptr_t)x1 | (uintptr_t)w1 | (uintptr_t)x2 | (uintptr_t)w2) % 16 == 0,
                "lga_f32_linears_sum: K in multiples of 4 and 16-B aligned operands needed");
  LGA_CHECK_ARG(parts == 1 || (parts > 1 && parts <= 8 && ml && hs > 0 && K1 % hs == 0 && K1 <= 8192 && K1 / hs <= 256),
                "lga_f32_linears_sum: 1 to 8 ranges of up to 256 heads, 8192 columns");
  const lga::F32LinearsSum a{x1, w1, b1, x2, w2, b2, residual, y, N, K1, K2, ml, parts, hs};
  const size_t joined = parts > 1 ? (size_t)K1 + (K1 / hs * 9 + 3) / 4 * 4 : 0;
  const int ahead = K1 > K2 / 2 || K2 > 8192 ? 0 : K2 <= 4096 ? 4 : 8;
  const size_t lds = (joined + (ahead ? K2 : 0)) * sizeof(float);
  auto go = [&](auto many) {
    constexpr bool PARTS = decltype(many)::value;
    return ahead == 0 ? lga::f32_linears_sum_kernel<PARTS, 0> : ahead == 4 ? lga::f32_linears_sum_kernel<PARTS, 4> : lga::f32_linears_sum_kernel<PARTS, 8>;
  };
  const auto kernel = parts > 1 ? go(std::true_type{}) : go(std::false_type{});
  kernel<<<(N + 3) / 4, 256, lds, stream>>>(a);
  LGA_LAUNCH_RETURN();
}

extern "C" int lga_f32_linear(const float* x, const float* w, const float* bias, const float* residual, float* y,
                              int M, int N, int K, hipStream_t stream) {
  return lga_f32_linear_act(x, w, bias, 0, residual, nullptr, y, M, N, K, stream);
}

extern "C" int lga_f32_layernorm(const float* x, const float* w, const float* b, float* y, int rows, int n, float eps,
                                 hipStream_t stream) {
  LGA_CHECK_ARG(x && w && y && rows > 0 && n > 0, "lga_f32_layernorm: bad arguments");
  lga::f32_layernorm_go(x, w, b, y, nullptr, nullptr, nullptr, rows, n, eps, 0.0f, stream);
  LGA_LAUNCH_RETURN();
}

extern "C" int lga_f32_layernorm_pair(const float* x, const float* w, const float* b, float* y, float eps, const float* w2,
                                      const float* b2, float* y2, float eps2, int rows, int n, hipStream_t stream) {
  LGA_CHECK_ARG(x && w && y && w2 && y2 && rows > 0 && n > 0, "lga_f32_layernorm_pair: bad arguments");
  lga::f32_layernorm_go(x, w, b, y, w2, b2, y2, rows, n, eps, eps2, stream);
  LGA_LAUNCH_RETURN();
}

extern "C" int lga_f32_gelu(const float* a, float* y, long n, int approximate_tanh, hipStream_t stream) {
  LGA_CHECK_ARG(a && y && n > 0, "lga_f32_gelu: bad arguments");
  lga::f32_gelu_kernel<<<lga::elementwise_blocks((size_t)n), 256, 0, stream>>>(a, y, (size_t)n, approximate_tanh);
  LGA_LAUNCH_RETURN();
}

extern "C" int lga_f32_add(const float* a, const float* b, float* y, long n, hipStream_t stream) {
  LGA_CHECK_ARG(a && b && y && n > 0, "lga_f32_add: bad arguments");
  lga::f32_add_kernel<<<lga::elementwise_blocks((size_t)n), 256, 0, stream>>>(a, b, y, (size_t)n);
  LGA_LAUNCH_RETURN();
}

extern "C" int lga_f32_rope_kv_append(const float* qkv, float* q_out, float* k_cache, float* v_cache,
                                      const int64_t* cache_pos, const int64_t* rope_pos, const float* cos,
                                      const float* sin, int rope_rows, int T, int n_head, int n_query_groups,
                                      int head_size, int rope_n_elem, int max_seq, hipStream_t stream) {
  LGA_CHECK_ARG(qkv && q_out && k_cache && v_cache && cache_pos && rope_pos && cos && sin,
                "lga_f32_rope_kv_append: null pointer");
  LGA_CHECK_ARG(T > 0 && n_query_groups > 0 && n_head % n_query_groups == 0 && head_size > 0 &&
                    rope_n_elem % 2 == 0 && rope_n_elem <= head_size && max_seq > 0 && rope_rows > 0,
                "lga_f32_rope_kv_append: bad geometry");
  lga::f32_rope_kv_kernel<<<dim3(T, n_query_groups), 256, 0, stream>>>(qkv, q_out, k_cache, v_cache, cache_pos,
                                                                       rope_pos, cos, sin, n_head, n_query_groups,
                                                                       head_size, rope_n_elem, max_seq, rope_rows);
  LGA_LAUNCH_RETURN();
}

extern "C" int lga_f32_attention(const float* q, const float* k_cache, const float* v_cache, const int64_t* input_pos,
                                 float* y, int T, int n_head, int n_query_groups, int head_size, int max_seq,
                                 float scale, hipStream_t stream) {
  LGA_CHECK_ARG(q && k_cache && v_cache && input_pos && y, "lga_f32_attention: null pointer");
  LGA_CHECK_ARG(T > 0 && T <= 65535 && n_query_groups > 0 && n_head % n_query_groups == 0 && head_size > 0 &&
                    head_size <= 256,
                "lga_f32_attention: bad geometry (head_size <= 256)");
  LGA_CHECK_ARG(max_seq > 0 && max_seq <= 32768, "lga_f32_attention: max_seq must be in [1, 32768] (scores in LDS)");
  if (head_size % 4 == 0 && ((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) % 16 == 0) {
    const lga::F32AttnArgs a{q, (float*)k_cache, (float*)v_cache, input_pos, y, n_head, n_query_groups, head_size, max_seq, scale,
                             nullptr, nullptr, nullptr, 0, 0, 1, nullptr};
    lga::f32_attention_go<false>(a, T, stream);
    LGA_LAUNCH_RETURN();
  }
  const size_t lds = ((size_t)max_seq + 256) * sizeof(float);
  lga::f32_attention_kernel<<<dim3(T, n_head), 256, lds, stream>>>(q, k_cache, v_cache, input_pos, y, n_head,
                                                                    n_query_groups, head_size, max_seq, scale);
  LGA_LAUNCH_RETURN();
}

extern "C" int lga_f32_attention_decode_parts(const float* qkv, float* k_cache, float* v_cache, const int64_t* cache_pos,
                                              const int64_t* rope_pos, const float* cos, const float* sin, int rope_rows,
                                              float* y, float* ml, int parts, int n_head, int n_query_groups, int head_size,
                                              int rope_n_elem, int max_seq, float scale, hipStream_t stream) {
  LGA_CHECK_ARG(qkv && k_cache && v_cache && cache_pos && rope_pos && cos && sin && y,
                "lga_f32_attention_decode: null pointer");
  LGA_CHECK_ARG(parts == 1 || (parts > 1 && parts <= 8 && ml), "lga_f32_attention_decode: 1 to 8 ranges");
  LGA_CHECK_ARG(n_query_groups > 0 && n_head > 0 && n_head <= 65535 && n_head % n_query_groups == 0 && head_size > 0 &&
                    head_size <= 256 && head_size % 4 == 0 && rope_n_elem >= 0 && rope_n_elem % 2 == 0 &&
                    rope_n_elem <= head_size && rope_rows > 0 && max_seq > 0 && max_seq <= 32768,
                "lga_f32_attention_decode: bad geometry (head_size a multiple of 4 up to 256, max_seq <= 32768)");
  LGA_CHECK_ARG(((uintptr_t)k_cache | (uintptr_t)v_cache) % 16 == 0, "lga_f32_attention_decode: aligned caches");
  const lga::F32AttnArgs a{qkv, k_cache, v_cache, cache_pos, y, n_head, n_query_groups, head_size, max_seq, scale,
                           rope_pos, cos, sin, rope_n_elem, rope_rows, parts, ml};
  lga::f32_attention_go<true>(a, 1, stream);
  LGA_LAUNCH_RETURN();
}

extern "C" int lga_f32_attention_parts(int n_head, int max_seq) {
  // (ranges of 64 keys or more, whatever the position; eight are joined in one round of loads)
  return n_head > 0 && max_seq > 0 ? std::min(8, (max_seq + 63) / 64) : 0;
}

extern "C" int lga_f32_attention_decode(const float* qkv, float* k_cache, float* v_cache, const int64_t* cache_pos,
                                        const int64_t* rope_pos, const float* cos, const float* sin, int rope_rows, float* y,
                                        int n_head, int n_query_groups, int head_size, int rope_n_elem, int max_seq,
                                        float scale, hipStream_t stream) {
  return lga_f32_attention_decode_parts(qkv, k_cache, v_cache, cache_pos, rope_pos, cos, sin, rope_rows, y, nullptr, 1, n_head,
                                        n_query_groups, head_size, rope_n_elem, max_seq, scale, stream);
}
