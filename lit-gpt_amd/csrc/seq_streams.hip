// Multi-stream residual (hyper-connections) of the layered models, fp32 throughout.
//
// The residual is kept in `s` parallel streams x[t][0 .. s)[W]. A sublayer reads a fixed weighted sum of the
// streams, u = sum_i a[i] x_i, through an RMS norm; its output y goes back into every stream while the streams
// are mixed: x_j <- sum_i m[i][j] x_i + b[j] y. With s = 1, a = b = m = 1 this is the ordinary residual sum.
//
//   lgs_embed_streams   x[t][j] = table[tokens[t]] * scale for every stream j
//   lgs_streams_step    one launch per sublayer boundary: the write-back of the sublayer that just ran (optional)
//                       followed by the read + norm of the next one (optional), so the streams are read once
//   lgs_streams_held    a boundary of a prompt that makes the streams anew from the embedding (or stored streams) and the
//                       sublayers' outputs since, instead of storing and reading them
//   lgs_sandwich_step   the boundary of layers with one residual whose sublayers are normed on the way in (and
//                       optionally out): the norms and the average of up to two branch outputs, the output norm times
//                       the layer scale, the residual add, a learned average over the depth at a layer's end or what
//                       joins the residual ahead of a pass over looped layers, and the next sublayer's input norm in
//                       one launch
#include "seq_common.h"

namespace lgs {

constexpr int kMaxStreams = 8;

template <bool WF32>
__global__ void __launch_bounds__(256) embed_streams_kernel(const int* __restrict__ tokens, const void* __restrict__ table,
                                                            float scale, float* __restrict__ x, int W, int vocab, int streams) {
  const size_t t = blockIdx.x;
  const size_t src = (size_t)min(max(tokens[t], 0), vocab - 1) * W;  // (the host validates ids; never read out of bounds)
  for (int i = blockIdx.y * 256 + threadIdx.x; i < W; i += gridDim.y * 256) {
    const float v = wload<WF32>(table, src + i) * scale;
    for (int j = 0; j < streams; ++j) x[(t * streams + j) * W + i] = v;
  }
}

struct StreamArgs {
  float* x;          // [T][s][W]
  const float* y;    // [T][W] sublayer output to write back (null: no write-back)
  const float* mix;  // [s][s] indexed [from][to]
  const float* out;  // [s]
  const float* in;   // [s] read weights of the next sublayer (null: no read)
  const float* w;    // [W] norm weight of the next sublayer (null: the weighted sum itself is the result)
  float* h;          // [T][W] normed read
  uint16_t* h16;     // optional bf16 copy of h
  float eps;
  int W, s;
};

// grid (T): a workgroup owns a token; thread i owns columns i, i + 256, ... in every stream
__global__ void __launch_bounds__(256) streams_step_kernel(StreamArgs p) {
  __shared__ float red[4];
  __shared__ float cm[kMaxStreams * kMaxStreams], cb[kMaxStreams], ca[kMaxStreams];
  const int s = p.s, W = p.W;
  if (threadIdx.x < s * s) cm[threadIdx.x] = p.mix ? p.mix[threadIdx.x] : 0.0f;
  if (threadIdx.x < s) {
    cb[threadIdx.x] = p.out ? p.out[threadIdx.x] : 0.0f;
    ca[threadIdx.x] = p.in ? p.in[threadIdx.x] : 0.0f;
  }
  __syncthreads();
  float* xt = p.x + (size_t)blockIdx.x * s * W;
  const float* yt = p.y ? p.y + (size_t)blockIdx.x * W : nullptr;
  float ss = 0.0f;
  for (int i = threadIdx.x; i < W; i += 256) {
    float v[kMaxStreams];
#pragma unroll
    for (int j = 0; j < kMaxStreams; ++j) v[j] = j < s ? xt[(size_t)j * W + i] : 0.0f;
    if (yt) {
      const float y = yt[i];
      float nv[kMaxStreams];
#pragma unroll
      for (int j = 0; j < kMaxStreams; ++j) {
        float acc = 0.0f;
#pragma unroll
        for (int k = 0; k < kMaxStreams; ++k)
          if (k < s && j < s) acc = fmaf(cm[k * s + j], v[k], acc);
        nv[j] = j < s ? fmaf(cb[j], y, acc) : 0.0f;
      }
#pragma unroll
      for (int j = 0; j < kMaxStreams; ++j) {
        v[j] = nv[j];
        if (j < s) xt[(size_t)j * W + i] = nv[j];
      }
    }
    if (p.in) {
      float u = 0.0f;
#pragma unroll
      for (int j = 0; j < kMaxStreams; ++j)
        if (j < s) u = fmaf(ca[j], v[j], u);
      ss = fmaf(u, u, ss);
      p.h[(size_t)blockIdx.x * W + i] = u;  // normed below
    }
  }
  if (!p.in || !p.w) return;
  ss = block_sum_256(ss, red);
  const float rstd = 1.0f / sqrtf(ss / (float)W + p.eps);
  for (int i = threadIdx.x; i < W; i += 256) {
    const size_t at = (size_t)blockIdx.x * W + i;
    const float v = p.h[at] * rstd * p.w[i];  // (each thread re-reads what it wrote itself)
    p.h[at] = v;
    if (p.h16) p.h16[at] = f2bf(v);
  }
}

// The same step with a token's columns in registers: thread i owns columns i + 256 c, c < CPT (W <= 256 CPT), of
// SMAX >= s streams. All loads are issued before the first use and the normed read is written from registers, so a
// one-token step is one round trip to memory instead of one per column block.
// (NT threads per token: 256 for prompts, 1024 for steps of a few tokens, whose one workgroup per token is then
// four times shorter.)
template <int SMAX, int CPT, int NT>
__global__ void __launch_bounds__(NT) streams_step_reg_kernel(StreamArgs p) {
  __shared__ float red[NT / 64];
  __shared__ float cm[kMaxStreams * kMaxStreams], cb[kMaxStreams], ca[kMaxStreams];
  const int s = p.s, W = p.W, tid = threadIdx.x;
  float* xt = p.x + (size_t)blockIdx.x * s * W;
  const float* yt = p.y ? p.y + (size_t)blockIdx.x * W : nullptr;
  // (streams and columns past the last: those again, left out below; a load under a condition of its own is a branch. One token of four
  // streams of 2048: 5.1 us with branches and the links' loads ahead, 4.5 here)
  float v[SMAX][CPT], y[CPT], nw[CPT], mix = 0.0f, wr = 0.0f, rd = 0.0f;
#pragma unroll
  for (int c = 0; c < CPT; ++c)
#pragma unroll
    for (int j = 0; j < SMAX; ++j) v[j][c] = xt[(size_t)min(j, s - 1) * W + min(tid + NT * c, W - 1)];
  if (yt) {
#pragma unroll
    for (int c = 0; c < CPT; ++c) y[c] = yt[min(tid + NT * c, W - 1)];
  }
  if (p.in && p.w) {
#pragma unroll
    for (int c = 0; c < CPT; ++c) nw[c] = p.w[min(tid + NT * c, W - 1)];
  }
  if (p.mix) mix = p.mix[min(tid, s * s - 1)];
  if (p.out) wr = p.out[min(tid, s - 1)];
  if (p.in) rd = p.in[min(tid, s - 1)];
  if (tid < s * s) cm[tid] = mix;
  if (tid < s) cb[tid] = wr, ca[tid] = rd;
#pragma unroll
  for (int c = 0; c < CPT; ++c)
    if (tid + NT * c >= W) {
      y[c] = 0.0f;
#pragma unroll
      for (int j = 0; j < SMAX; ++j) v[j][c] = 0.0f;
    }
  __syncthreads();
  float u[CPT], ss = 0.0f;
#pragma unroll
  for (int c = 0; c < CPT; ++c) {
    const int i = threadIdx.x + NT * c;
    if (yt) {
      float nv[SMAX];
#pragma unroll
      for (int j = 0; j < SMAX; ++j) {
        float acc = 0.0f;
#pragma unroll
        for (int k = 0; k < SMAX; ++k)
          if (k < s && j < s) acc = fmaf(cm[k * s + j], v[k][c], acc);
        nv[j] = j < s ? fmaf(cb[j], y[c], acc) : 0.0f;
      }
#pragma unroll
      for (int j = 0; j < SMAX; ++j) {
        v[j][c] = nv[j];
        if (j < s && i < W) xt[(size_t)j * W + i] = nv[j];
      }
    }
    float a = 0.0f;
#pragma unroll
    for (int j = 0; j < SMAX; ++j)
      if (j < s) a = fmaf(ca[j], v[j][c], a);
    u[c] = a;
    ss = fmaf(a, a, ss);
  }
  if (!p.in) return;
  float rstd = 1.0f;
  if (p.w) {
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    ss = 0.0f;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) ss += red[w];
    rstd = 1.0f / sqrtf(ss / (float)W + p.eps);
  }
#pragma unroll
  for (int c = 0; c < CPT; ++c) {
    const int i = threadIdx.x + NT * c;
    if (i >= W) continue;
    const size_t at = (size_t)blockIdx.x * W + i;
    const float r = p.w ? u[c] * rstd * nw[c] : u[c];
    p.h[at] = r;
    if (p.h16) p.h16[at] = f2bf(r);
  }
}

template <int SMAX>
static bool streams_step_reg(const StreamArgs& p, int T, hipStream_t stream) {
  if (T <= 32 && p.W > 512) {
    if (p.W <= 2048) streams_step_reg_kernel<SMAX, 2, 1024><<<T, 1024, 0, stream>>>(p);
    else if (p.W <= 4096) streams_step_reg_kernel<SMAX, 4, 1024><<<T, 1024, 0, stream>>>(p);
    else if (p.W <= 8192) streams_step_reg_kernel<SMAX, 8, 1024><<<T, 1024, 0, stream>>>(p);
    else return false;
    return true;
  }
  if (p.W <= 1024) streams_step_reg_kernel<SMAX, 4, 256><<<T, 256, 0, stream>>>(p);
  else if (p.W <= 2048) streams_step_reg_kernel<SMAX, 8, 256><<<T, 256, 0, stream>>>(p);
  else if (p.W <= 4096 && SMAX <= 4) streams_step_reg_kernel<SMAX, 16, 256><<<T, 256, 0, stream>>>(p);
  else return false;
  return true;
}

// A boundary of a prompt without the write-back: the streams are made anew, in registers, from where they last stood (the embedding, or
// streams that were stored) and the outputs of the K sublayers since, and stored only where `x` is given. The values are
// those of K steps of the kernels above, operation by operation; thread i owns columns i, i + 256, ... as there, so the sums
// of squares are theirs too.
//
// Bound by memory: 2407 rows of 4096, four streams, us (and TB/s) with 0, 1, 4 and 8 outputs since the embedding 16.6 (2.4), 23 (3.4),
// 43 (4.6), 79 (4.7), where a step that stores took 92 (4.1); the embedding's own 50 are gone. Storing s streams costs 2 s rows of
// fp32 a boundary, reading what they are made of one row per sublayer since, so four streams go on from the embedding (half a
// row) for eight sublayers and from stored streams for three (seq_ops.streams_hold). Columns come in two portions in turn, the next
// one's loads ahead of the sums.
constexpr int kMaxHeld = 8;
struct HeldArgs {
  const int* tokens;  // embedding base: x_j = table[tokens[t]] * scale
  const void* table;
  int w_f32, vocab;
  float scale;
  const float* base;  // stored base [T][s][W]
  float* x;           // where the streams are stored (null: nowhere; base itself or another place)
  const float* y[kMaxHeld];
  const float* mix[kMaxHeld];
  const float* out[kMaxHeld];
  const float *in, *w;  // w null: the weighted sum itself is the result
  float* h;             // fp32 result (may be null beside h16)
  uint16_t* h16;
  float eps;
  int W;
};

// FROM: the embedding in bf16 (0) or fp32 (1), or stored streams (2)
template <int S, int K, int FROM>
__global__ void __launch_bounds__(256) streams_held_kernel(HeldArgs p) {
  constexpr int CPT = 16, ROWS = K + (FROM == 2 ? S : 1);          // columns of a thread (W <= 4096); rows that they are made of
  constexpr int CH = ROWS <= 2 ? 16 : ROWS <= 4 ? 8 : 4;           // ... at a time
  __shared__ float us[CPT * 256];  // the weighted sums, until the norm is known (every thread its own)
  __shared__ float red[4];
  const int tid = threadIdx.x, W = p.W;
  const size_t t = blockIdx.x;
  const float* base = FROM == 2 ? p.base + t * S * W : nullptr;
  const size_t row = FROM == 2 ? 0 : (size_t)min(max(p.tokens[t], 0), p.vocab - 1) * W;  // (as above)
  const float* table32 = (const float*)p.table + row;
  const uint16_t* table16 = (const uint16_t*)p.table + row;
  struct Columns {
    float y[K + 1][CH], v[FROM == 2 ? S : 1][CH];
  };
  auto load = [&](int i0, Columns& o) {  // (columns past the end repeat the last one, never stored or summed)
#pragma unroll
    for (int k = 0; k < K; ++k) {
      int at = k;
      asm volatile("" : "+s"(at));  // (all outputs' addresses at once are too many scalars)
      const float* y = p.y[at] + t * W;
#pragma unroll
      for (int c = 0; c < CH; ++c) o.y[k][c] = y[min(i0 + 256 * c, W - 1)];
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int i = min(i0 + 256 * c, W - 1);
      if constexpr (FROM == 2) {
#pragma unroll
        for (int j = 0; j < S; ++j) o.v[j][c] = base[(size_t)j * W + i];
      } else if constexpr (FROM == 1) {
        o.v[0][c] = table32[i];
      } else {
        o.v[0][c] = __uint_as_float((uint32_t)table16[i]);
      }
    }
  };
  // A sublayer's links come as scalars, for all columns at a time and one sublayer ahead (read from LDS five operations need a
  // read). The index is hidden from the compiler, or it fetches all sublayers' first, more than there are scalar registers.
  using Scalars = const __attribute__((address_space(4))) float*;
  struct Links {
    float mix[S * S], out[S];
  };
  auto fetch = [&](int k, Links& o) {
    asm volatile("" : "+s"(k));
    const Scalars mix = (Scalars)p.mix[k], out = (Scalars)p.out[k];
#pragma unroll
    for (int e = 0; e < S * S; ++e) o.mix[e] = mix[e];
#pragma unroll
    for (int e = 0; e < S; ++e) o.out[e] = out[e];
  };
  float ss = 0.0f;
  auto work = [&](int i0, const Columns& a) {
    float v[CH][S];
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
      for (int j = 0; j < S; ++j) {
        if constexpr (FROM == 2) v[c][j] = a.v[j][c];
        else if constexpr (FROM == 1) v[c][j] = a.v[0][c] * p.scale;
        else v[c][j] = __uint_as_float(__float_as_uint(a.v[0][c]) << 16) * p.scale;
      }
    Links l[2];
    if constexpr (K > 0) fetch(0, l[0]);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (k + 1 < K) fetch(k + 1, l[(k + 1) & 1]);
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        float nv[S];
#pragma unroll
        for (int j = 0; j < S; ++j) {
          float acc = 0.0f;
#pragma unroll
          for (int f = 0; f < S; ++f) acc = fmaf(l[k & 1].mix[f * S + j], v[c][f], acc);
          nv[j] = fmaf(l[k & 1].out[j], a.y[k][c], acc);
        }
#pragma unroll
        for (int j = 0; j < S; ++j) v[c][j] = nv[j];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int i = i0 + 256 * c;
      float r = 0.0f;
#pragma unroll
      for (int j = 0; j < S; ++j) r = fmaf(((Scalars)p.in)[j], v[c][j], r);
      us[i] = r;  // (without a branch, or the sums above move behind it, and behind all the links' loads)
      const float more = fmaf(r, r, ss);
      ss = i < W ? more : ss;
    }
    if (p.x) {
#pragma unroll
      for (int c = 0; c < CH; ++c)
        if (i0 + 256 * c < W) {
#pragma unroll
          for (int j = 0; j < S; ++j) p.x[(t * S + j) * W + i0 + 256 * c] = v[c][j];
        }
    }
  };
  constexpr int STEP = CH * 256;
  Columns a, b;  // (two in turn: a copy would wait for the loads ahead)
  load(tid, a);
#pragma unroll 1
  for (int i0 = tid; i0 < W; i0 += 2 * STEP) {
    if (CH < CPT) load(i0 + STEP, b);
    __builtin_amdgcn_sched_barrier(0);
    work(i0, a);
    if (CH == CPT || i0 + STEP >= W) break;
    load(i0 + 2 * STEP, a);
    __builtin_amdgcn_sched_barrier(0);
    work(i0 + STEP, b);
  }
  float rstd = 1.0f, nw[CPT];
  if (p.w) {
#pragma unroll
    for (int c = 0; c < CPT; ++c) nw[c] = p.w[min(tid + 256 * c, W - 1)];
    ss = wave_sum(ss);
    if ((tid & 63) == 0) red[tid >> 6] = ss;
    __syncthreads();
    ss = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) ss += red[w];
    rstd = 1.0f / sqrtf(ss / (float)W + p.eps);
  }
#pragma unroll
  for (int c = 0; c < CPT; ++c) {
    const int i = tid + 256 * c;
    if (i >= W) break;
    const float r = p.w ? us[i] * rstd * nw[c] : us[i];
    if (p.h) p.h[t * W + i] = r;
    if (p.h16) p.h16[t * W + i] = f2bf(r);
  }
}

template <int S, int FROM, int K = FROM == 2 ? 1 : 0>
static bool streams_held(const HeldArgs& p, int T, int count, hipStream_t stream) {
  if (count == K) {
    streams_held_kernel<S, K, FROM><<<T, 256, 0, stream>>>(p);
    return true;
  }
  if constexpr (K < (FROM == 2 ? 3 : 2 * S)) return streams_held<S, FROM, K + 1>(p, T, count, stream);
  return false;
}
template <int S>
static bool streams_held_from(const HeldArgs& p, int T, int count, hipStream_t stream) {
  return p.base ? streams_held<S, 2>(p, T, count, stream)
                : p.w_f32 ? streams_held<S, 1>(p, T, count, stream) : streams_held<S, 0>(p, T, count, stream);
}

// ------------------------------------------------------------------------------------------------ sandwich norms
// One boundary between two sublayers of a layer whose sublayers are normed on the way in AND on the way out.
// With y0 (the sublayer that ran; up to two branches): b_i = w_i ? y_i / rms(y_i) * w_i : y_i, s = coef * sum_i b_i,
// x <- x + s / rms(s) * post_w (post_w: the output norm's weight times the layer's per-channel scale; null: no output
// norm, x <- x + s). With depth_w (a layer's end, average over the depth): this x is X_n, what the layer itself produced, kept in row
// block n of `hist` when there is room, and x <- depth_w[n] X_n + sum_{j < n} depth_w[j] hist[j]. x may be read from
// another place (x_in) than it is written to. With add_vec (ahead of a pass over looped layers): x <- x + add_vec + add (a
// row of its own, if given). Then with next_w: h = x / rms(x) * next_w, the next sublayer's input (fp32 and / or its bf16 rounding). Every root mean
// square has eps inside the root. grid (rows); a row lives in registers up to 256 * CPT columns, else it is re-read.
struct SandwichArgs {
  const float* x_in;
  float* x;
  const float *y0, *w0, *y1, *w1;
  float coef;
  const float* post_w;
  const float* next_w;
  float* h;
  uint16_t* h16;
  float eps;
  int n;
  float* hist;  // [hist_rows][rows][n]: X_0, X_1, ...
  const float* depth_w;
  int n_prev, hist_rows;
  const float* add_vec;  // [n]
  const float* add;      // [rows][n] or null
};

// sums of two values over the 256 threads of a workgroup at once (`red` holds 8 floats)
__device__ __forceinline__ void block_sum2_256(float& u, float& v, float* red) {
  u = wave_sum(u);
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    red[threadIdx.x >> 6] = u;
    red[4 + (threadIdx.x >> 6)] = v;
  }
  __syncthreads();
  u = (red[0] + red[1]) + (red[2] + red[3]);
  v = (red[4] + red[5]) + (red[6] + red[7]);
}

template <int CPT, bool DEPTH, bool PASS>
__global__ void __launch_bounds__(256) sandwich_step_kernel(SandwichArgs p) {
  __shared__ float red[8];
  const size_t r = blockIdx.x;
  const int n = p.n, tid = threadIdx.x;
  float* xr = p.x + r * n;
  const float* xi = p.x_in + r * n;
  const float inv_n = 1.0f / (float)n;
  // every operand of the registers' share of the row is fetched up front, so that the reductions below wait for
  // one batch of loads only
  float xv[CPT], av[CPT], bv[CPT], w0[CPT], w1[CPT], wp[CPT], wn[CPT], pv[PASS ? CPT : 1];
  const float *a = p.y0 ? p.y0 + r * n : nullptr, *b = p.y1 ? p.y1 + r * n : nullptr;
  // (past the end the last column, left out below: a load under a condition of its own is a branch each; us with them / here: 3 rows of
  // 4096 6.0 / 4.8, 8 of 2048 4.4 / 3.5, 2407 of 4096 30.9 / 28.6)
  auto get = [&](float (&v)[CPT], const float* from, float none) {
    if (from) {
#pragma unroll
      for (int e = 0; e < CPT; ++e) v[e] = from[min(tid + 256 * e, n - 1)];
    } else {
#pragma unroll
      for (int e = 0; e < CPT; ++e) v[e] = none;
    }
  };
  get(xv, xi, 0.0f), get(av, a, 0.0f), get(bv, b, 0.0f);
  get(w0, a ? p.w0 : nullptr, 1.0f), get(w1, b ? p.w1 : nullptr, 1.0f);
  get(wp, p.post_w, 0.0f), get(wn, p.next_w, 0.0f);
  if constexpr (PASS) {
    get(pv, p.add_vec, 0.0f);
    if (p.add)
#pragma unroll
      for (int e = 0; e < CPT; ++e) pv[e] += p.add[r * n + min(tid + 256 * e, n - 1)];
  }
#pragma unroll
  for (int e = 0; e < CPT; ++e)
    if (tid + 256 * e >= n) xv[e] = av[e] = bv[e] = 0.0f;
  // the earlier layers' share of the average needs nothing of this sublayer: its loads run beside the reductions
  const size_t hs = (size_t)gridDim.x * n;
  float hv[CPT];
  if (DEPTH) {
#pragma unroll
    for (int e = 0; e < CPT; ++e) hv[e] = 0.0f;
    constexpr int HB = CPT > 8 ? 2 : 4;  // earlier results fetched side by side
    for (int j = 0; j < p.n_prev; j += HB) {
      float t[HB][CPT], c[HB];
#pragma unroll
      for (int k = 0; k < HB; ++k) {
        const bool there = j + k < p.n_prev;
        c[k] = there ? p.depth_w[j + k] : 0.0f;
#pragma unroll
        for (int e = 0; e < CPT; ++e) {
          const int i = tid + 256 * e;
          t[k][e] = (there && i < n) ? p.hist[(j + k) * hs + r * n + i] : 0.0f;
        }
      }
#pragma unroll
      for (int k = 0; k < HB; ++k)
#pragma unroll
        for (int e = 0; e < CPT; ++e) hv[e] = fmaf(c[k], t[k][e], hv[e]);
    }
  }
  if (a) {
    float sa = 0.0f, sb = 0.0f;
#pragma unroll
    for (int e = 0; e < CPT; ++e) {
      sa = fmaf(av[e], av[e], sa);
      sb = fmaf(bv[e], bv[e], sb);
    }
    for (int i = tid + 256 * CPT; i < n; i += 256) {
      sa = fmaf(a[i], a[i], sa);
      if (b) sb = fmaf(b[i], b[i], sb);
    }
    float ra = 1.0f, rb = 1.0f;
    if (p.w0 || (b && p.w1)) {
      block_sum2_256(sa, sb, red);
      if (p.w0) ra = 1.0f / sqrtf(sa * inv_n + p.eps);
      if (b && p.w1) rb = 1.0f / sqrtf(sb * inv_n + p.eps);
    }
    auto joined = [&](float ya, float yb, float wa, float wb) {
      float s = p.w0 ? ya * ra * wa : ya;
      if (b) s += p.w1 ? yb * rb * wb : yb;
      return s * p.coef;
    };
    auto joined_at = [&](int i) {
      return joined(a[i], b ? b[i] : 0.0f, p.w0 ? p.w0[i] : 1.0f, (b && p.w1) ? p.w1[i] : 1.0f);
    };
    float ss = 0.0f;
#pragma unroll
    for (int e = 0; e < CPT; ++e) {
      av[e] = tid + 256 * e < n ? joined(av[e], bv[e], w0[e], w1[e]) : 0.0f;  // (av now holds the joined value)
      ss = fmaf(av[e], av[e], ss);
    }
    for (int i = tid + 256 * CPT; i < n; i += 256) {
      const float s = joined_at(i);
      ss = fmaf(s, s, ss);
    }
    float rs = 1.0f;
    if (p.post_w) rs = 1.0f / sqrtf(block_sum_256(ss, red) * inv_n + p.eps);
#pragma unroll
    for (int e = 0; e < CPT; ++e) {
      const int i = tid + 256 * e;
      if (i < n) {
        xv[e] = p.post_w ? fmaf(av[e] * rs, wp[e], xv[e]) : xv[e] + av[e];
        if (!DEPTH && !PASS) xr[i] = xv[e];
      }
    }
    for (int i = tid + 256 * CPT; i < n; i += 256) {
      const float s = joined_at(i);
      xr[i] = p.post_w ? fmaf(s * rs, p.post_w[i], xi[i]) : xi[i] + s;
    }
  }
  if (DEPTH) {
    const float cn = p.depth_w[p.n_prev];
    float* keep = p.n_prev < p.hist_rows ? p.hist + p.n_prev * hs + r * n : nullptr;
#pragma unroll
    for (int e = 0; e < CPT; ++e) {
      const int i = tid + 256 * e;
      if (i < n) {
        if (keep) keep[i] = xv[e];
        xv[e] = fmaf(cn, xv[e], hv[e]);
        xr[i] = xv[e];
      }
    }
    for (int i = tid + 256 * CPT; i < n; i += 256) {
      const float x = a ? xr[i] : xi[i];  // (a: written by this thread above)
      float v = 0.0f;
      for (int j = 0; j < p.n_prev; ++j) v = fmaf(p.depth_w[j], p.hist[j * hs + r * n + i], v);
      if (keep) keep[i] = x;
      xr[i] = fmaf(cn, x, v);
    }
  }
  if (PASS) {
#pragma unroll
    for (int e = 0; e < CPT; ++e) {
      const int i = tid + 256 * e;
      if (i < n) {
        xv[e] += pv[e];
        xr[i] = xv[e];
      }
    }
    for (int i = tid + 256 * CPT; i < n; i += 256) {
      const float x = a ? xr[i] : xi[i];  // (a: written by this thread above)
      xr[i] = x + (p.add_vec[i] + (p.add ? p.add[r * n + i] : 0.0f));
    }
  }
  if (!p.next_w) return;
  float sx = 0.0f;
#pragma unroll
  for (int e = 0; e < CPT; ++e) sx = fmaf(xv[e], xv[e], sx);
  const float* xs = (a || DEPTH || PASS) ? xr : xi;  // (xr: written by this thread above)
  for (int i = tid + 256 * CPT; i < n; i += 256) sx = fmaf(xs[i], xs[i], sx);
  const float rx = 1.0f / sqrtf(block_sum_256(sx, red) * inv_n + p.eps);
#pragma unroll
  for (int e = 0; e < CPT; ++e) {
    const int i = tid + 256 * e;
    if (i < n) {
      const float o = xv[e] * rx * wn[e];
      if (p.h) p.h[r * n + i] = o;
      if (p.h16) p.h16[r * n + i] = f2bf(o);
    }
  }
  for (int i = tid + 256 * CPT; i < n; i += 256) {
    const float o = xs[i] * rx * p.next_w[i];
    if (p.h) p.h[r * n + i] = o;
    if (p.h16) p.h16[r * n + i] = f2bf(o);
  }
}

}  // namespace lgs

extern "C" int lgs_embed_streams(const int* tokens, const void* table, int w_f32, float scale, float* x, int T, int W,
                                 int vocab, int streams, hipStream_t stream) {
  LGA_CHECK_ARG(tokens && table && x && T > 0 && W > 0 && vocab > 0, "lgs_embed_streams: bad arguments");
  LGA_CHECK_ARG(streams >= 1 && streams <= lgs::kMaxStreams, "lgs_embed_streams: 1 to 8 streams");
  const dim3 grid = lgs::embed_grid(T, W);
  if (w_f32) lgs::embed_streams_kernel<true><<<grid, 256, 0, stream>>>(tokens, table, scale, x, W, vocab, streams);
  else lgs::embed_streams_kernel<false><<<grid, 256, 0, stream>>>(tokens, table, scale, x, W, vocab, streams);
  LGA_LAUNCH_RETURN();
}

extern "C" int lgs_streams_step(float* x, const float* y, const float* mix, const float* out, const float* in,
                                const float* norm_w, float* h, void* h_bf16, float eps, int T, int W, int streams,
                                hipStream_t stream) {
  LGA_CHECK_ARG(x && T > 0 && W > 0, "lgs_streams_step: bad arguments");
  LGA_CHECK_ARG(streams >= 1 && streams <= lgs::kMaxStreams, "lgs_streams_step: 1 to 8 streams");
  LGA_CHECK_ARG(!y || (mix && out), "lgs_streams_step: a write-back needs the mix matrix and the output weights");
  LGA_CHECK_ARG(!in || h, "lgs_streams_step: a read needs a result buffer");
  LGA_CHECK_ARG(norm_w || !h_bf16, "lgs_streams_step: the bf16 copy is made by the norm");
  LGA_CHECK_ARG(y || in, "lgs_streams_step: nothing to do");
  lgs::StreamArgs p{x, y, mix, out, in, norm_w, h, (uint16_t*)h_bf16, eps, W, streams};
  bool done;
  if (streams == 1) done = lgs::streams_step_reg<1>(p, T, stream);
  else if (streams == 2) done = lgs::streams_step_reg<2>(p, T, stream);
  else if (streams <= 4) done = lgs::streams_step_reg<4>(p, T, stream);
  else done = lgs::streams_step_reg<8>(p, T, stream);
  if (!done) lgs::streams_step_kernel<<<T, 256, 0, stream>>>(p);  // wide rows: column blocks one after the other
  LGA_LAUNCH_RETURN();
}

extern "C" int lgs_streams_held(const int* tokens, const void* table, int w_f32, float scale, int vocab, const float* base,
                                float* x, const float* const* y, const float* const* mix, const float* const* out, int count,
                                const float* in, const float* norm_w, float* h, void* h_bf16, float eps, int T, int W,
                                int streams, hipStream_t stream) {
  LGA_CHECK_ARG(T > 0 && W > 0 && W <= 4096, "lgs_streams_held: rows of up to 4096 columns");
  LGA_CHECK_ARG(streams >= 2 && streams <= 4, "lgs_streams_held: 2 to 4 streams");
  LGA_CHECK_ARG((base != nullptr) != (tokens != nullptr), "lgs_streams_held: stored streams, or tokens");
  LGA_CHECK_ARG(!tokens || (table && vocab > 0), "lgs_streams_held: tokens without a table");
  LGA_CHECK_ARG(count >= (base ? 1 : 0) && count <= (base ? 3 : 2 * streams),
                "lgs_streams_held: 1 to 3 outputs on stored streams, up to 2 s on the embedding");
  LGA_CHECK_ARG(count == 0 || (y && mix && out), "lgs_streams_held: an output needs its mix matrix and weights");
  LGA_CHECK_ARG(in && (h || h_bf16) && (norm_w || !h_bf16), "lgs_streams_held: a read with a place for it (bf16: made by the norm)");
  lgs::HeldArgs p{};
  p.tokens = tokens, p.table = table, p.w_f32 = w_f32, p.vocab = vocab, p.scale = scale, p.base = base, p.x = x;
  for (int k = 0; k < count; ++k) {
    LGA_CHECK_ARG(y[k] && mix[k] && out[k], "lgs_streams_held: an output needs its mix matrix and weights");
    p.y[k] = y[k], p.mix[k] = mix[k], p.out[k] = out[k];
  }
  p.in = in, p.w = norm_w, p.h = h, p.h16 = (uint16_t*)h_bf16, p.eps = eps, p.W = W;
  bool done = false;
  if (streams == 2) done = lgs::streams_held_from<2>(p, T, count, stream);
  else if (streams == 3) done = lgs::streams_held_from<3>(p, T, count, stream);
  else done = lgs::streams_held_from<4>(p, T, count, stream);
  LGA_CHECK_ARG(done, "lgs_streams_held: no such form");
  LGA_LAUNCH_RETURN();
}

extern "C" int lgs_sandwich_step(const float* x_in, float* x, const float* y0, const float* w0, const float* y1,
                                 const float* w1, float coef, const float* post_w, const float* next_w, float* h,
                                 void* h_bf16, float eps, int rows, int n, float* hist, const float* depth_w, int n_prev,
                                 int hist_rows, const float* add, const float* add_vec, hipStream_t stream) {
  LGA_CHECK_ARG(x && rows > 0 && n > 0, "lgs_sandwich_step: bad arguments");
  LGA_CHECK_ARG(y0 || !y1, "lgs_sandwich_step: a second branch without a first");
  LGA_CHECK_ARG(y0 || next_w || depth_w || add_vec, "lgs_sandwich_step: nothing to do");
  LGA_CHECK_ARG(add_vec ? !depth_w : !add, "lgs_sandwich_step: a pass's vector (without an average over the depth), or no row");
  LGA_CHECK_ARG(!next_w || h || h_bf16, "lgs_sandwich_step: the next input needs a place");
  LGA_CHECK_ARG(!depth_w || (hist && n_prev >= 1 && n_prev <= hist_rows),
                "lgs_sandwich_step: the average over the depth needs the earlier results");
  lgs::SandwichArgs p{x_in ? x_in : x, x, y0, w0, y1, w1, coef, post_w, next_w, h, (uint16_t*)h_bf16, eps, n,
                      hist, depth_w, n_prev, hist_rows, add_vec, add};
#define LGS_SANDWICH(CPT)                                                                      \
  do {                                                                                         \
    if (depth_w) lgs::sandwich_step_kernel<CPT, true, false><<<rows, 256, 0, stream>>>(p);     \
    else if (add_vec) lgs::sandwich_step_kernel<CPT, false, true><<<rows, 256, 0, stream>>>(p); \
    else lgs::sandwich_step_kernel<CPT, false, false><<<rows, 256, 0, stream>>>(p);            \
  } while (0)
  if (n <= 1024) LGS_SANDWICH(4);
  else if (n <= 2048) LGS_SANDWICH(8);
  else LGS_SANDWICH(16);
#undef LGS_SANDWICH
  LGA_LAUNCH_RETURN();
}
