// Selective state-space mixer (Mamba-2 form) of the layered models; everything that enters the recurrence is fp32.
//
//   lgs_conv_silu        per-channel causal convolution over a packed batch + bias + silu; the last taps - 1 inputs
//                        of every sequence are part of its state (a slot-indexed buffer) and are read at the start
//                        of a step that continues a sequence and rewritten at its end
//   lgs_ssm_scan         per head: dt = softplus(raw + bias), a = exp(-exp(A_log) dt),
//                        S <- a S + dt B x^T (S is N x dv, fp32, one per cache slot), y = S^T C + D x;
//                        heads share B and C in groups. Token by token (decode, short portions), or for prompts
//                        in chunks of 64 tokens as fp32 matrix products with the chunks side by side
//   lgs_ssm_one          the same for steps of one token a sequence
//   lgs_ssm_walk         the same with a sequence's chunks one after another and the state in registers
//   lgs_channel_scan     the selective scan with a diagonal state matrix per channel (the Mamba form):
//                        s_n <- 2^(dt a2_n) s_n + (dt x) B_n per channel, output (s . C + D x) silu(z);
//                        token by token, or for prompts in chunks of 64 tokens side by side
//   lgs_gated_group_norm out = unit_rms_per_group(y * silu(z)) * w: gating first, the grouped norm on the gated values
#include "seq_common.h"

namespace lgs {

constexpr int kMaxTaps = 16;
constexpr int kConvTile = 16;  // tokens per workgroup (>= kMaxTaps - 1: only a sequence's first tile reads the state)

struct ConvArgs {
  const float* u;  // [T][ld] inputs (the channels start at u)
  long ld;
  const void* w;   // [C][taps]
  const void* b;   // [C]
  float* state;    // [slots][taps - 1][C]: the inputs at the last taps - 1 positions, oldest first
  const int *seq_start, *seq_slot, *seq_pos0;
  float* out;      // [T][C]
  int C, taps;
};

__device__ __forceinline__ float softplus_f(float z) { return z > 20.0f ? z : log1pf(expf(z)); }

// grid (ceil(C / 256), tiles, B): thread = channel; tile = kConvTile consecutive tokens of sequence b. The first
// tile of a sequence reads the stored inputs (unless the sequence starts at position 0: then they count as zeros)
// and, after it, writes the inputs that the step leaves behind.
template <bool WF32>
__global__ void __launch_bounds__(256) conv_silu_kernel(ConvArgs p) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  const int b = blockIdx.z;
  const int r0 = p.seq_start[b], n = p.seq_start[b + 1] - r0;
  const int first = blockIdx.y * kConvTile;
  if (c >= p.C || first >= n) return;
  const int taps = p.taps, hist = taps - 1;
  const int pos0 = p.seq_pos0[b];
  float* st = p.state + (size_t)p.seq_slot[b] * hist * p.C + c;
  // the window's last entry is the current token; weights are aligned to it (zeros in front of the first tap)
  float w[kMaxTaps], win[kMaxTaps];
#pragma unroll
  for (int k = 0; k < kMaxTaps; ++k) {
    w[kMaxTaps - 1 - k] = k < taps ? wload<WF32>(p.w, (size_t)c * taps + (taps - 1 - k)) : 0.0f;
    float v = 0.0f;  // the input k tokens before the tile's first
    if (k >= 1 && k <= hist) {
      const int src = first - k;  // relative to the sequence's first row of this step
      if (src >= 0) v = p.u[(size_t)(r0 + src) * p.ld + c];
      else if (pos0 + src >= 0) v = st[(size_t)(hist + src) * p.C];  // (first == 0 here: the stored inputs)
    }
    win[kMaxTaps - 1 - k] = v;
  }
  const float bias = wload<WF32>(p.b, c);
  const int last = min(first + kConvTile, n);
  for (int i = first; i < last; ++i) {
    win[kMaxTaps - 1] = p.u[(size_t)(r0 + i) * p.ld + c];
    float acc = bias;
#pragma unroll
    for (int j = 0; j < kMaxTaps; ++j) acc = fmaf(w[j], win[j], acc);
    p.out[(size_t)(r0 + i) * p.C + c] = acc / (1.0f + expf(-acc));
#pragma unroll
    for (int j = 0; j < kMaxTaps - 1; ++j) win[j] = win[j + 1];
  }
  if (first == 0) {
    // what the step leaves behind: the inputs at positions pos0 + n - hist + j. A stored input is read at a higher
    // index than any written before it, so ascending order works in place.
    for (int j = 0; j < hist; ++j) {
      const int src = n - hist + j;
      float v = 0.0f;
      if (src >= 0) v = p.u[(size_t)(r0 + src) * p.ld + c];
      else if (pos0 + src >= 0) v = st[(size_t)(hist + src) * p.C];
      st[(size_t)j * p.C] = v;
    }
  }
}

// The same for four taps: a tile's inputs are loaded ahead of its sums, so that a thread makes one trip to memory and not one a token,
// and a sequence's only token keeps the inputs that it leaves behind in registers. The same sums in the same order. Bound by memory
// (5.7 TB/s). us, the kernel above / this: 2407 tokens of 10240 channels 48.2 / 34.7, 2048 of 6144 25.0 / 20.6, of 3072 15.9 / 13.0,
// one of 10240 3.4 / 2.8 (without the wait ahead of the stores 70.8, 39.7, 21.3).
template <bool WF32>
__global__ void __launch_bounds__(256) conv4_silu_kernel(ConvArgs p) {
  constexpr int H = 3;
  const int c = blockIdx.x * 256 + threadIdx.x;
  const int b = blockIdx.z;
  const int r0 = p.seq_start[b], n = p.seq_start[b + 1] - r0;
  const int first = blockIdx.y * kConvTile;
  if (c >= p.C || first >= n) return;
  const int pos0 = p.seq_pos0[b], count = min(kConvTile, n - first);
  float* st = p.state + (size_t)p.seq_slot[b] * H * p.C + c;
  const float* u = p.u + (size_t)(r0 + first) * p.ld + c;
  float in[H + kConvTile], w[4];
#pragma unroll
  for (int k = 0; k < H; ++k) {  // the inputs at first - 3, - 2, - 1
    in[k] = 0.0f;
    if (first > 0) in[k] = (u - (size_t)(H - k) * p.ld)[0];
    else if (pos0 + k >= H) in[k] = st[(size_t)k * p.C];
  }
  if (count == kConvTile) {
#pragma unroll
    for (int i = 0; i < kConvTile; ++i) in[H + i] = u[(size_t)i * p.ld];
  } else {
    for (int i = 0; i < kConvTile; ++i) in[H + i] = u[(size_t)min(i, count - 1) * p.ld];
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) w[k] = wload<WF32>(p.w, (size_t)c * 4 + k);
  const float bias = wload<WF32>(p.b, c);
  float* out = p.out + (size_t)(r0 + first) * p.C + c;
  lga::wait_loads(in);  // (or every store waits for the one before)
#pragma unroll
  for (int i = 0; i < kConvTile; ++i) {
    if (i >= count) break;
    float acc = bias;
#pragma unroll
    for (int k = 0; k < 4; ++k) acc = fmaf(w[k], in[i + k], acc);
    out[(size_t)i * p.C] = acc / (1.0f + expf(-acc));
  }
  if (first > 0) return;
  // what the step leaves behind, as above
  if (n == 1) {
#pragma unroll
    for (int j = 0; j < H; ++j) st[(size_t)j * p.C] = in[j + 1];
    return;
  }
#pragma unroll
  for (int j = 0; j < H; ++j) {
    const int src = n - H + j;
    float v = in[H - 1];
    if (src >= 0) v = u[(size_t)src * p.ld];
    st[(size_t)j * p.C] = v;  // (two tokens keep the input before them)
  }
}

struct ScanArgs {
  const float* xbc;  // [T][ldx]: x (heads * dv) | B (groups * N) | C (groups * N) after the convolution
  long ldx;
  const float* dt;   // [T][ldd] raw step sizes, one per head (at dt)
  long ldd;
  const float *dt_bias, *A_log, *D;  // [heads]
  float* state;      // [slots][heads][N][dv]
  const int *seq_start, *seq_slot, *seq_pos0;
  float* y;          // [T][heads * dv]
  int heads, groups, N, dv;
};

constexpr int kScanBatch = 8;  // tokens between two barriers

// grid (ceil(dv / 64), heads, B): a workgroup owns 64 columns of one head's state; wave w owns the state rows
// [w NR, (w + 1) NR), lane = column. Tokens are taken kScanBatch at a time: every wave advances its rows through the
// batch and leaves its share of each token's output in LDS; wave 0 sums the four shares in a fixed order.
template <int NR>
__global__ void __launch_bounds__(256) ssm_scan_kernel(ScanArgs p) {
  __shared__ float part[4][kScanBatch][64];
  __shared__ float sdt[kScanBatch], sa[kScanBatch];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int hd = blockIdx.y, b = blockIdx.z;
  const int col = blockIdx.x * 64 + lane;
  const bool live = col < p.dv;
  const int N = p.N, dv = p.dv, H = p.heads;
  const int g = hd / (H / p.groups);
  const int r0 = p.seq_start[b], n = p.seq_start[b + 1] - r0;
  const int inner = H * dv;
  float* st = p.state + (((size_t)p.seq_slot[b] * H + hd) * N) * dv;
  const int n0 = wave * NR;
  float S[NR];
  const bool fresh = p.seq_pos0[b] == 0;
#pragma unroll
  for (int i = 0; i < NR; ++i) S[i] = (!fresh && live && n0 + i < N) ? st[(size_t)(n0 + i) * dv + col] : 0.0f;
  const float bias = p.dt_bias[hd], rate = expf(p.A_log[hd]), Dh = p.D[hd];
  for (int t0 = 0; t0 < n; t0 += kScanBatch) {
    const int nb = min(kScanBatch, n - t0);
    if (threadIdx.x < nb) {
      const float d = softplus_f(p.dt[(size_t)(r0 + t0 + threadIdx.x) * p.ldd + hd] + bias);
      sdt[threadIdx.x] = d;
      sa[threadIdx.x] = expf(-rate * d);
    }
    __syncthreads();
    for (int t = 0; t < nb; ++t) {
      const float* row = p.xbc + (size_t)(r0 + t0 + t) * p.ldx;
      const float d = sdt[t], a = sa[t];
      const float dx = live ? d * row[hd * dv + col] : 0.0f;
      const float* Bt = row + inner + g * N + n0;
      const float* Ct = row + inner + p.groups * N + g * N + n0;
      float acc = 0.0f;
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        if (n0 + i < N) {
          S[i] = fmaf(a, S[i], Bt[i] * dx);
          acc = fmaf(S[i], Ct[i], acc);
        }
      }
      part[wave][t][lane] = acc;
    }
    __syncthreads();
    if (wave == 0 && live) {
      for (int t = 0; t < nb; ++t) {
        const size_t r = (size_t)(r0 + t0 + t);
        const float x = p.xbc[r * p.ldx + hd * dv + col];
        const float v = (part[0][t][lane] + part[1][t][lane]) + (part[2][t][lane] + part[3][t][lane]);
        p.y[r * inner + hd * dv + col] = fmaf(Dh, x, v);
      }
    }
    // (the next batch's writes to `part` come after its first barrier, which wave 0 reaches after these reads)
  }
  lga::wait_loads(S);  // (or every store waits for the one before)
  if (live) {
#pragma unroll
    for (int i = 0; i < NR; ++i)
      if (n0 + i < N) st[(size_t)(n0 + i) * dv + col] = S[i];
  }
}

// Steps of one token a sequence, to the bits of ssm_scan_kernel: a wave takes 16 columns of a head, its lane groups the quarters of the
// rows, and everything that it needs is on its way at once (there, the step size, x, B and C, and the state come one behind the other, on a
// quarter as many compute units). Bound by latency. us, there / here: 64 heads of 128 x 64 of one
// sequence 7.0 / 3.2, of three 8.5 / 5.5, 128 heads 7.3 / 3.7. Where there are many, memory bounds both and rows of 64 bytes are the worse
// ones: eight sequences of 64 heads 10.8 / 11.9, of 128 14.4 / 19.2, so up to 1024 waves.
// grid (ceil(dv / 16), heads, B), 64 threads; VEC: N = 4 NR, rows of B and C on 16 bytes
template <int NR, bool VEC>
__global__ void __launch_bounds__(64) ssm_one_kernel(ScanArgs p) {
  const int lane = threadIdx.x, hd = blockIdx.y, b = blockIdx.z, n0 = (lane >> 4) * NR;
  const int N = p.N, dv = p.dv, H = p.heads, inner = H * dv, g = hd / (H / p.groups);
  const int col = blockIdx.x * 16 + (lane & 15), cc = min(col, dv - 1);
  const size_t r = p.seq_start[b];
  const bool fresh = p.seq_pos0[b] == 0;
  float* st = p.state + (((size_t)p.seq_slot[b] * H + hd) * N) * dv;
  const float* row = p.xbc + r * p.ldx;
  const float *Bp = row + inner + (size_t)g * N, *Cp = Bp + (size_t)p.groups * N;
  float S[NR], Bt[NR], Ct[NR];
  if constexpr (VEC) {
    typedef float four_t __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int i = 0; i < NR; i += 4) {
      const four_t bv = *(const four_t*)(Bp + n0 + i), cv = *(const four_t*)(Cp + n0 + i);
#pragma unroll
      for (int e = 0; e < 4; ++e) Bt[i + e] = bv[e], Ct[i + e] = cv[e];
    }
  } else {
#pragma unroll
    for (int i = 0; i < NR; ++i) Bt[i] = Bp[min(n0 + i, N - 1)], Ct[i] = Cp[min(n0 + i, N - 1)];
  }
  const float raw = p.dt[r * p.ldd + hd], bias = p.dt_bias[hd], rate = expf(p.A_log[hd]), Dh = p.D[hd], x = row[hd * dv + cc];
  if (fresh) {
#pragma unroll
    for (int i = 0; i < NR; ++i) S[i] = 0.0f;
  } else {
#pragma unroll
    for (int i = 0; i < NR; ++i) S[i] = st[(size_t)min(n0 + i, N - 1) * dv + cc];
  }
  const float d = softplus_f(raw + bias), a = expf(-rate * d), dx = d * x;
  float acc = 0.0f;
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    if (!VEC && n0 + i >= N) break;
    S[i] = fmaf(a, S[i], Bt[i] * dx);
    acc = fmaf(S[i], Ct[i], acc);
  }
  acc = lga::lanes_join_sum<16>(acc);  // (the quarters' sums in twos, then those)
  lga::wait_loads(S);
  if (col >= dv) return;
  if (lane < 16) p.y[r * inner + hd * dv + col] = fmaf(Dh, x, acc);
#pragma unroll
  for (int i = 0; i < NR; ++i)
    if (VEC || n0 + i < N) st[(size_t)(n0 + i) * dv + col] = S[i];
}

// The prompt form of the scan: chunks of 64 tokens as fp32 matrix products (v_mfma_f32_16x16x4_f32), all chunks of
// all sequences side by side. With l_i the running sum of log a over the chunk's tokens up to i, S0 the state at the
// chunk's start and n its token count:
//   y_i = exp(l_i) C_i^T S0 + sum_{j <= i} exp(l_i - l_j) dt_j (C_i . B_j) x_j + D x_i
//   S'  = exp(l_{n-1}) S0 + sum_j exp(l_{n-1} - l_j) dt_j B_j x_j^T
// ssd_state_kernel: the second term of S' of every chunk -> workspace, the chunk's whole decay -> wdec. ssd_carry_kernel
// turns these into the state at each chunk's start (an elementwise recurrence over the chunks, which also leaves the
// final state in the slot). ssd_out_kernel: the outputs of every chunk.
//
// Both chunk kernels, grid (B * max_chunks, heads / HPW, ceil(dv / 64)): a workgroup takes HPW heads of one group in
// turn. What the heads share stays in registers: B (or C) as the first operand of every product, and the scores C B^T.
// Of a head only x and the state are staged in LDS, loaded into registers while the head before it is worked on; two
// workgroups fit a compute unit. Four rows of the inner index at a time are one instruction: lane group q takes rows
// 16 t + 4 q + e, so that first operands are read 16 bytes at a time. N <= 128.
// Bound by memory and the fp32 matrix instruction in about equal parts: 2407 tokens of 128 heads of 128 x 64 take 97 us
// and 181 us, their bytes 50 and 70 (with one head a workgroup, and B, C and four copies of the state's loads, 286 and 717; D waited for
// where it is used, and with it every store for the one before, 202).
typedef float f32x4_t __attribute__((ext_vector_type(4)));
constexpr int kSC = 64;
constexpr int kXS = 68;      // LDS row of x, state and scores: rows 4 apart fall 16 banks apart
constexpr int kBS = 132;     // ... of B
constexpr int kTiles = 8;    // 16-row pieces of N, at most

struct SsdArgs {
  const float* xbc;
  long ldx;
  const float* dt;
  long ldd;
  const float *dt_bias, *A_log, *D;
  float* state;
  const int *seq_start, *seq_slot, *seq_pos0;
  float* y;
  float* ws;    // [B * max_chunks][heads][N][dv]
  float* wdec;  // [B * max_chunks][heads]
  int heads, groups, N, dv, max_chunks, hpw;  // hpw: heads per workgroup
};

// four values at `at`, those from `left` on are zero. VEC: they start on 16 bytes and are all there or none
template <bool VEC>
__device__ __forceinline__ float4 ssd_load4(const float* at, int left) {
  if (VEC) return left > 0 ? *(const float4*)at : make_float4(0.f, 0.f, 0.f, 0.f);
  return make_float4(left > 0 ? at[0] : 0.0f, left > 1 ? at[1] : 0.0f, left > 2 ? at[2] : 0.0f, left > 3 ? at[3] : 0.0f);
}
__device__ __forceinline__ f32x4_t ssd_mma(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// four rows' values at `at`, of 16 columns each: read for the instructions of the next four rows while those of these run (2407 tokens of
// 128 heads of 128 x 64: read as they are used, every two instructions wait for LDS first, 189 us; 181 here)
__device__ __forceinline__ void ssd_read(float (&v)[16], const float* at) {
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int c = 0; c < 4; ++c) v[e * 4 + c] = at[e * kXS + c * 16];
}
// lane i's step size d and running sum of log a up to token i, from the raw step size (0 from token n on)
__device__ __forceinline__ float ssd_decay(const SsdArgs& p, int h, int lane, int n, float raw, float* d) {
  *d = lane < n ? softplus_f(raw + p.dt_bias[h]) : 0.0f;
  float l = lane < n ? -expf(p.A_log[h]) * *d : 0.0f;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float v = __shfl_up(l, o);
    if (lane >= o) l += v;
  }
  return l;
}

template <bool VEC>
__global__ void __launch_bounds__(256) ssd_state_kernel(SsdArgs p) {
  __shared__ __attribute__((aligned(16))) float Xs[kSC * kXS];
  __shared__ float wgt[4][kSC];
  const int b = blockIdx.x / p.max_chunks, cidx = blockIdx.x % p.max_chunks;
  const int h0 = blockIdx.y * p.hpw, col0 = blockIdx.z * 64;
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 15, fk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // (matrix instructions stand in scalar branches only)
  const int tc = p.seq_start[b] + cidx * kSC, n = min(kSC, p.seq_start[b + 1] - tc);
  if (n <= 0) return;
  const int N = p.N, dv = p.dv, H = p.heads, inner = H * dv, g = h0 / (H / p.groups);
  const int tiles = (N + 15) / 16;
  // wave w: rows 16 (w + 4 i) + fr of B^T, tokens 16 t + 4 fk + e
  float ba[2][4][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = (wave + 4 * i) * 16 + fr, j = 16 * t + 4 * fk + e;
        ba[i][t][e] = row < N && j < n ? p.xbc[(size_t)(tc + j) * p.ldx + inner + (size_t)g * N + row] : 0.0f;
      }
  float4 xr[4];
  float raw = 0.0f;
  auto fetch = [&](int h) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int row = (tid >> 4) + 16 * k, c = (tid & 15) * 4;
      xr[k] = ssd_load4<VEC>(p.xbc + (size_t)(tc + min(row, n - 1)) * p.ldx + (size_t)h * dv + col0 + c,
                             row < n ? dv - col0 - c : 0);
    }
    raw = p.dt[(size_t)(tc + min(lane, n - 1)) * p.ldd + h];
  };
  fetch(h0);
  for (int h = h0; h < h0 + p.hpw; ++h) {
    float d;
    const float l = ssd_decay(p, h, lane, n, raw, &d), last = __shfl(l, n - 1);
    wgt[wave][lane] = expf(last - l) * d;
    __syncthreads();  // the head before is done with Xs
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int row = (tid >> 4) + 16 * k;
      const float w = wgt[wave][row];
      *(float4*)(Xs + row * kXS + (tid & 15) * 4) = make_float4(xr[k].x * w, xr[k].y * w, xr[k].z * w, xr[k].w * w);
    }
    if (h + 1 < h0 + p.hpw) fetch(h + 1);
    __syncthreads();
    f32x4_t s[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c) s[i][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float x = Xs[(16 * t + 4 * fk + e) * kXS + c * 16 + fr];
#pragma unroll
          for (int i = 0; i < 2; ++i) s[i][c] = ssd_mma(ba[i][t][e], x, s[i][c]);
        }
    float* out = p.ws + ((size_t)blockIdx.x * H + h) * N * dv;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      if (wave + 4 * i < tiles)
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int row = (wave + 4 * i) * 16 + fk * 4 + r, col = col0 + c * 16 + fr;
            if (row < N && col < dv) out[(size_t)row * dv + col] = s[i][c][r];
          }
    if (tid == 0 && blockIdx.z == 0) p.wdec[(size_t)blockIdx.x * H + h] = expf(last);
  }
}

template <bool VEC>
__global__ void __launch_bounds__(256, 2) ssd_out_kernel(SsdArgs p) {
  __shared__ __attribute__((aligned(16))) float Xs[kSC * kXS], Ss[kTiles * 16 * kXS], Gs[kSC * kXS];
  __shared__ float la[4][kSC], dts[4][kSC];
  static_assert(kSC * kBS <= kTiles * 16 * kXS, "B is staged where the state will be");
  const int b = blockIdx.x / p.max_chunks, cidx = blockIdx.x % p.max_chunks;
  const int h0 = blockIdx.y * p.hpw, col0 = blockIdx.z * 64;
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 15, fk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // (matrix instructions stand in scalar branches only)
  const int tc = p.seq_start[b] + cidx * kSC, n = min(kSC, p.seq_start[b + 1] - tc);
  if (n <= 0) return;
  const int N = p.N, dv = p.dv, H = p.heads, inner = H * dv, g = h0 / (H / p.groups);
  const int tiles = (N + 15) / 16;
  const float* bc = p.xbc + (size_t)tc * p.ldx + inner + (size_t)g * N;
  // wave w owns tokens 16 w .. + 15: C of row 16 w + fr, states 16 t + 4 fk + e
  const int ti = wave;
  float4 ca[kTiles];
#pragma unroll
  for (int t = 0; t < kTiles; ++t) {
    const int row = ti * 16 + fr, k = 16 * t + 4 * fk;
    ca[t] = ssd_load4<VEC>(bc + (size_t)min(row, n - 1) * p.ldx + (size_t)p.groups * N + min(k, N - 1), row < n ? N - k : 0);
  }
  for (int i = tid; i < kSC * kTiles * 4; i += 256) {
    const int row = i / (kTiles * 4), k = i % (kTiles * 4) * 4;
    *(float4*)(Ss + row * kBS + k) = ssd_load4<VEC>(bc + (size_t)min(row, n - 1) * p.ldx + min(k, N - 1), row < n ? N - k : 0);
  }
  float4 xr[4], sr[kTiles];
  float raw = 0.0f, Dn = 0.0f;
  auto fetch = [&](int h) {
    const int c = (tid & 15) * 4;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int row = (tid >> 4) + 16 * k;
      xr[k] = ssd_load4<VEC>(p.xbc + (size_t)(tc + min(row, n - 1)) * p.ldx + (size_t)h * dv + col0 + c,
                             row < n ? dv - col0 - c : 0);
    }
#pragma unroll
    for (int k = 0; k < kTiles; ++k) {
      const int row = (tid >> 4) + 16 * k;
      sr[k] = ssd_load4<VEC>(p.ws + (((size_t)blockIdx.x * H + h) * N + min(row, N - 1)) * dv + col0 + c,
                             row < N ? dv - col0 - c : 0);
    }
    raw = p.dt[(size_t)(tc + min(lane, n - 1)) * p.ldd + h];
    Dn = p.D[h];
  };
  fetch(h0);
  __syncthreads();
  f32x4_t cb[4];  // C_i . B_j of this wave's rows, j in piece tj <= ti
#pragma unroll
  for (int tj = 0; tj < 4; ++tj) cb[tj] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < kTiles; ++t) {
    if (t >= tiles) continue;
    float4 k4[4];
#pragma unroll
    for (int tj = 0; tj < 4; ++tj) k4[tj] = *(const float4*)(Ss + (tj * 16 + fr) * kBS + 16 * t + 4 * fk);
    const float av[4] = {ca[t].x, ca[t].y, ca[t].z, ca[t].w};
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int tj = 0; tj < 4; ++tj)
        if (tj <= ti) cb[tj] = ssd_mma(av[e], e == 0 ? k4[tj].x : (e == 1 ? k4[tj].y : (e == 2 ? k4[tj].z : k4[tj].w)), cb[tj]);
  }
  for (int h = h0; h < h0 + p.hpw; ++h) {
    float d;
    const float l = ssd_decay(p, h, lane, n, raw, &d), Dh = Dn;
    la[wave][lane] = l, dts[wave][lane] = d;
    __syncthreads();  // the head before is done with Xs and Ss (the first: the scores with B)
#pragma unroll
    for (int k = 0; k < 4; ++k) *(float4*)(Xs + ((tid >> 4) + 16 * k) * kXS + (tid & 15) * 4) = xr[k];
#pragma unroll
    for (int k = 0; k < kTiles; ++k) *(float4*)(Ss + ((tid >> 4) + 16 * k) * kXS + (tid & 15) * 4) = sr[k];
    if (h + 1 < h0 + p.hpw) fetch(h + 1);
    float li[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) li[r] = la[wave][ti * 16 + fk * 4 + r];
#pragma unroll
    for (int tj = 0; tj < 4; ++tj) {  // (a wave's own rows: no barrier)
      const int j = tj * 16 + fr;
      const float lj = la[wave][j], dj = dts[wave][j];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = ti * 16 + fk * 4 + r;
        if (tj <= ti) Gs[i * kXS + j] = j <= i ? cb[tj][r] * expf(li[r] - lj) * dj : 0.0f;
      }
    }
    __syncthreads();
    f32x4_t o[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) o[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto mul = [&](float4 a, const float (&v)[16]) {  // += a . four rows
      const float av[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int c = 0; c < 4; ++c) o[c] = ssd_mma(av[e], v[e * 4 + c], o[c]);
    };
    // (rows past the last are read all the same, in bounds, and not used: a read under a condition cannot be counted)
    float v[2][16];
    float4 ga[4];
    ssd_read(v[0], Ss + 4 * fk * kXS + fr);
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
      if (t + 1 < kTiles) ssd_read(v[(t + 1) & 1], Ss + (16 * (t + 1) + 4 * fk) * kXS + fr);
      else ssd_read(v[0], Xs + 4 * fk * kXS + fr);
      if (t == kTiles - 1)
#pragma unroll
        for (int u = 0; u < 4; ++u) ga[u] = *(const float4*)(Gs + (ti * 16 + fr) * kXS + 16 * u + 4 * fk);
      __builtin_amdgcn_sched_barrier(0);
      if (t < tiles) mul(ca[t], v[t & 1]);
      __builtin_amdgcn_sched_barrier(0);
    }
    static_assert(kTiles % 2 == 0, "x follows in v[0]");
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[c][r] *= expf(li[r]);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (t < 3) ssd_read(v[(t + 1) & 1], Xs + (16 * (t + 1) + 4 * fk) * kXS + fr);
      __builtin_amdgcn_sched_barrier(0);
      if (t <= ti) mul(ga[t], v[t & 1]);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = ti * 16 + fk * 4 + r, col = col0 + c * 16 + fr;
        if (i < n && col < dv)
          p.y[(size_t)(tc + i) * inner + (size_t)h * dv + col] = fmaf(Dh, Xs[i * kXS + c * 16 + fr], o[c][r]);
      }
  }
}

// grid (B, heads, ceil(N dv / 256)): one state element per thread walks its sequence's chunks: the workspace's local
// sums become the states at the chunks' starts, and the state after the last chunk goes back to the slot
__global__ void __launch_bounds__(256) ssd_carry_kernel(SsdArgs p) {
  const int b = blockIdx.x, h = blockIdx.y;
  const int e = blockIdx.z * 256 + threadIdx.x;
  const int nd = p.N * p.dv;
  if (e >= nd) return;
  const int chunks = (p.seq_start[b + 1] - p.seq_start[b] + kSC - 1) / kSC;
  float* st = p.state + ((size_t)p.seq_slot[b] * p.heads + h) * nd + e;
  float s = p.seq_pos0[b] > 0 ? *st : 0.0f;
  for (int c = 0; c < chunks; ++c) {
    const size_t idx = ((size_t)b * p.max_chunks + c) * p.heads + h;
    const float local = p.ws[idx * nd + e];
    p.ws[idx * nd + e] = s;
    s = fmaf(p.wdec[idx], s, local);
  }
  *st = s;
}

// The prompt form with the chunks one after another: a workgroup walks a sequence through 64 columns of one head with the state in
// registers, so that no chunk's state goes to memory. Wave w owns columns 16 w .. + 15 and all NT * 16 rows. With rows 16 t + 4 q + e in
// lane group q a matrix instruction's result is laid out as its operands are read: the state's accumulators are the operand of C S, x is
// loaded in the layout of the outputs and serves the scores' product, and the scores (B C^T, made once a group by
// ssd_scores_kernel) become the operand of theirs. C and B of a chunk are staged in LDS while the chunk before is worked on. The sums
// stand in the order of the kernels above, so the results have their bits.
// Bound by the fp32 matrix instruction: 296 of 32 clocks a chunk and wave for N = 128, two thirds of the time it takes (6.1 us a chunk
// and workgroup). 1500 + 777 + 130 tokens of 128 heads of 128 x 64 take 177 us, the three kernels above 340 (their chunks' states are
// 640 MB written and read); four times 500 tokens of 64 heads 65 against 110; one chunk 16 to 19 against 24 to 29 whatever the heads.
// With operands read as late as the instruction group before 180, with everything a chunk needs loaded and written at the start of a half
// 188, with decays and scores' exponentials made by every wave 240, with row offsets held in registers (and spilled) 450.
struct WalkArgs {
  SsdArgs s;
  float* scores;  // [B * max_chunks][groups][10][64][4]
  float* decays;  // [B * max_chunks][heads][4][64]: l, d, exp(l_last - l) d, exp(l)
};
constexpr int kScoreTiles = 10;  // 16 x 16 pieces (ti, tj), tj <= ti, at ti (ti + 1) / 2 + tj

// grid (B * max_chunks, groups + ceil(heads / 4)): the scores of a group, or the decays of four heads, a wave each
template <int NT>
__global__ void __launch_bounds__(256) ssd_scores_kernel(WalkArgs a) {
  const SsdArgs& p = a.s;
  const int b = blockIdx.x / p.max_chunks, cidx = blockIdx.x % p.max_chunks, g = blockIdx.y;
  const int lane = threadIdx.x & 63, fr = lane & 15, fk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tc = p.seq_start[b] + cidx * kSC, n = min(kSC, p.seq_start[b + 1] - tc);
  if (n <= 0) return;
  if (g >= p.groups) {
    const int h = (g - p.groups) * 4 + wave;
    if (h >= p.heads) return;
    float d;
    const float l = ssd_decay(p, h, lane, n, p.dt[(size_t)(tc + min(lane, n - 1)) * p.ldd + h], &d), last = __shfl(l, n - 1);
    float* out = a.decays + ((size_t)blockIdx.x * p.heads + h) * 4 * kSC + lane;
    out[0] = l, out[kSC] = d, out[2 * kSC] = expf(last - l) * d, out[3 * kSC] = expf(l);
    if (lane == 0) p.wdec[(size_t)blockIdx.x * p.heads + h] = expf(last);
    return;
  }
  const float* bc = p.xbc + (size_t)tc * p.ldx + (size_t)p.heads * p.dv + (size_t)g * p.N + 4 * fk;
  float4* out = (float4*)a.scores + ((size_t)blockIdx.x * p.groups + g) * kScoreTiles * 64 + lane;
  for (int i = wave; i < kScoreTiles; i += 4) {
    const int ti = i >= 6 ? 3 : (i >= 3 ? 2 : (i >= 1 ? 1 : 0)), tj = i - ti * (ti + 1) / 2;
    const int ri = ti * 16 + fr, rj = tj * 16 + fr;
    const float* bj = bc + (size_t)min(rj, n - 1) * p.ldx;
    const float* ci = bc + (size_t)min(ri, n - 1) * p.ldx + (size_t)p.groups * p.N;
    float4 bv[NT], cv[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      bv[t] = ssd_load4<true>(bj + 16 * t, rj < n ? 4 : 0);
      cv[t] = ssd_load4<true>(ci + 16 * t, ri < n ? 4 : 0);
    }
    f32x4_t s = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      s = ssd_mma(bv[t].x, cv[t].x, s);
      s = ssd_mma(bv[t].y, cv[t].y, s);
      s = ssd_mma(bv[t].z, cv[t].z, s);
      s = ssd_mma(bv[t].w, cv[t].w, s);
    }
    out[i * 64] = make_float4(s[0], s[1], s[2], s[3]);
  }
}

// grid (heads, ceil(dv / 64), B)
template <int NT>
__global__ void __launch_bounds__(256, 2) ssd_walk_kernel(WalkArgs a) {
  constexpr int N = NT * 16, LS = N + 4, KV = NT * 4, LD = kSC * KV / 256;  // KV: 16-byte pieces of a row, LD: of a thread
  __shared__ __attribute__((aligned(16))) float Cs[kSC * LS], Bs[kSC * LS], Gs[12 * 256];  // (two pieces of Gs are not read)
  __shared__ __attribute__((aligned(16))) float el[kSC], wgt[kSC];
  const SsdArgs& p = a.s;
  const int H = p.heads, dv = p.dv, b = blockIdx.z, inner = H * dv;
  // an XCD takes neighbouring heads, which share B and C
  const int h = H % 8 == 0 ? (blockIdx.x % 8) * (H / 8) + blockIdx.x / 8 : blockIdx.x;
  const int g = h / (H / p.groups);
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 15, fk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r0 = __builtin_amdgcn_readfirstlane(p.seq_start[b]), len = __builtin_amdgcn_readfirstlane(p.seq_start[b + 1]) - r0;
  const int col = blockIdx.y * 64 + wave * 16 + fr;
  const bool live = col < dv;
  const float Dh = p.D[h];
  // a chunk's rows through buffer descriptors that end after its last row: rows past it read as zeros and are not written. Addresses
  // are a step after the one before (as multiples of the row they would be held in registers, and spilled)
  auto rows = [&](const float* base, int ld, int n) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, n * ld * 4, 0x00020000);
  };
  auto step = [](unsigned& at, unsigned by) {
    at += by;
    asm volatile("" : "+v"(at));
  };
  const int ldx = (int)p.ldx;
  constexpr unsigned dead = 0x7ffffff0;  // (past every descriptor's end, with 64 rows added too)
  const unsigned at_bc = ((tid / KV) * ldx + tid % KV * 4) * 4, at_x = live ? (4 * fk * ldx + col) * 4 : dead;
  const unsigned at_y = live ? (4 * fk * inner + col) * 4 : dead;
  f32x4_t cr[LD], br[LD], sc[3], lj[3], dj[3];
  float x[16], li[3], dec = 0.0f, whole = 0.0f;
  const float *Bp = p.xbc + inner + (size_t)g * N, *Cp = Bp + (size_t)p.groups * N, *Xp = p.xbc + (size_t)h * dv;
  auto chunk_of = [&](const float* from, int c) { return rows(from + (size_t)(r0 + c * kSC) * ldx, ldx, min(kSC, len - c * kSC)); };
  auto fetch_row = [&](f32x4_t& v, const auto& rs, unsigned& at) {  // a piece of a chunk's B or C
    v = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, at, 0, 0));
    step(at, 256 / KV * 4 * ldx);
  };
  auto fetch_x = [&](int k, const auto& rs, unsigned& at) {  // token 16 (k / 4) + 4 fk + k % 4
    x[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, at, 0, 0));
    step(at, (k % 4 == 3 ? 13 : 1) * 4 * ldx);
  };
  // this wave's pieces of the scores (ti, tj) = wave, wave + 4, wave + 8 and what decays them
  auto piece = [&](int k, int& ti, int& tj) {
    const int i = min(wave + 4 * k, kScoreTiles - 1);
    ti = i >= 6 ? 3 : (i >= 3 ? 2 : (i >= 1 ? 1 : 0)), tj = i - ti * (ti + 1) / 2;
    return i;
  };
  auto fetch_score = [&](int k, size_t at) {
    const f32x4_t* from = (const f32x4_t*)a.scores + (at * p.groups + g) * kScoreTiles * 64;
    const float* de = a.decays + (at * H + h) * 4 * kSC;
    int ti, tj;
    const int i = piece(k, ti, tj);
    sc[k] = (from + i * 64)[(unsigned)lane];
    li[k] = (de + ti * 16)[(unsigned)fr];
    lj[k] = ((const f32x4_t*)(de + tj * 16))[(unsigned)fk];
    dj[k] = ((const f32x4_t*)(de + kSC + tj * 16))[(unsigned)fk];
  };
  auto fetch_decay = [&](size_t at) {
    dec = (a.decays + ((at * H + h) * 4 + 2) * kSC)[(unsigned)(tid & 127)];
    whole = p.wdec[at * H + h];
  };
  auto decay_scores = [&](int k) {  // in place
    int ti, tj;
    piece(k, ti, tj);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float v = sc[k][r] * expf(li[k] - lj[k][r]) * dj[k][r];
      sc[k][r] = ti > tj || 4 * fk + r <= fr ? v : 0.0f;
    }
  };
  // the state at the sequence's start: zeros (a descriptor that ends before its first value) at position 0
  f32x4_t S[NT];
  const int slot = __builtin_amdgcn_readfirstlane(p.seq_slot[b]), old = __builtin_amdgcn_readfirstlane(p.seq_pos0[b]) > 0;
  float* st = p.state + ((size_t)slot * H + h) * N * dv;
  const auto sr = rows(st, dv, old ? N : 0);
  const unsigned at_s = live ? (4 * fk * dv + col) * 4 : dead;
  {
    unsigned at = at_s;
#pragma unroll
    for (int k = 0; k < 4 * NT; ++k) {
      S[k / 4][k % 4] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(sr, at, 0, 0));
      step(at, (k % 4 == 3 ? 13 : 1) * 4 * dv);
    }
  }
  const int chunks = (len + kSC - 1) / kSC;
  auto put_row = [&](float* to, const f32x4_t& v, int k) {
    const int i = tid + 256 * k;
    *(f32x4_t*)(to + i / KV * LS + i % KV * 4) = v;
  };
  auto put_scores = [&](int k) {
    decay_scores(k);
    *(f32x4_t*)(Gs + ((wave + 4 * k) * 64 + lane) * 4) = sc[k];
  };
  auto put_el = [&]() {
    if (tid >= kSC && tid < 2 * kSC) el[tid - kSC] = dec;
  };
  const size_t at0 = (size_t)b * p.max_chunks;
  if (chunks > 0) {
    const auto bs = chunk_of(Bp, 0), cs = chunk_of(Cp, 0);
    unsigned ab = at_bc, ac = at_bc;
#pragma unroll
    for (int k = 0; k < 3; ++k) fetch_score(k, at0);
    fetch_decay(at0);
#pragma unroll
    for (int k = 0; k < LD; ++k) fetch_row(cr[k], cs, ac), fetch_row(br[k], bs, ab);
#pragma unroll
    for (int k = 0; k < LD; ++k) put_row(Cs, cr[k], k);
    put_el();
#pragma unroll
    for (int k = 0; k < 3; ++k) put_scores(k);
  }
  // Of a chunk, C and the scores are read before the middle barrier and B after it: the next chunk's are written in the other half.
  // Loads and writes stand one or two behind every four matrix instructions (all together at the start of a half, the matrix cores
  // waited for their issue). The next chunk's loads are those of this one again where it is the last: under a condition they could
  // not be counted, and would be waited for as one.
  for (int c = 0; c < chunks; ++c) {
    const int next = min(c + 1, chunks - 1);
    const auto xs = chunk_of(Xp, c), cs = chunk_of(Cp, next), bs = chunk_of(Bp, next);
    const auto ys = rows(p.y + (size_t)(r0 + c * kSC) * inner + (size_t)h * dv, inner, min(kSC, len - c * kSC));
    unsigned ax = at_x, ac = at_bc, ab = at_bc, ay = at_y;
    f32x4_t o[4], ca[2][4];
#pragma unroll
    for (int ti = 0; ti < 4; ++ti) o[ti] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const float held = whole;
    __syncthreads();
    auto read_c = [&](f32x4_t& v, int t, int ti) { v = *(const f32x4_t*)(Cs + (ti * 16 + fr) * LS + 16 * t + 4 * fk); };
    auto read_g = [&](f32x4_t& v, int tj, int ti) {
      if (ti >= tj) v = *(const f32x4_t*)(Gs + ((ti * (ti + 1) / 2 + tj) * 64 + lane) * 4);
    };
#pragma unroll
    for (int ti = 0; ti < 4; ++ti) read_c(ca[0][ti], 0, ti);
    if (tid < kSC) wgt[tid] = dec;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * t + e;
        if (e == 0)
#pragma unroll
          for (int ti = 0; ti < 4; ++ti) {
            if (t + 1 < NT) read_c(ca[(t + 1) & 1][ti], t + 1, ti);
            else read_g(ca[(t + 1) & 1][ti], 0, ti);
          }
#pragma unroll
        for (int ti = 0; ti < 4; ++ti) o[ti] = ssd_mma(ca[t & 1][ti][e], S[t][e], o[ti]);
        if (i < 8) fetch_x(2 * i, xs, ax), fetch_x(2 * i + 1, xs, ax);
        if (i < LD) put_row(Bs, br[i], i);
        if (i >= 8 && i < 8 + LD) fetch_row(cr[i - 8], cs, ac);
        if (i >= 4 * NT - 4 && i < 4 * NT - 1) fetch_score(i - 4 * NT + 4, at0 + next);
        if (i == 4 * NT - 1) fetch_decay(at0 + next);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
    for (int ti = 0; ti < 4; ++ti) {
      const f32x4_t e = *(const f32x4_t*)&el[ti * 16 + 4 * fk];
#pragma unroll
      for (int r = 0; r < 4; ++r) o[ti][r] *= e[r];
    }
    static_assert(NT % 2 == 0, "the scores follow in ca[0]");
#pragma unroll
    for (int tj = 0; tj < 4; ++tj)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (tj < 3 && e == 0)
#pragma unroll
          for (int ti = 0; ti < 4; ++ti) read_g(ca[(tj + 1) & 1][ti], tj + 1, ti);
#pragma unroll
        for (int ti = 0; ti < 4; ++ti)
          if (ti >= tj) o[ti] = ssd_mma(ca[tj & 1][ti][e], x[tj * 4 + e], o[ti]);
        __builtin_amdgcn_sched_barrier(0);
      }
    __syncthreads();
    // the state: this chunk's sum onto the decayed state before it
    f32x4_t s[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) s[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float bv[2][NT];
    auto read_b = [&](float (&v)[NT], int k) {
#pragma unroll
      for (int t = 0; t < NT; ++t) v[t] = Bs[(16 * (k >> 2) + 4 * fk + (k & 3)) * LS + 16 * t + fr];
    };
    read_b(bv[0], 0);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const f32x4_t w = *(const f32x4_t*)&wgt[16 * u + 4 * fk];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[u][e] = fmaf(Dh, x[u * 4 + e], o[u][e]);
        x[u * 4 + e] *= w[e];
      }
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      if (k + 1 < 16) read_b(bv[(k + 1) & 1], k + 1);
#pragma unroll
      for (int t = 0; t < NT / 2; ++t) s[t] = ssd_mma(bv[k & 1][t], x[k], s[t]);
      if (k % 4 != 3) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = NT / 2; t < NT; ++t) s[t] = ssd_mma(bv[k & 1][t], x[k], s[t]);
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o[k / 4][k % 4]), ys, ay, 0, 0);
      step(ay, (k % 4 == 3 ? 13 : 1) * 4 * inner);
      if (k < LD) {
        put_row(Cs, cr[k], k);
        fetch_row(br[k], bs, ab);
      }
      if (k == 8) put_el();
      if (k % 4 == 3 && k < 12) {  // the next chunk's scores in the gaps of the matrix instructions
        put_scores(k / 4);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 96 / NT, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[t][r] = fmaf(held, S[t][r], s[t][r]);
  }
  const auto sw = rows(st, dv, N);
  unsigned at = at_s;
#pragma unroll
  for (int k = 0; k < 4 * NT; ++k) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(S[k / 4][k % 4]), sw, at, 0, 0);
    step(at, (k % 4 == 3 ? 13 : 1) * 4 * dv);
  }
}

template <int NT>
static void ssd_walk_launch(const WalkArgs& a, int B, hipStream_t stream) {
  ssd_scores_kernel<NT><<<dim3(B * a.s.max_chunks, a.s.groups + (a.s.heads + 3) / 4), 256, 0, stream>>>(a);
  ssd_walk_kernel<NT><<<dim3(a.s.heads, (a.s.dv + 63) / 64, B), 256, 0, stream>>>(a);
}

// ------------------------------------------------------------------------------------------------ channel scan
// Selective scan with a step size per channel and a diagonal state matrix (channels x N): nothing is shared between
// channels but B and C, and every (channel, state) pair decays at a rate of its own, so the work is
// elementwise: L lanes of a wave share one channel, each with NR of its N states in registers, and sum the output
// with shuffles. Lanes of one wave that hold the same states lie side by side, so that every access to the state, the
// inputs and the outputs is 64 / L consecutive floats. Tokens are taken kChanBatch at a time: the batch's x, z and step
// sizes are fetched into registers, its B and C rows into LDS.
// MODE 0, grid (blocks, 1, B): every sequence token by token from its stored state, outputs and final state.
// The prompt form runs chunks of kChanChunk tokens side by side, grid (blocks, max_chunks, B): MODE 1 leaves every
// chunk's state from a zero start in ws and the sum of its step sizes in wsum; channel_carry_kernel turns these into the
// state at each chunk's start (the decay over a chunk is exp(A sum dt)) and leaves the final state in the slot;
// MODE 2 walks every chunk from its start state and makes the outputs.
struct ChanArgs {
  const float* x;   // [T][inner]
  const float* z;   // [T][ldz]
  long ldz;
  const float* bc;  // [T][ldbc]: dt inner values (rank) | B (N) | C (N)
  long ldbc;
  int rank;
  const float* dt;  // [T][ldt] raw step sizes with their bias (null: w_dt)
  long ldt;
  const void* w_dt;  // [inner][rank]
  const float* dt_bias;
  const float* a2;   // [N][inner]
  const float* D;
  float* state;      // [slots][N][inner]
  const int *seq_start, *seq_slot, *seq_pos0;
  float* out;        // [T][inner]
  uint16_t* out16;   // instead of out
  int inner, N;
  float *ws, *wsum;
  int max_chunks;
};

constexpr int kChanChunk = 64, kChanBatch = 8;

template <int L, int NR, int MODE, bool LOWRANK, bool WF32>
__global__ void __launch_bounds__(256) channel_scan_kernel(ChanArgs p) {
  extern __shared__ float lds[];  // [kChanBatch][2 NP] B | C of the batch's tokens; LOWRANK: then [kChanBatch][rank]
  constexpr int NP = L * NR, CW = 64 / L;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int part = lane / CW, c = (blockIdx.x * 4 + wave) * CW + lane % CW;
  const int b = blockIdx.z, N = p.N, inner = p.inner;
  const bool live = c < inner;
  const int r0 = p.seq_start[b], n_seq = p.seq_start[b + 1] - r0;
  const int first = MODE == 0 ? 0 : blockIdx.y * kChanChunk;
  if (first >= n_seq) return;
  const int last = MODE == 0 ? n_seq : min(n_seq, first + kChanChunk);
  const size_t slot = p.seq_slot[b], chunk = (size_t)b * p.max_chunks + blockIdx.y;
  const int n0 = part * NR;
  float S[NR], a2[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const bool in = live && n0 + i < N;
    const size_t at = (size_t)(n0 + i) * inner + c;
    a2[i] = in ? p.a2[at] : 0.0f;
    S[i] = 0.0f;
    if (MODE == 0 && in && p.seq_pos0[b] > 0) S[i] = p.state[slot * N * inner + at];
    if (MODE == 2 && in) S[i] = p.ws[chunk * N * inner + at];
  }
  const float Dc = live ? p.D[c] : 0.0f;
  const float bias = (LOWRANK && live) ? p.dt_bias[c] : 0.0f;
  float dsum = 0.0f;
  float* dlow = lds + kChanBatch * 2 * NP;
  for (int t0 = first; t0 < last; t0 += kChanBatch) {
    const int nb = min(kChanBatch, last - t0);
    float xv[kChanBatch], zv[kChanBatch], dv[kChanBatch];
#pragma unroll
    for (int t = 0; t < kChanBatch; ++t) {
      const size_t r = (size_t)(r0 + t0 + t);
      const bool in = live && t < nb;
      xv[t] = in ? p.x[r * inner + c] : 0.0f;
      zv[t] = (MODE != 1 && in) ? p.z[r * p.ldz + c] : 0.0f;
      dv[t] = (!LOWRANK && in) ? p.dt[r * p.ldt + c] : 0.0f;
    }
    __syncthreads();  // the previous batch's rows are read
    for (int i = tid; i < nb * 2 * NP; i += 256) {
      const int t = i / (2 * NP), e = i % (2 * NP), half = e / NP, n = e % NP;
      lds[i] = n < N ? p.bc[(size_t)(r0 + t0 + t) * p.ldbc + p.rank + half * N + n] : 0.0f;
    }
    if (LOWRANK)
      for (int i = tid; i < nb * p.rank; i += 256)
        dlow[i] = aop<WF32>(p.bc[(size_t)(r0 + t0 + i / p.rank) * p.ldbc + i % p.rank]);
    __syncthreads();
#pragma unroll
    for (int t = 0; t < kChanBatch; ++t) {
      if (t >= nb) break;
      float d = dv[t];
      if (LOWRANK) {  // the channel's lanes share its row of the step-size map
        float acc = 0.0f;
        if (live) {
          const float* xr = dlow + t * p.rank;
          if ((p.rank & 7) == 0) {
            for (int r = 8 * part; r < p.rank; r += 8 * L) {
              float u[8];
              wload8<WF32>(p.w_dt, (size_t)c * p.rank + r, u);
#pragma unroll
              for (int e = 0; e < 8; ++e) acc = fmaf(xr[r + e], u[e], acc);
            }
          } else {
            for (int r = part; r < p.rank; r += L) acc = fmaf(xr[r], wload<WF32>(p.w_dt, (size_t)c * p.rank + r), acc);
          }
        }
        acc = lanes_join_sum<CW>(acc);
        d = acc + bias;
      }
      d = softplus_f(d);
      const float* Bt = lds + t * 2 * NP + n0;
      const float dx = d * xv[t];
      float acc = 0.0f;
      if (MODE == 1) dsum += d;
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        S[i] = fmaf(__builtin_amdgcn_exp2f(d * a2[i]), S[i], Bt[i] * dx);
        if (MODE != 1) acc = fmaf(S[i], Bt[NP + i], acc);
      }
      if (MODE != 1) {
        acc = lanes_join_sum<CW>(acc);
        if (part == 0 && live) {
          const float zz = zv[t];
          const float v = fmaf(Dc, xv[t], acc) * (zz / (1.0f + expf(-zz)));
          const size_t at = (size_t)(r0 + t0 + t) * inner + c;
          if (p.out16) p.out16[at] = f2bf(v);
          else p.out[at] = v;
        }
      }
    }
  }
  if (MODE == 2 || !live) return;
  float* dst = MODE == 0 ? p.state + slot * N * inner : p.ws + chunk * N * inner;
#pragma unroll
  for (int i = 0; i < NR; ++i)
    if (n0 + i < N) dst[(size_t)(n0 + i) * inner + c] = S[i];
  if (MODE == 1 && part == 0) p.wsum[chunk * inner + c] = dsum;
}

// grid (ceil(N inner / 256), B): per (state, channel) the recurrence over the chunks of a sequence
__global__ void __launch_bounds__(256) channel_carry_kernel(ChanArgs p) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x, ni = (size_t)p.N * p.inner;
  if (i >= ni) return;
  const int b = blockIdx.y, c = (int)(i % p.inner);
  const int n_seq = p.seq_start[b + 1] - p.seq_start[b], chunks = (n_seq + kChanChunk - 1) / kChanChunk;
  float* st = p.state + (size_t)p.seq_slot[b] * ni + i;
  const float a2 = p.a2[i];
  float S = p.seq_pos0[b] > 0 ? *st : 0.0f;
#pragma unroll 4
  for (int k = 0; k < chunks; ++k) {
    const size_t chunk = (size_t)b * p.max_chunks + k;
    float* w = p.ws + chunk * ni + i;
    const float local = *w;
    *w = S;
    S = fmaf(__builtin_amdgcn_exp2f(p.wsum[chunk * p.inner + c] * a2), S, local);
  }
  *st = S;
}

template <int L, int NR>
static int channel_scan_launch(const ChanArgs& p, int w_f32, int B, hipStream_t stream) {
  constexpr int CB = 4 * (64 / L);  // channels per workgroup
  const dim3 one((p.inner + CB - 1) / CB, 1, B);
  size_t lds = sizeof(float) * kChanBatch * 2 * L * NR;
  if (p.w_dt) {
    lds += sizeof(float) * kChanBatch * p.rank;
    if (w_f32) channel_scan_kernel<L, NR, 0, true, true><<<one, 256, lds, stream>>>(p);
    else channel_scan_kernel<L, NR, 0, true, false><<<one, 256, lds, stream>>>(p);
  } else if (!p.ws) {
    channel_scan_kernel<L, NR, 0, false, true><<<one, 256, lds, stream>>>(p);
  } else {
    const dim3 grid(one.x, p.max_chunks, B);
    channel_scan_kernel<L, NR, 1, false, true><<<grid, 256, lds, stream>>>(p);
    const size_t ni = (size_t)p.N * p.inner;
    channel_carry_kernel<<<dim3((unsigned)((ni + 255) / 256), B), 256, 0, stream>>>(p);
    channel_scan_kernel<L, NR, 2, false, true><<<grid, 256, lds, stream>>>(p);
  }
  return 0;
}

// grid (T, groups): out[t][g n + i] = v / sqrt(mean_g(v^2) + eps) * w[g n + i], v = y * silu(z)
__global__ void __launch_bounds__(256) gated_group_norm_kernel(const float* __restrict__ y, const float* __restrict__ z,
                                                               long ldz, const float* __restrict__ w, float eps,
                                                               float* __restrict__ out, uint16_t* __restrict__ out16,
                                                               int n, int inner) {
  __shared__ float red[4];
  const size_t t = blockIdx.x;
  const int c0 = blockIdx.y * n;
  float ss = 0.0f;
  for (int i = threadIdx.x; i < n; i += 256) {
    const float zz = z[t * ldz + c0 + i];
    const float v = y[t * inner + c0 + i] * (zz / (1.0f + expf(-zz)));
    out[t * inner + c0 + i] = v;
    ss = fmaf(v, v, ss);
  }
  ss = block_sum_256(ss, red);
  const float rstd = 1.0f / sqrtf(ss / (float)n + eps);
  for (int i = threadIdx.x; i < n; i += 256) {
    const float v = out[t * inner + c0 + i] * rstd * w[c0 + i];
    out[t * inner + c0 + i] = v;
    if (out16) out16[t * inner + c0 + i] = f2bf(v);
  }
}

// The same for groups of up to 256 NV columns: the values stay in registers, where the kernel above writes `out`, reads it again and
// writes it twice; beside a bf16 copy `out` may be null. The same sums in the same order. us, the kernel above / this: 2407 tokens of 8
// groups of 1024, bf16 alone 76.4 / 29.9, 2000 of 4 of 2048, fp32 49.8 / 30.2, 2048 of 8 of 512 26.5 / 17.4, one token 2.6 / 2.2.
template <int NV>
__global__ void __launch_bounds__(256) gated_group_norm_reg_kernel(const float* __restrict__ y, const float* __restrict__ z,
                                                                   long ldz, const float* __restrict__ w, float eps,
                                                                   float* __restrict__ out, uint16_t* __restrict__ out16,
                                                                   int n, int inner) {
  __shared__ float red[4];
  const size_t t = blockIdx.x;
  const int c0 = blockIdx.y * n;
  float yv[NV], zv[NV], wv[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int i = c0 + min((int)threadIdx.x + 256 * k, n - 1);
    yv[k] = y[t * inner + i], zv[k] = z[t * ldz + i], wv[k] = w[i];
  }
  float ss = 0.0f;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    yv[k] *= zv[k] / (1.0f + expf(-zv[k]));
    if ((int)threadIdx.x + 256 * k < n) ss = fmaf(yv[k], yv[k], ss);
  }
  ss = block_sum_256(ss, red);
  const float rstd = 1.0f / sqrtf(ss / (float)n + eps);
  lga::wait_loads(wv);  // (or every store waits for the one before)
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int i = threadIdx.x + 256 * k;
    if (i >= n) break;
    const float v = yv[k] * rstd * wv[k];
    if (out) out[t * inner + c0 + i] = v;
    if (out16) out16[t * inner + c0 + i] = f2bf(v);
  }
}

}  // namespace lgs

extern "C" int lgs_conv_silu(const float* u, long ld, const void* w, const void* bias, int w_f32, float* state,
                             const int* seq_start, const int* seq_slot, const int* seq_pos0, float* out, int B,
                             int max_len, int C, int taps, hipStream_t stream) {
  LGA_CHECK_ARG(u && w && bias && state && seq_start && seq_slot && seq_pos0 && out, "lgs_conv_silu: null pointer");
  LGA_CHECK_ARG(B > 0 && B <= 65535 && max_len > 0 && C > 0 && ld >= C, "lgs_conv_silu: bad sizes");
  LGA_CHECK_ARG(taps >= 1 && taps <= lgs::kMaxTaps, "lgs_conv_silu: 1 to 16 taps");
  lgs::ConvArgs p{u, ld, w, bias, state, seq_start, seq_slot, seq_pos0, out, C, taps};
  const int tiles = (max_len + lgs::kConvTile - 1) / lgs::kConvTile;
  LGA_CHECK_ARG(tiles <= 65535, "lgs_conv_silu: a sequence brings too many tokens to one step");
  const dim3 grid((C + 255) / 256, tiles, B);
  if (taps == 4) {
    if (w_f32) lgs::conv4_silu_kernel<true><<<grid, 256, 0, stream>>>(p);
    else lgs::conv4_silu_kernel<false><<<grid, 256, 0, stream>>>(p);
  } else if (w_f32) lgs::conv_silu_kernel<true><<<grid, 256, 0, stream>>>(p);
  else lgs::conv_silu_kernel<false><<<grid, 256, 0, stream>>>(p);
  LGA_LAUNCH_RETURN();
}

extern "C" int lgs_ssm_scan(const float* xbc, long ldx, const float* dt, long ldd, const float* dt_bias,
                            const float* A_log, const float* D, float* state, const int* seq_start,
                            const int* seq_slot, const int* seq_pos0, float* y, int B, int heads, int groups, int N,
                            int dv, float* ws, float* wdec, int max_chunks, hipStream_t stream) {
  LGA_CHECK_ARG(xbc && dt && dt_bias && A_log && D && state && seq_start && seq_slot && seq_pos0 && y,
                "lgs_ssm_scan: null pointer");
  LGA_CHECK_ARG(B > 0 && B <= 65535 && heads > 0 && heads <= 65535 && groups > 0 && heads % groups == 0,
                "lgs_ssm_scan: heads must be a multiple of the groups");
  LGA_CHECK_ARG(N > 0 && N <= 256 && dv > 0, "lgs_ssm_scan: state size 1 to 256");
  LGA_CHECK_ARG(ldx >= (long)heads * dv + 2L * groups * N && ldd >= heads, "lgs_ssm_scan: rows shorter than their parts");
  if (ws) {  // the prompt form
    LGA_CHECK_ARG(wdec && max_chunks > 0 && N <= 128, "lgs_ssm_scan: the prompt form serves state sizes up to 128");
    LGA_CHECK_ARG((long)B * max_chunks < (1L << 31) && (dv + 63) / 64 <= 65535, "lgs_ssm_scan: too many chunks");
    lgs::SsdArgs p{xbc, ldx, dt, ldd, dt_bias, A_log, D, state, seq_start, seq_slot, seq_pos0, y, ws, wdec,
                   heads, groups, N, dv, max_chunks, 1};
    // heads per workgroup: up to four share the scores, as long as two workgroups for every compute unit are left
    const int per_group = heads / groups;
    while (p.hpw < 4 && per_group % (p.hpw * 2) == 0 && (long)B * max_chunks * heads / (p.hpw * 2) >= 512) p.hpw *= 2;
    const dim3 grid(B * max_chunks, heads / p.hpw, (dv + 63) / 64);
    const bool vec = N % 4 == 0 && dv % 4 == 0 && ldx % 4 == 0 && ((uintptr_t)xbc | (uintptr_t)ws) % 16 == 0;
    if (vec) lgs::ssd_state_kernel<true><<<grid, 256, 0, stream>>>(p);
    else lgs::ssd_state_kernel<false><<<grid, 256, 0, stream>>>(p);
    lgs::ssd_carry_kernel<<<dim3(B, heads, (N * dv + 255) / 256), 256, 0, stream>>>(p);
    if (vec) lgs::ssd_out_kernel<true><<<grid, 256, 0, stream>>>(p);
    else lgs::ssd_out_kernel<false><<<grid, 256, 0, stream>>>(p);
    LGA_LAUNCH_RETURN();
  }
  lgs::ScanArgs p{xbc, ldx, dt, ldd, dt_bias, A_log, D, state, seq_start, seq_slot, seq_pos0, y, heads, groups, N, dv};
  const dim3 grid((dv + 63) / 64, heads, B);
  const int nr = (N + 3) / 4;
  if (nr <= 8) lgs::ssm_scan_kernel<8><<<grid, 256, 0, stream>>>(p);
  else if (nr <= 16) lgs::ssm_scan_kernel<16><<<grid, 256, 0, stream>>>(p);
  else if (nr <= 32) lgs::ssm_scan_kernel<32><<<grid, 256, 0, stream>>>(p);
  else lgs::ssm_scan_kernel<64><<<grid, 256, 0, stream>>>(p);
  LGA_LAUNCH_RETURN();
}

extern "C" int lgs_ssm_one(const float* xbc, long ldx, const float* dt, long ldd, const float* dt_bias, const float* A_log,
                           const float* D, float* state, const int* seq_start, const int* seq_slot, const int* seq_pos0,
                           float* y, int B, int heads, int groups, int N, int dv, hipStream_t stream) {
  LGA_CHECK_ARG(xbc && dt && dt_bias && A_log && D && state && seq_start && seq_slot && seq_pos0 && y,
                "lgs_ssm_one: null pointer");
  LGA_CHECK_ARG(B > 0 && B <= 65535 && heads > 0 && heads <= 65535 && groups > 0 && heads % groups == 0,
                "lgs_ssm_one: heads must be a multiple of the groups");
  LGA_CHECK_ARG(N > 0 && N <= 128 && dv > 0, "lgs_ssm_one: state size 1 to 128");
  LGA_CHECK_ARG(ldx >= (long)heads * dv + 2L * groups * N && ldd >= heads, "lgs_ssm_one: rows shorter than their parts");
  lgs::ScanArgs p{xbc, ldx, dt, ldd, dt_bias, A_log, D, state, seq_start, seq_slot, seq_pos0, y, heads, groups, N, dv};
  const dim3 grid((dv + 15) / 16, heads, B);
  const bool vec = ldx % 4 == 0 && (heads * dv) % 4 == 0 && (uintptr_t)xbc % 16 == 0;
  const int nr = (N + 3) / 4;
  if (vec && N == 128) lgs::ssm_one_kernel<32, true><<<grid, 64, 0, stream>>>(p);
  else if (vec && N == 64) lgs::ssm_one_kernel<16, true><<<grid, 64, 0, stream>>>(p);
  else if (nr <= 8) lgs::ssm_one_kernel<8, false><<<grid, 64, 0, stream>>>(p);
  else if (nr <= 16) lgs::ssm_one_kernel<16, false><<<grid, 64, 0, stream>>>(p);
  else lgs::ssm_one_kernel<32, false><<<grid, 64, 0, stream>>>(p);
  LGA_LAUNCH_RETURN();
}

extern "C" int lgs_ssm_walk(const float* xbc, long ldx, const float* dt, long ldd, const float* dt_bias,
                            const float* A_log, const float* D, float* state, const int* seq_start,
                            const int* seq_slot, const int* seq_pos0, float* y, int B, int heads, int groups, int N,
                            int dv, float* ws, int max_chunks, hipStream_t stream) {
  LGA_CHECK_ARG(xbc && dt && dt_bias && A_log && D && state && seq_start && seq_slot && seq_pos0 && y && ws,
                "lgs_ssm_walk: null pointer");
  LGA_CHECK_ARG(B > 0 && B <= 65535 && heads > 0 && groups > 0 && heads % groups == 0 && groups + (heads + 3) / 4 <= 65535,
                "lgs_ssm_walk: heads must be a multiple of the groups");
  LGA_CHECK_ARG((N == 64 || N == 128) && dv > 0 && (dv + 63) / 64 <= 65535, "lgs_ssm_walk: state size 64 or 128");
  LGA_CHECK_ARG(ldx >= (long)heads * dv + 2L * groups * N && ldd >= heads, "lgs_ssm_walk: rows shorter than their parts");
  LGA_CHECK_ARG(ldx < (1L << 22) && ldd < (1L << 22), "lgs_ssm_walk: 64 rows are more than 32 bits address");
  LGA_CHECK_ARG(dv % 4 == 0 && ldx % 4 == 0 && ((uintptr_t)xbc | (uintptr_t)ws) % 16 == 0, "lgs_ssm_walk: rows in 16 bytes");
  LGA_CHECK_ARG(max_chunks > 0 && (long)B * max_chunks < (1L << 31), "lgs_ssm_walk: too many chunks");
  const size_t chunks = (size_t)B * max_chunks;
  float* decays = ws + chunks * groups * lgs::kScoreTiles * 256;
  lgs::WalkArgs a{{xbc, ldx, dt, ldd, dt_bias, A_log, D, state, seq_start, seq_slot, seq_pos0, y, nullptr,
                   decays + chunks * heads * 4 * lgs::kSC, heads, groups, N, dv, max_chunks, 1}, ws, decays};
  if (N == 128) lgs::ssd_walk_launch<8>(a, B, stream);
  else lgs::ssd_walk_launch<4>(a, B, stream);
  LGA_LAUNCH_RETURN();
}

extern "C" int lgs_channel_scan(const float* x, const float* z, long ldz, const float* bc, long ldbc, int rank,
                                const float* dt_raw, long ldt, const void* w_dt, int w_f32, const float* dt_bias,
                                const float* a2, const float* D, float* state, const int* seq_start, const int* seq_slot,
                                const int* seq_pos0, void* out, int out_bf16, int B, int inner, int N, float* ws,
                                float* wsum, int max_chunks, hipStream_t stream) {
  LGA_CHECK_ARG(x && z && bc && a2 && D && state && seq_start && seq_slot && seq_pos0 && out,
                "lgs_channel_scan: null pointer");
  LGA_CHECK_ARG(B > 0 && B <= 65535 && inner > 0 && N > 0 && N <= 256 && rank > 0, "lgs_channel_scan: state size 1 to 256");
  LGA_CHECK_ARG(ldz >= inner && ldbc >= (long)rank + 2L * N, "lgs_channel_scan: rows shorter than their parts");
  LGA_CHECK_ARG((dt_raw && !w_dt && ldt >= inner) || (!dt_raw && w_dt && dt_bias && rank <= 1024),
                "lgs_channel_scan: raw step sizes, or their low-rank map (rank <= 1024) and bias");
  LGA_CHECK_ARG(!ws || (wsum && dt_raw && max_chunks > 0 && max_chunks <= 65535),
                "lgs_channel_scan: the prompt form needs both workspaces and the step sizes");
  lgs::ChanArgs p{x, z, ldz, bc, ldbc, rank, dt_raw, ldt, w_dt, dt_bias, a2, D, state, seq_start, seq_slot, seq_pos0,
                  out_bf16 ? nullptr : (float*)out, out_bf16 ? (uint16_t*)out : nullptr, inner, N, ws, wsum, max_chunks};
  int rc;
  if (ws) {  // many chunks fill the chip: up to 16 states per lane
    if (N <= 8) rc = lgs::channel_scan_launch<1, 8>(p, w_f32, B, stream);
    else if (N <= 16) rc = lgs::channel_scan_launch<1, 16>(p, w_f32, B, stream);
    else if (N <= 32) rc = lgs::channel_scan_launch<2, 16>(p, w_f32, B, stream);
    else if (N <= 64) rc = lgs::channel_scan_launch<4, 16>(p, w_f32, B, stream);
    else if (N <= 128) rc = lgs::channel_scan_launch<8, 16>(p, w_f32, B, stream);
    else rc = lgs::channel_scan_launch<16, 16>(p, w_f32, B, stream);
  } else {  // few tokens: more lanes per channel
    if (N <= 4) rc = lgs::channel_scan_launch<1, 4>(p, w_f32, B, stream);
    else if (N <= 8) rc = lgs::channel_scan_launch<2, 4>(p, w_f32, B, stream);
    else if (N <= 16) rc = lgs::channel_scan_launch<4, 4>(p, w_f32, B, stream);
    else if (N <= 32) rc = lgs::channel_scan_launch<8, 4>(p, w_f32, B, stream);
    else if (N <= 64) rc = lgs::channel_scan_launch<16, 4>(p, w_f32, B, stream);
    else rc = lgs::channel_scan_launch<16, 16>(p, w_f32, B, stream);
  }
  if (rc) return rc;
  LGA_LAUNCH_RETURN();
}

extern "C" int lgs_gated_group_norm(const float* y, const float* z, long ldz, const float* w, float eps, float* out,
                                    void* out_bf16, int T, int inner, int groups, hipStream_t stream) {
  LGA_CHECK_ARG(y && z && w && (out || out_bf16) && T > 0 && inner > 0, "lgs_gated_group_norm: bad arguments");
  LGA_CHECK_ARG(groups > 0 && groups <= 65535 && inner % groups == 0,
                "lgs_gated_group_norm: inner must divide into the groups");
  const int n = inner / groups;
  LGA_CHECK_ARG(out || n <= 2048, "lgs_gated_group_norm: a bf16 result alone is made in groups of up to 2048 columns");
  const dim3 grid(T, groups);
  auto run = [&](auto* kernel) { kernel<<<grid, 256, 0, stream>>>(y, z, ldz, w, eps, out, (uint16_t*)out_bf16, n, inner); };
  if (n <= 256) run(lgs::gated_group_norm_reg_kernel<1>);
  else if (n <= 512) run(lgs::gated_group_norm_reg_kernel<2>);
  else if (n <= 1024) run(lgs::gated_group_norm_reg_kernel<4>);
  else if (n <= 2048) run(lgs::gated_group_norm_reg_kernel<8>);
  else run(lgs::gated_group_norm_kernel);
  LGA_LAUNCH_RETURN();
}
