// Gated delta rule of the layered models: a per-head outer-product memory S (d x dv, fp32, one per cache slot) that is
// decayed, corrected towards the value of the current key, and read by the query:
//   S <- diag(g) S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q
// g is one number per head, or one per head and key channel (the rows of S). Query / key heads may be shared by
// groups of value heads (head h reads q / k head h / (H / G)). Everything that enters the recurrence is fp32.
// The same kernels serve the plain gated rule without the correction, S <- diag(g) S + k v^T (gated linear attention:
// u = v, no beta), whose decay is sigmoid(raw + bias)^(1 / tau) and whose q is only scaled.
//
//   lgs_delta_prepare   per token: q and k (after their convolution) become unit vectors per head, q times q_scale
//                       (or q is only scaled); beta = sigmoid(raw); g = exp(-exp(A_log) softplus(raw + dt_bias)) or
//                       sigmoid(raw + bias)^(1 / tau); k . q per key head. Steps of few rows spread the decays (each
//                       a low-rank product) over workgroups of their own
//   lgs_delta_step_prepare  the same for a step in which every sequence brings one token, with the short convolution
//                       of q | k | v (and the shift of its stored inputs) in the same launch
//   lgs_gated_delta     the recurrence, token by token for every step kind. The columns of S never mix, so a column
//                       is owned by LPC adjacent lanes that hold d / LPC of its rows in registers; the two dot
//                       products over the rows (both against the decayed state: o = S'^T q + u (k . q)) are summed
//                       inside those lanes with DPP adds (no LDS, no barrier);
//                       q, k, g, v, beta of 16 tokens at a time are staged in LDS, the next 16 prefetched in registers
//                       (8 at a time for key dims above 256)
#include <utility>

#include "gemm_tiles.h"
#include "seq_common.h"

namespace lgs {

__device__ __forceinline__ float softplus_d(float z) { return z > 20.0f ? z : log1pf(expf(z)); }

struct DeltaPrepArgs {
  float* qkv;  // [T][ld]: q [G][d] | k [G][d] | v [H][dv] after the convolution; q and k are normalised in place
  long ld;
  const float* a;  // raw decay inputs, row stride lda: [H][d] (per_channel) or [H]
  long lda;
  const float* b;  // raw beta inputs [H], row stride ldb
  long ldb;
  const float *A_log, *dt_bias;  // [H]; [H][d] or [H]
  float* dec;                    // [T][H][d] or [T][H]
  float* beta;                   // [T][H]
  float* kq;                     // [T][G]: k . q of the prepared vectors
  int H, G, d, per_channel;
  float q_scale, norm_eps;
  // optional second map of a low-rank decay input: a holds `rank` values per row and the raw input of entry i is
  // w_a2[i] . a (w_a2 [H d or H][rank], bf16 or fp32)
  const void* w_a2;
  int rank, a2_f32;
  // unit: q and k become unit vectors (0: q is only scaled, k stays as it is). decay_form 0:
  // exp(-exp(A_log) softplus(raw + dt_bias)); 1: sigmoid(raw + dt_bias)^(1 / tau) (A_log unused). b NULL: no betas.
  int unit, decay_form;
  float tau;
  // the fused one-token form only: the convolution's inputs u [B][ldu] (C = 2 G d + H dv channels), its weights
  // [C][taps] and its slot-indexed history [slots][taps - 1][C]
  const float* u;
  long ldu;
  const void* conv_w;
  int conv_f32, taps, C;
  float* conv_state;
  const int *seq_slot, *seq_pos0;
};

// the decay of one entry from its raw input z (bias added): form 0 exp(-exp(A_log[head]) softplus(z)); form 1
// sigmoid(z)^(1 / tau) = exp(-softplus(-z) / tau)
__device__ __forceinline__ float decay_of(const DeltaPrepArgs& p, float z, int head) {
  if (p.decay_form == 1) return expf(-softplus_d(-z) / p.tau);
  return expf(-expf(p.A_log[head]) * softplus_d(z));
}

// One row's preparation by a whole workgroup: wave w makes the vectors w, w + 4, ... of the 2 G query / key heads
// unit vectors; all threads walk the decays and betas; then k . q per key head.
constexpr int kMaxRank = 512;  // inner size of a low-rank second map that is folded into a consuming kernel

// part 0 of a row's work: the vectors (wave w takes the vectors w, w + 4, ...), the betas and k . q per key head;
// part y >= 1: the decays [256 (y - 1), 256 y) - with `whole` (one workgroup per row) all of them
template <bool A2F32>
__device__ __forceinline__ void delta_prepare_row(const DeltaPrepArgs& p, size_t t, int part, bool whole) {
  __shared__ float a1[kMaxRank];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int d = p.d;
  float* row = p.qkv + t * p.ld;
  if (part > 0 || whole) {
    if (p.w_a2) {
      for (int r = threadIdx.x; r < p.rank; r += 256) a1[r] = aop<A2F32>(p.a[t * p.lda + r]);
      __syncthreads();
    }
    const int dc = p.per_channel ? d : 1, n = p.H * dc;
    const int lo = whole ? 0 : 256 * (part - 1), hi = whole ? n : min(n, lo + 256);
    for (int i = lo + threadIdx.x; i < hi; i += 256) {
      const float raw = p.w_a2 ? lowrank_dot<A2F32>(p.w_a2, i, a1, p.rank) : p.a[t * p.lda + i];
      p.dec[t * n + i] = decay_of(p, raw + p.dt_bias[i], i / dc);
    }
    if (!whole) return;
  }
  for (int vec = wave; vec < 2 * p.G; vec += 4) {
    float* x = row + (size_t)vec * d;
    float s = vec < p.G ? p.q_scale : 1.0f;
    if (p.unit) {
      float ss = 0.0f;
      for (int i = lane; i < d; i += 64) ss = fmaf(x[i], x[i], ss);
      ss = wave_sum(ss);
      s = s / sqrtf(ss + p.norm_eps);
    }
    if (s != 1.0f)
      for (int i = lane; i < d; i += 64) x[i] *= s;
  }
  if (p.b)
    for (int h = threadIdx.x; h < p.H; h += 256) p.beta[t * p.H + h] = sigmoid_f(p.b[t * p.ldb + h]);
  __syncthreads();  // the prepared vectors of all heads are written
  for (int g = wave; g < p.G; g += 4) {
    const float *q = row + (size_t)g * d, *k = row + (size_t)(p.G + g) * d;
    float s = 0.0f;
    for (int i = lane; i < d; i += 64) s = fmaf(q[i], k[i], s);
    s = wave_sum(s);
    if (lane == 0) p.kq[t * p.G + g] = s;
  }
}

// grid (T), or for steps of few rows (T, 1 + ceil(n / 256)): the decays in workgroups of their own
template <bool A2F32>
__global__ void __launch_bounds__(256) delta_prepare_kernel(DeltaPrepArgs p) {
  delta_prepare_row<A2F32>(p, blockIdx.x, blockIdx.y, gridDim.y == 1);
}

// Prompts: the same numbers from more waves with fewer trips to memory. Workgroups of the first `vecs` make q and k of some (token,
// key head) pairs, a wave several side by side, and their k . q from registers; those of the next `decs` the decays of 256 entries
// of eight tokens, each row of the low-rank map read once for all eight (a workgroup per token reads all 256 KB of a map of 2048 x
// 64 for itself); the last ones 256 betas each. CPT: columns a lane holds. 2048 tokens, us for a workgroup per token / here:
// 16 heads of 128 with a decay per channel 95 / 42, 8 heads with one each 12 / 12; 200 tokens 22 / 12.
// Few heads keep the workgroup per token up to 2048 rows, its waves being as many as there is work: us there / here of 200 and 1200
// rows, 4 heads with a decay each 4.3 / 6.1, 5.4 / 6.9, 8 heads 6.1 / 6.3, 7.5 / 8.5, of a low-rank map 6.9 / 8.9, 8.5 / 11.4, 2 heads of
// 128 with a decay per channel of one 6.1 / 11.4, 13.7 / 11.8; 8 such heads 8.1 / 6.8, 12.8 / 11.5, 16 with one each 9.2 / 6.5, 11.1 /
// 11.7; 2048 rows of 4 heads 7.3 / 7.6, of 8 11.2 / 10.9.
constexpr int kPrepTokens = 8, kMapTokens = 16;
static bool prepare_rows_pay(int T, int H, int G, int d, bool per_channel, bool low_rank) {
  return T >= 2048 || (T > 64 && (per_channel ? H * d >= 1024 : G >= 16 && !low_rank));
}
// MAP: the decays' raw inputs by lowrank_tiles, 16 tokens and 256 entries a workgroup. In a prompt of 2048 tokens, 2048 entries of 64 inner
// values: a product's launch 29 us and the preparation behind it 33, here 37.
template <bool A2F32, int CPT, bool MAP>
__global__ void __launch_bounds__(256) delta_prepare_rows_kernel(DeltaPrepArgs p, int T, int vecs, int decs) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, d = p.d;
  int blk = blockIdx.x;
  if (blk < vecs) {
    constexpr int U = CPT <= 2 ? 4 : 1;  // pairs of a wave, side by side
    const long first = ((long)blk * 4 + wave) * U, end = (long)T * p.G;
    float qv[U][CPT], kv[U][CPT];
    float *q[U], *k[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const long at = min(first + u, end - 1), t = at / p.G;
      q[u] = p.qkv + t * p.ld + (size_t)(at % p.G) * d, k[u] = q[u] + (size_t)p.G * d;
#pragma unroll
      for (int c = 0; c < CPT; ++c) {
        const int i = lane + 64 * c;
        qv[u][c] = i < d ? q[u][i] : 0.0f, kv[u][c] = i < d ? k[u][i] : 0.0f;
      }
    }
    float qs[U], ks[U], dot[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float qn = 0.0f, kn = 0.0f;
      qs[u] = p.q_scale, ks[u] = 1.0f;
      if (p.unit) {
#pragma unroll
        for (int c = 0; c < CPT; ++c) qn = fmaf(qv[u][c], qv[u][c], qn), kn = fmaf(kv[u][c], kv[u][c], kn);
        qn = wave_sum(qn), kn = wave_sum(kn);
        qs[u] = qs[u] / sqrtf(qn + p.norm_eps), ks[u] = ks[u] / sqrtf(kn + p.norm_eps);
      }
      dot[u] = 0.0f;
#pragma unroll
      for (int c = 0; c < CPT; ++c) {
        qv[u][c] *= qs[u], kv[u][c] *= ks[u];
        dot[u] = fmaf(qv[u][c], kv[u][c], dot[u]);
      }
      dot[u] = wave_sum(dot[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (first + u >= end) break;
#pragma unroll
      for (int c = 0; c < CPT; ++c) {
        const int i = lane + 64 * c;
        if (i < d) q[u][i] = qv[u][c], k[u][i] = kv[u][c];
      }
      if (lane == 0) p.kq[first + u] = dot[u];
    }
    return;
  }
  blk -= vecs;
  const int dc = p.per_channel ? d : 1, n = p.H * dc;
  if (blk >= decs) {
    const long at = (long)(blk - decs) * 256 + threadIdx.x;
    if (at < (long)T * p.H) p.beta[at] = sigmoid_f(p.b[at / p.H * p.ldb + at % p.H]);
    return;
  }
  const int cols = (n + 255) / 256, i = blk % cols * 256 + threadIdx.x;
  if constexpr (MAP) {
    const int first = blk / cols * kMapTokens, i0 = blk % cols * 256 + wave * 64, fr = lane & 15, fk = lane >> 4;
    map_f32x4 raw[4];
    lowrank_tiles<4>(p.a, p.lda, first, T, (const uint16_t*)p.w_a2, i0, n, p.rank, lane, raw);
    float bias[4], rate[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = min(i0 + 16 * j + fr, n - 1);
      bias[j] = p.dt_bias[c], rate[j] = p.decay_form == 1 ? 0.0f : expf(p.A_log[c / dc]);
    }
    lga::wait_loads(bias), lga::wait_loads(rate);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = first + 4 * fk + r, c = i0 + 16 * j + fr;
        const float z = raw[j][r] + bias[j], v = p.decay_form == 1 ? decay_of(p, z, 0) : expf(-rate[j] * softplus_d(z));
        if (t < T && c < n) p.dec[(size_t)t * n + c] = v;
      }
    return;
  }
  const long t0 = (long)(blk / cols) * kPrepTokens;
  float raw[kPrepTokens];
  if (p.w_a2) {
    __shared__ __attribute__((aligned(16))) float a1[kPrepTokens][kMaxRank];
    for (int x = threadIdx.x; x < kPrepTokens * p.rank; x += 256) {
      const int u = x / p.rank, r = x % p.rank;
      a1[u][r] = aop<A2F32>(p.a[min(t0 + u, (long)T - 1) * p.lda + r]);
    }
    __syncthreads();
    if (i >= n) return;
#pragma unroll
    for (int u = 0; u < kPrepTokens; ++u) raw[u] = 0.0f;
    int r = 0;
    if ((p.rank & 7) == 0)
      for (; r < p.rank; r += 8) {
        float w[8];
        wload8<A2F32>(p.w_a2, (size_t)i * p.rank + r, w);
#pragma unroll
        for (int u = 0; u < kPrepTokens; ++u)
#pragma unroll
          for (int e = 0; e < 8; ++e) raw[u] = fmaf(a1[u][r + e], w[e], raw[u]);
      }
    for (; r < p.rank; ++r) {
      const float w = wload<A2F32>(p.w_a2, (size_t)i * p.rank + r);
#pragma unroll
      for (int u = 0; u < kPrepTokens; ++u) raw[u] = fmaf(a1[u][r], w, raw[u]);
    }
  } else {
    if (i >= n) return;
#pragma unroll
    for (int u = 0; u < kPrepTokens; ++u) raw[u] = p.a[min(t0 + u, (long)T - 1) * p.lda + i];
  }
  const float bias = p.dt_bias[i], rate = p.decay_form == 1 ? 0.0f : expf(p.A_log[i / dc]);
#pragma unroll
  for (int u = 0; u < kPrepTokens; ++u) {
    const float z = raw[u] + bias;
    if (t0 + u < T) p.dec[(t0 + u) * n + i] = p.decay_form == 1 ? decay_of(p, z, 0) : expf(-rate * softplus_d(z));
  }
}

// One channel of the short convolution for a one-token step: the weighted sum of the token's input and the slot's
// stored inputs (zeros before the sequence's start), which are shifted by one; returns silu of the sum.
template <bool WF32>
__device__ __forceinline__ float conv_step_channel(const DeltaPrepArgs& p, int b, int c, int pos0, float* st) {
  const int taps = p.taps, hist = taps - 1, C = p.C;
  const float cur = p.u[(size_t)b * p.ldu + c];
  float acc = wload<WF32>(p.conv_w, (size_t)c * taps + hist) * cur;
  float prev = cur;  // walks the history from the newest stored input to the oldest, shifting it on the way
  for (int j = hist - 1; j >= 0; --j) {
    const float x = pos0 - (hist - j) >= 0 ? st[(size_t)j * C + c] : 0.0f;
    acc = fmaf(wload<WF32>(p.conv_w, (size_t)c * taps + j), x, acc);
    st[(size_t)j * C + c] = prev;
    prev = x;
  }
  return acc / (1.0f + expf(-acc));
}

// The one-token step (every sequence brings one token; row b belongs to sequence b): convolution + silu of the
// token's q | k | v channels and the row's preparation in one launch. grid (B, G + ceil(H dv / 256) + ceil(n / 256)):
// workgroup y < G convolves and normalises q and k of key head y and leaves their k . q; the next ones convolve 256
// value channels each; the last ones make 256 decays each (the first of them also the betas).
template <bool WF32, bool A2F32>
__global__ void __launch_bounds__(256) delta_step_prepare_kernel(DeltaPrepArgs p) {
  __shared__ float buf[2 * 512];
  __shared__ float red[4];
  const int b = blockIdx.x, y = blockIdx.y, tid = threadIdx.x;
  const int d = p.d, G = p.G, C = p.C, hist = p.taps - 1;
  const int pos0 = p.seq_pos0[b];
  float* st = p.conv_state + (size_t)p.seq_slot[b] * max(hist, 1) * C;
  float* row = p.qkv + (size_t)b * p.ld;
  const int nv = C - 2 * G * d, parts_v = (nv + 255) / 256;
  if (y < G) {
    for (int i = tid; i < 2 * d; i += 256) {
      const int c = i < d ? y * d + i : (G + y) * d + (i - d);
      buf[i] = conv_step_channel<WF32>(p, b, c, pos0, st);
    }
    __syncthreads();
    float sq = 0.0f, sk = 0.0f;
    for (int i = tid; i < d; i += 256) {
      sq = fmaf(buf[i], buf[i], sq);
      sk = fmaf(buf[d + i], buf[d + i], sk);
    }
    sq = block_sum_256(sq, red);
    sk = block_sum_256(sk, red);
    const float fq = p.q_scale / sqrtf(sq + p.norm_eps), fk = 1.0f / sqrtf(sk + p.norm_eps);
    float kq = 0.0f;
    for (int i = tid; i < d; i += 256) {
      const float qn = buf[i] * fq, kn = buf[d + i] * fk;
      row[(size_t)y * d + i] = qn;
      row[(size_t)(G + y) * d + i] = kn;
      kq = fmaf(qn, kn, kq);
    }
    kq = block_sum_256(kq, red);
    if (tid == 0) p.kq[(size_t)b * G + y] = kq;
  } else if (y < G + parts_v) {
    const int c = 2 * G * d + (y - G) * 256 + tid;
    if (c < C) row[c] = conv_step_channel<WF32>(p, b, c, pos0, st);
  } else {
    const int blk = y - G - parts_v;
    const int dc = p.per_channel ? d : 1, n = p.H * dc;
    if (p.w_a2) {
      for (int r = tid; r < p.rank; r += 256) buf[r] = aop<A2F32>(p.a[(size_t)b * p.lda + r]);
      __syncthreads();
    }
    const int i = blk * 256 + tid;
    if (i < n) {
      const float raw = p.w_a2 ? lowrank_dot<A2F32>(p.w_a2, i, buf, p.rank) : p.a[(size_t)b * p.lda + i];
      p.dec[(size_t)b * n + i] = decay_of(p, raw + p.dt_bias[i], i / dc);
    }
    if (blk == 0)
      for (int h = tid; h < p.H; h += 256) p.beta[(size_t)b * p.H + h] = sigmoid_f(p.b[(size_t)b * p.ldb + h]);
  }
}

struct DeltaArgs {
  const float* qkv;  // [T][ld]: unit q [G][d] | unit k [G][d] | v [H][dv]
  long ld;
  const float* dec;   // [T][H][dc], dc = d or 1
  const float* beta;  // [T][H]
  const float* kq;    // [T][G]
  float* state;       // [slots][H][d][dv]
  const int *seq_start, *seq_slot, *seq_pos0;
  float* out;  // [T][H * dv]
  int H, G, d, dv, per_channel;
  int ncb, items;  // column blocks per head; work items = B * H * ncb
};
// DELTA false: the plain gated rule S <- diag(g) S + k v^T (u = v: no correction towards the key's value, no beta)

template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
// sum over LPC adjacent lanes (aligned, inside a row of 16 lanes); every lane of the group gets the sum. The order
// of the additions is fixed: neighbours, pairs, then the mirrored halves. Two values at once: their steps interleave.
template <int LPC>
__device__ __forceinline__ void lanes_sum2(float& a, float& b) {
  float x = dpp_f<0xB1>(a), y = dpp_f<0xB1>(b);
  a += x, b += y;
  x = dpp_f<0x4E>(a), y = dpp_f<0x4E>(b);
  a += x, b += y;
  if (LPC >= 8) {
    x = dpp_f<0x141>(a), y = dpp_f<0x141>(b);
    a += x, b += y;
  }
  if (LPC >= 16) {
    x = dpp_f<0x140>(a), y = dpp_f<0x140>(b);
    a += x, b += y;
  }
}

// grid (B * H * ceil(dv / CW) rounded up to 8), CW = 256 / LPC columns per workgroup. Lane l of a wave: r = l % LPC, column
// l / LPC of the wave's 64 / LPC; the lane holds the rows 4 (r + LPC j) + e, j < NR4, e < 4, of its column.
// ONE: sequences of one token (of more, too, but slowly): nothing is staged for tokens that do not come, and the state is on its way
// beside the rows. us, the general form / this, a decay per channel: 8 sequences of 16 heads of 128 x 128 9.3 / 7.1, 3 7.7 / 6.3, 32 19.9 /
// 15.1, 8 of 32 heads 11.0 / 8.7, 4 of 4 heads of 256 x 256 8.5 / 6.9, 3 of 512 x 64 11.8 / 10.6.
template <int NR4, int LPC, bool DELTA, bool ONE>
__global__ void __launch_bounds__(256) gated_delta_kernel(DeltaArgs p) {
  constexpr int DP = 4 * NR4 * LPC;      // rows, padded
  constexpr int CW = 256 / LPC;          // columns per workgroup
  constexpr int ROW = 3 * DP + CW + 4;   // staged floats per token: q | k | g | v | beta (rows stay 16-byte aligned)
  constexpr int kDeltaTB = ONE ? 1 : DP > 256 ? 8 : (DP > 128 ? 16 : 32);  // tokens staged at a time
  constexpr int EPT = (ROW + 255) / 256;       // staged entries per thread and token
  constexpr int KEEP = (kDeltaTB + LPC - 1) / LPC;  // outputs of a batch that a lane keeps
  __shared__ __attribute__((aligned(16))) float st[(kDeltaTB + 1) * ROW];  // (a batch's last token reads one row ahead)
  __shared__ float os[kDeltaTB][CW];
  const int tid = threadIdx.x;
  const int r = tid % LPC, cw = tid / LPC;  // cw: column inside the workgroup
  // Workgroups are dealt to the 8 XCDs in turn. The column blocks of one (sequence, head) read the same q, k and
  // decays, so consecutive work items go to ONE XCD (and its L2): item = xcd * per_xcd + turn.
  const int per_xcd = (p.items + 7) / 8;
  const int item = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (item >= p.items) return;
  const int cblk = item % p.ncb, hd = (item / p.ncb) % p.H, b = item / (p.ncb * p.H);
  const int col = cblk * CW + cw;
  const int d = p.d, dv = p.dv, H = p.H;
  const bool live = col < dv;
  const int g = hd / (H / p.G);
  // (a sequence without tokens loads the first row ahead, for nothing: its own place may be past the last one)
  const int first = p.seq_start[b], n = p.seq_start[b + 1] - first, r0 = n > 0 ? first : 0;
  const int dc = p.per_channel ? d : 1;
  float* sp = p.state + (((size_t)p.seq_slot[b] * H + hd) * d) * dv;
  const bool fresh = p.seq_pos0[b] == 0;
  float S[NR4][4];
#pragma unroll
  for (int j = 0; j < NR4; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 4 * (r + LPC * j) + e;
      if (ONE) S[j][e] = sp[(size_t)min(row, d - 1) * dv + min(col, dv - 1)];
      else S[j][e] = (!fresh && live && row < d) ? sp[(size_t)row * dv + col] : 0.0f;
    }
  // (the loads of S end here: left to the token loop's first use, every batch there would wait for the next one's loads)
  if constexpr (!ONE)
#pragma unroll
    for (int j = 0; j < NR4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(S[j][e]));
  // Entry e = tid + 256 i of a token's staged row comes from one place whatever the token: a pointer to it at the
  // sequence's first row, the distance to the next token's, and the value of an entry that has no source (padding).
  // (an entry without a source loads a valid address all the same, so that the loads carry no branches)
  const float* src[EPT];
  long step[EPT];
  float pad[EPT];
  bool has[EPT];
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    const int e = tid + 256 * i;
    src[i] = nullptr, step[i] = 0, pad[i] = 0.0f;
    if (e < 2 * DP) {  // q, then k
      const int c = e < DP ? e : e - DP;
      if (c < d) src[i] = p.qkv + (size_t)r0 * p.ld + (size_t)((e < DP ? g : p.G + g)) * d + c, step[i] = p.ld;
    } else if (e < 3 * DP) {
      const int c = e - 2 * DP;
      pad[i] = 1.0f;
      if (c < d) src[i] = p.dec + ((size_t)r0 * H + hd) * dc + (dc == 1 ? 0 : c), step[i] = (long)H * dc;
    } else if (e < 3 * DP + CW) {
      const int c = cblk * CW + (e - 3 * DP);
      if (c < dv) src[i] = p.qkv + (size_t)r0 * p.ld + (size_t)2 * p.G * d + (size_t)hd * dv + c, step[i] = p.ld;
    } else if (e == 3 * DP + CW && DELTA) {
      src[i] = p.beta + (size_t)r0 * H + hd, step[i] = H;
    } else if (e == 3 * DP + CW + 1) {
      src[i] = p.kq + (size_t)r0 * p.G + g, step[i] = p.G;
    }
    has[i] = src[i] != nullptr;
    if (!has[i]) src[i] = p.kq + (size_t)r0 * p.G + g;
  }
  float pre[kDeltaTB][EPT];
  auto prefetch = [&](int t0) {  // (past the end: the last token again)
#pragma unroll
    for (int t = 0; t < kDeltaTB; ++t)
#pragma unroll
      for (int i = 0; i < EPT; ++i) {
        pre[t][i] = *src[i];
        src[i] += t0 + t < n - 1 ? step[i] : 0;
      }
  };
  prefetch(0);
  if constexpr (ONE)
#pragma unroll
    for (int j = 0; j < NR4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (fresh || !live || 4 * (r + LPC * j) + e >= d) S[j][e] = 0.0f;

  struct Token {
    float4 k[NR4], g[NR4], q[NR4];
    float v, beta, kq;
  };
  auto fetch = [&](const float* row, Token& x) {
#pragma unroll
    for (int j = 0; j < NR4; ++j) {
      const int at = 4 * (r + LPC * j);
      x.g[j] = *(const float4*)(row + 2 * DP + at);
      x.k[j] = *(const float4*)(row + DP + at);
      x.q[j] = *(const float4*)(row + at);
    }
    x.v = row[3 * DP + cw];
    x.beta = row[3 * DP + CW];
    x.kq = row[3 * DP + CW + 1];
  };
  // With S' = diag(g) S the output is o = S'^T q + u (k . q): both products with S' run side by side and share one
  // round of lane sums, and the write S' + k u^T leaves the output's dependent chain. Four partial sums per product
  // keep the chains short.
  auto one = [&](auto&& g_at, auto&& k_at, auto&& q_at, float v, float beta, float kq) {
    float4 k4[NR4];
    float ka = 0.0f, kb = 0.0f, kc = 0.0f, kd = 0.0f, oa = 0.0f, ob = 0.0f, oc = 0.0f, od = 0.0f;
#pragma unroll
    for (int j = 0; j < NR4; ++j) {
      k4[j] = k_at(j);
      const float4 g4 = g_at(j), q4 = q_at(j);
      S[j][0] *= g4.x;
      S[j][1] *= g4.y;
      S[j][2] *= g4.z;
      S[j][3] *= g4.w;
      if (DELTA) {
        ka = fmaf(S[j][0], k4[j].x, ka);
        kb = fmaf(S[j][1], k4[j].y, kb);
        kc = fmaf(S[j][2], k4[j].z, kc);
        kd = fmaf(S[j][3], k4[j].w, kd);
      }
      oa = fmaf(S[j][0], q4.x, oa);
      ob = fmaf(S[j][1], q4.y, ob);
      oc = fmaf(S[j][2], q4.z, oc);
      od = fmaf(S[j][3], q4.w, od);
    }
    float ks = (ka + kb) + (kc + kd), qs = (oa + ob) + (oc + od);
    lanes_sum2<LPC>(ks, qs);
    const float u = DELTA ? beta * (v - ks) : v;
#pragma unroll
    for (int j = 0; j < NR4; ++j) {
      S[j][0] = fmaf(k4[j].x, u, S[j][0]);
      S[j][1] = fmaf(k4[j].y, u, S[j][1]);
      S[j][2] = fmaf(k4[j].z, u, S[j][2]);
      S[j][3] = fmaf(k4[j].w, u, S[j][3]);
    }
    return fmaf(u, kq, qs);
  };
  auto held = [&](const Token& x) {
    return one([&](int j) { return x.g[j]; }, [&](int j) { return x.k[j]; }, [&](int j) { return x.q[j]; }, x.v, x.beta, x.kq);
  };

  for (int t0 = 0; t0 < n; t0 += kDeltaTB) {
    const int nb = min(kDeltaTB, n - t0);
    __syncthreads();  // the previous batch's reads of st and os are done
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if (tid + 256 * i < ROW)
#pragma unroll
        for (int t = 0; t < kDeltaTB; ++t) st[t * ROW + tid + 256 * i] = has[i] ? pre[t][i] : pad[i];
    __syncthreads();
    if (t0 + kDeltaTB < n) prefetch(t0 + kDeltaTB);
    // A full batch of up to 16 rows a lane: the next token's operands are read while one is worked on, and the output of
    // every LPC-th token stays in one lane's register instead of a branch and a store per token. 2048 tokens of 16 heads
    // of 128 x 128: 438 us, one token's reads after the other's work 667; with 32 rows a lane the second set of operands
    // does not fit the registers (8 x 512 tokens of 8 heads of 256 x 256: 623 us against 462).
    if (!ONE && NR4 <= 4 && nb == kDeltaTB) {
      Token x[2];
      const float* row = st;
      fetch(row, x[0]);
      float keep[KEEP];
#pragma unroll
      for (int m = 0; m < KEEP; ++m) {
        keep[m] = 0.0f;
#pragma unroll 1
        for (int t = 0; t < (kDeltaTB < LPC ? kDeltaTB : LPC); t += 2) {
          fetch(row + ROW, x[1]);
          float o = held(x[0]);
          if (t == r) keep[m] = o;
          row += 2 * ROW;
          fetch(row, x[0]);
          o = held(x[1]);
          if (t + 1 == r) keep[m] = o;
        }
      }
#pragma unroll
      for (int m = 0; m < KEEP; ++m)
        if (m * LPC + r < kDeltaTB) os[m * LPC + r][cw] = keep[m];
    } else {
#pragma unroll 2
      for (int t = 0; t < nb; ++t) {
        const float* row = st + t * ROW;
        auto at = [&](int part, int j) { return *(const float4*)(row + part * DP + 4 * (r + LPC * j)); };
        const float o = one([&](int j) { return at(2, j); }, [&](int j) { return at(1, j); }, [&](int j) { return at(0, j); },
                            row[3 * DP + cw], row[3 * DP + CW], row[3 * DP + CW + 1]);
        if (r == 0) os[t][cw] = o;
      }
    }
    __syncthreads();
    for (int i = tid; i < nb * CW; i += 256) {
      const int t = i / CW, c = i % CW;
      if (cblk * CW + c < dv)
        p.out[(size_t)(r0 + t0 + t) * H * dv + (size_t)hd * dv + cblk * CW + c] = os[t][c];
    }
  }
  lga::wait_loads();
  if (live) {
#pragma unroll
    for (int j = 0; j < NR4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = 4 * (r + LPC * j) + e;
        if (row < d) sp[(size_t)row * dv + col] = S[j][e];
      }
  }
}

// The same recurrence for key dims of 128 with 32 lanes a column, to the bits of gated_delta_kernel<2, 16>: of the four partial
// sums per product there, ka + kb stand in one lane and kc + kd in its neighbour, whose sum is the first of the lane sums.
//
// Bound by the instructions of a lone wave on each SIMD, four clocks each, and by LDS. Three things keep a token short. The key's product is
// summed over the lanes at once, but the query's is not needed before the output: eight tokens' partial sums go through the same
// tree together, two tokens at a time in the two halves of a group of lanes, then four, then eight, which leaves every token's sum in
// lanes of its own, while the next eight tokens' chains run: an instruction's result reaches a DPP or a lane swap two instructions
// later, and those places are filled with the query's product and the tree (left to the compiler they were waits of eight clocks, five a
// token). The lanes are numbered for it: the tree's levels are, from the rows' lowest bit on, the mirrored eight, the mirrored
// sixteen, the other sixteen, neighbours and pairs, of which a DPP's bank mask tells the first two apart and a lane swap the third. The
// operands come by LDS-DMA, batches of eight tokens in a ring of six, and are read two tokens ahead, over the ends of batches too.
//
// us of 2048 tokens with heads of 128 x 128, when 32 tokens were staged through registers and every sum ran at its token / here: 16
// heads with a decay per channel 304 / 258, 8 heads with one each 271 / 235, 32 heads (two workgroups on a CU) 408 / 344; 1024 and 512
// tokens together of 16 heads 194 / 165. LDS by the lanes' 16 bytes in a row, which only DMAs of four bytes a lane can lay out: 288 of 16
// heads, 435 of 32. The reads between the sums' steps instead of ahead of them: 259 and 254. Beyond 512 workgroups (two on each CU) a
// third would wait for a whole chain, and the form of 16 lanes is the better one: 2048 tokens of 48 heads.
//
// grid (B * H * ceil(dv / 8) rounded up to 8). A column's lane p is number l of the rows 64 j + 2 l + e, j, e < 2.
// (PC: a decay per channel; otherwise it stands beside the betas.)
template <bool PC>
struct DeltaWide {
  static constexpr int D = 128, CW = 8, TB = 8, RING = 6, PARTS = PC ? 3 : 2;
  // a batch in floats: the tokens' q | k, their decays, a value of each column and token, then beta, k . q and decays by token
  static constexpr int G = TB * 2 * D, V = TB * PARTS * D, SC = V + TB * CW, SLOT = SC + (PC ? 2 : 3) * 64, LDS = RING * SLOT * 4;
  static constexpr int LOADS = PARTS + 1;  // DMAs of a wave and batch: 1 KB of q and k each of two tokens, and decays of two; values or scalars
  // more of it that nobody uses (gated_delta_wide_launch)
  static constexpr int ALONE = (kCuLds / 2 + 4096 - LDS) / 1024 * 1024;
  static_assert(2 * LDS <= kCuLds, "two on a CU");
  static_assert(2 * (LDS + ALONE) > kCuLds && LDS + ALONE + kPromptAttnLds > kCuLds, "alone on a CU");
};
typedef float delta_f2 __attribute__((ext_vector_type(2)));  // (the compiler's own: reads of HIP's would wait for every DMA)
typedef float delta_f4 __attribute__((ext_vector_type(4)));
// SIZE bytes a lane into LDS. Through a buffer resource: behind a flat-encoded load the compiler waits for every read of LDS in flight
// wherever it needs one; and what lies past the resource's bytes is not read (zeros)
template <int SIZE>
__device__ __forceinline__ void delta_dma(const void* base, int bytes, unsigned off, unsigned char* lds) {
#ifdef __HIP_DEVICE_COMPILE__  // (a device builtin: the host pass only type-checks the body)
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, bytes, 0x00020000);
  if constexpr (SIZE == 16) __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, off, 0, 0, 0);
  else __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 4, off, 0, 0, 0);
#endif
}
template <int... I, class F>
__device__ __forceinline__ void delta_steps(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N>  // until at most N of this wave's LDS operations are on their way
__device__ __forceinline__ void delta_wait_lds() {
  asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory");
}
template <bool DELTA, bool PC>
__global__ void __launch_bounds__(256) gated_delta_wide_kernel(DeltaArgs p) {
  using T = DeltaWide<PC>;
  constexpr int D = T::D, CW = T::CW, TB = T::TB, RING = T::RING, PARTS = T::PARTS, SLOT = T::SLOT;
  __shared__ __attribute__((aligned(16))) unsigned char lds[T::LDS];
  const int tid = threadIdx.x, lane = tid & 31, cw = tid >> 5, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // (lane = the levels' distances 7, 15, 16, 1, 2 by the bits of l)
  const int l = ((lane >> 2 ^ lane >> 3) & 1) | (lane >> 3 & 1) << 1 | (lane >> 4 & 1) << 2 | ((lane ^ lane >> 2) & 1) << 3 |
                ((lane >> 1 ^ lane >> 2) & 1) << 4;
  const int per_xcd = (p.items + 7) / 8;  // (a head's column blocks on one XCD, as above)
  const int item = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (item >= p.items) return;
  const int cblk = item % p.ncb, hd = (item / p.ncb) % p.H, b = item / (p.ncb * p.H);
  const int dv = p.dv, H = p.H, col = cblk * CW + cw;
  const bool live = col < dv;
  const int g = hd / (H / p.G);
  const int r0 = p.seq_start[b], n = p.seq_start[b + 1] - r0;
  float* sp = p.state + (((size_t)p.seq_slot[b] * H + hd) * D) * dv;
  const bool fresh = p.seq_pos0[b] == 0;
  auto row_of = [&](int i) { return 64 * (i >> 1) + 2 * l + (i & 1); };
  float S[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) S[i] = !fresh && live ? sp[(size_t)row_of(i) * dv + col] : 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(S[i]));  // (as above: the loads of S end here)

  // A wave brings q and k of the tokens 2 w and 2 w + 1 of a batch, their decays, and the values (wave 0), betas (1), k . q (2) or decays of a
  // head (3) of all eight. Addresses go on batch by batch; rows past the sequence's end are past the resource's bytes.
  const int lane64 = tid & 63;
  const char* qk = (const char*)(p.qkv + (size_t)r0 * p.ld + (size_t)g * D);
  const char* dec = (const char*)(p.dec + ((size_t)r0 * H + hd) * (PC ? D : 1));
  const char* few = (const char*)(p.kq + (size_t)r0 * p.G + g);
  const int ld4 = (int)p.ld * 4, dstep = H * (PC ? D : 1) * 4;
  int fstep = p.G * 4, few_end = 4;  // bytes of a row, and those read of the last one
  if (wave == 0) {
    few = (const char*)(p.qkv + (size_t)r0 * p.ld + (size_t)2 * p.G * D + (size_t)hd * dv + cblk * CW);
    fstep = ld4, few_end = 4 * min(CW, dv - cblk * CW);
  }
  if (wave == 1 && DELTA) few = (const char*)(p.beta + (size_t)r0 * H + hd), fstep = H * 4;
  if (wave == 3 && !PC) few = dec, fstep = dstep;
  const int few_to = (wave == 0 ? T::V : T::SC + (wave == 1 ? 0 : wave == 3 && !PC ? 2 : 1) * 64) * 4;
  const unsigned qk_off = (lane64 >> 5) * (unsigned)(p.G * D * 4) + 16 * (lane64 & 31);
  const unsigned g_off = (2 * wave + (lane64 >> 5)) * (unsigned)dstep + 16 * (lane64 & 31);
  const unsigned few_off = (wave == 0 ? lane64 >> 3 : lane64 & 7) * (unsigned)fstep + (wave == 0 ? 4 * (lane64 & 7) : 0);
  auto slot_at = [&](int slot) { return lds + slot * (SLOT * 4); };
  int left = n;  // rows that are not loaded yet
  auto load = [&](int slot) {
    unsigned char* to = slot_at(slot);
    const int rows = __builtin_amdgcn_readfirstlane(min(max(left, 0), TB));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int t = 2 * wave + i;
      delta_dma<16>(qk + (long)t * ld4, t < rows ? (p.G + 1) * D * 4 : 0, qk_off, to + t * 1024);
    }
    if constexpr (PC) delta_dma<16>(dec, max(rows * dstep - (dstep - D * 4), 0), g_off, to + (T::G + 2 * wave * D) * 4);
    delta_dma<4>(few, max(rows * fstep - (fstep - few_end), 0), few_off, to + few_to);
    left -= TB;
    qk += (long)TB * ld4, dec += (long)TB * dstep, few += (long)TB * fstep;
  };

  struct Token {
    delta_f2 q[2], k[2], g[2];
  };
  // A batch's vectors as this lane reads them: six addresses that the compiler cannot tell apart from strangers, or it joins two reads of 8
  // bytes into one instruction, whose two places fall on the same banks (64 clocks of four waves where two reads take 21, measured)
  struct Places {
    unsigned q[2], k[2], g[2];
  };
  auto places = [&](int slot, Places& o) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      o.q[j] = slot * (SLOT * 4) + 256 * j + 8 * l;
      o.k[j] = o.q[j] + 512;
      asm volatile("" : "+v"(o.q[j]), "+v"(o.k[j]));
      if constexpr (PC) {
        o.g[j] = slot * (SLOT * 4) + T::G * 4 + 256 * j + 8 * l;
        asm volatile("" : "+v"(o.g[j]));
      }
    }
  };
  auto fetch = [&](const Places& at, int t, Token& x) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if constexpr (PC) x.g[j] = *(const delta_f2*)(lds + at.g[j] + t * 512);
      x.k[j] = *(const delta_f2*)(lds + at.k[j] + t * 1024);
      x.q[j] = *(const delta_f2*)(lds + at.q[j] + t * 1024);
    }
  };
  auto add16 = [](float v) {
    const LanePair rows = lane_pair<16>(v);
    return rows.a + rows.b;
  };
  auto pin = [] { __builtin_amdgcn_sched_barrier(0); };
  auto here = [](float& v) { asm volatile("" : "+v"(v)); };  // (made here, not where it is used)
  // One token: the decayed state's product with the key over all lanes and, between its steps, that with the query, left as this lane's
  // share, and what `fill` does at five places; then the correction and the write. Returns u.
  auto one = [&](const Token& x, float v, float beta, float gate, float& qs, auto&& fill) {
    S[0] *= PC ? x.g[0].x : gate, S[1] *= PC ? x.g[0].y : gate, S[2] *= PC ? x.g[1].x : gate, S[3] *= PC ? x.g[1].y : gate;
    float u = v;
    if constexpr (DELTA) {
      float ks = fmaf(S[2], x.k[1].x, S[0] * x.k[0].x) + fmaf(S[3], x.k[1].y, S[1] * x.k[0].y);
      pin();
      float a = S[0] * x.q[0].x, c = S[1] * x.q[0].y;
      here(a), here(c);
      pin();
      ks += dpp_f<0x141>(ks);  // mirrored eight, then sixteen
      pin();
      a = fmaf(S[2], x.q[1].x, a), c = fmaf(S[3], x.q[1].y, c);
      here(a), here(c);
      pin();
      ks += dpp_f<0x140>(ks);
      float mate = ks;
      here(mate);  // (a copy)
      pin();
      qs = a + c;
      here(qs);
      fill(std::integral_constant<int, 0>{});
      pin();
      const LanePair rows = lane_swap<16>(ks, mate);
      ks = rows.a + rows.b;
      pin();
      fill(std::integral_constant<int, 1>{});
      fill(std::integral_constant<int, 2>{});
      pin();
      ks += dpp_f<0xB1>(ks);
      pin();
      fill(std::integral_constant<int, 3>{});
      fill(std::integral_constant<int, 4>{});
      pin();
      ks += dpp_f<0x4E>(ks);
      u = beta * (v - ks);
    } else {
      qs = fmaf(S[2], x.q[1].x, S[0] * x.q[0].x) + fmaf(S[3], x.q[1].y, S[1] * x.q[0].y);
      here(qs);
      fill(std::integral_constant<int, 0>{});
      fill(std::integral_constant<int, 1>{});
      fill(std::integral_constant<int, 2>{});
      fill(std::integral_constant<int, 3>{});
      fill(std::integral_constant<int, 4>{});
    }
    S[0] = fmaf(x.k[0].x, u, S[0]), S[1] = fmaf(x.k[0].y, u, S[1]), S[2] = fmaf(x.k[1].x, u, S[2]), S[3] = fmaf(x.k[1].y, u, S[3]);
    return u;
  };
  const int own = lane >> 2;  // of eight tokens the one whose sum this lane gets
  const long ostep = (long)H * dv * 4;
  char* out = (char*)(p.out + (size_t)r0 * H * dv + (size_t)hd * dv);
  const unsigned o_off = own * (unsigned)ostep + 4 * col;
  // eight tokens whose output is still to be made, and the tree over them in 31 steps (some empty: five to a token)
  struct Eight {
    float q[8], a[8], two[4], b[4], four[2], sum, u, kq;
  } eight;
  auto tree = [&](auto at, Eight& o) {
    constexpr int I = decltype(at)::value;
    if constexpr (I < 8) o.a[I] = o.q[I] + dpp_f<0x141>(o.q[I]), here(o.a[I]);
    else if constexpr (I < 12) o.two[I - 8] = lane_dpp<0xE4, 0xa>(o.a[2 * (I - 8)], o.a[2 * (I - 8) + 1]), here(o.two[I - 8]);
    else if constexpr (I < 16) o.b[I - 12] = o.two[I - 12] + dpp_f<0x128>(o.two[I - 12]), here(o.b[I - 12]);
    else if constexpr (I < 18) o.four[I - 16] = lane_dpp<0xE4, 0xc>(o.b[2 * (I - 16)], o.b[2 * (I - 16) + 1]), here(o.four[I - 16]);
    else if constexpr (I == 20) {
      const LanePair rows = lane_swap<16>(o.four[0], o.four[1]);
      o.sum = rows.a + rows.b, here(o.sum);
    } else if constexpr (I == 25) o.sum += dpp_f<0xB1>(o.sum), here(o.sum);
    else if constexpr (I == 30) o.sum += dpp_f<0x4E>(o.sum), here(o.sum);
  };
  auto finish = [&] {  // (out: of the tokens behind them)
    if (live) *(float*)(out - TB * ostep + o_off) = fmaf(eight.u, eight.kq, eight.sum);  // (four lanes alike)
  };

  // batch t0 is worked on in slot `slot`; the five behind it are in LDS or on their way there
  int slot = 0;
  Token x[4];
  Places at;
  float cv[8], cb[8], cg[8];
  auto scalars = [&](const unsigned char* from, int half) {  // four tokens' v, beta and decay
#pragma unroll
    for (int t = 4 * half; t < 4 * half + 4; ++t) cv[t] = *(const float*)(from + (T::V + t * CW + cw) * 4);
    if constexpr (DELTA) {
      const delta_f4 v = *(const delta_f4*)(from + (T::SC + 4 * half) * 4);
      cb[4 * half] = v.x, cb[4 * half + 1] = v.y, cb[4 * half + 2] = v.z, cb[4 * half + 3] = v.w;
    }
    if constexpr (!PC) {
      const delta_f4 v = *(const delta_f4*)(from + (T::SC + 128 + 4 * half) * 4);
      cg[4 * half] = v.x, cg[4 * half + 1] = v.y, cg[4 * half + 2] = v.z, cg[4 * half + 3] = v.w;
    }
  };
  // this wave's DMAs of the next batch have landed, and it has read all that it reads of the batch before (what it issued since are
  // the reads of the two tokens ahead); and so has everyone
  auto begin = [&] {
    lga::gemm_wait_vm<3 * T::LOADS>();
    delta_wait_lds<4 * PARTS>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  if (n > TB) {
#pragma unroll
    for (int i = 0; i < RING - 1; ++i) load(i);
    begin();
    places(0, at);
    fetch(at, 0, x[0]);
    fetch(at, 1, x[1]);
    scalars(slot_at(0), 0);
  } else if (n > 0) {
    load(0);
    lga::gemm_wait_vm<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
  bool any = false;  // eight tokens before these
#pragma unroll
  for (int i = 0; i < 8; ++i) eight.q[i] = 0.0f;
  int t0 = 0;
  auto next_slot = [&](int s) { return s == RING - 1 ? 0 : s + 1; };
  for (; t0 + TB <= n && n > TB; t0 += TB) {
    if (t0 > 0) begin();
    load(slot == 0 ? RING - 1 : slot - 1);
    const int ns = next_slot(slot);
    Places behind;
    places(ns, behind);
    float us = 0.0f, qs[8];
    const float kq_own = *(const float*)(slot_at(slot) + (T::SC + 64 + own) * 4);
    auto token = [&](auto i) {
      constexpr int I = decltype(i)::value;
      fetch(I < 6 ? at : behind, (I + 2) & 7, x[(I + 2) & 3]);
      if constexpr (I == 1) scalars(slot_at(slot), 1);
      if constexpr (I == 5) scalars(slot_at(ns), 0);
      pin();
      const float u = one(x[I & 3], cv[I], cb[I], cg[I], qs[I], [&](auto f) { tree(std::integral_constant<int, I * 5 + decltype(f)::value>{}, eight); });
      us = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(us), __float_as_int(u), 0xE4, I < 4 ? 0x5 : 0xa, 1 << (I & 3), false));
    };
    token(std::integral_constant<int, 0>{});
    token(std::integral_constant<int, 1>{});
    token(std::integral_constant<int, 2>{});
    token(std::integral_constant<int, 3>{});
    token(std::integral_constant<int, 4>{});
    token(std::integral_constant<int, 5>{});
    token(std::integral_constant<int, 6>{});
    token(std::integral_constant<int, 7>{});
    if (any) finish();
#pragma unroll
    for (int i = 0; i < 8; ++i) eight.q[i] = qs[i];
    eight.u = us, eight.kq = kq_own, any = true;
    out += TB * ostep;
    slot = ns, at = behind;
  }
  if (any) {
    delta_steps(std::make_integer_sequence<int, 31>{}, [&](auto at) { tree(at, eight); });
    finish();
  }
  if (t0 < n) {  // fewer than eight are left, or are all there are
    if (n > TB) begin();
    const unsigned char* from = slot_at(slot);
    places(slot, at);
    for (int t = 0; t < n - t0; ++t) {
      Token y;
      fetch(at, t, y);
      float qs;
      const float u = one(y, *(const float*)(from + (T::V + t * CW + cw) * 4), DELTA ? *(const float*)(from + (T::SC + t) * 4) : 0.0f,
                          PC ? 0.0f : *(const float*)(from + (T::SC + 128 + t) * 4), qs, [](auto) {});
      const float kq_t = *(const float*)(from + (T::SC + 64 + t) * 4);
      qs += dpp_f<0x141>(qs);
      qs += dpp_f<0x140>(qs);
      qs = add16(qs);
      qs += dpp_f<0xB1>(qs);
      qs += dpp_f<0x4E>(qs);
      if (live && lane == 0) *(float*)(out + (size_t)t * ostep + 4 * col) = fmaf(u, kq_t, qs);
    }
  }
  lga::gemm_wait_vm<0>();  // no DMA may outlive the workgroup's LDS
  if (live) {
#pragma unroll
    for (int i = 0; i < 4; ++i) sp[(size_t)row_of(i) * dv + col] = S[i];
  }
}

constexpr long kDeltaWideItems = 512;  // workgroups of eight columns (the figures stand above)
static void gated_delta_wide_launch(DeltaArgs p, int B, bool plain, hipStream_t stream) {
  p.ncb = (p.dv + 7) / 8;
  p.items = B * p.H * p.ncb;
  const unsigned grid = (unsigned)((p.items + 7) / 8 * 8);
  // Up to half as many workgroups as the chip has CUs: LDS that nobody uses keeps a CU from two of them and from one beside a
  // workgroup of the prompts' attention (kPromptAttnLds). The rule of 8 heads runs beside its layer's attention on another stream: with
  // 32 tokens staged at a time 354 to 424 us of 2048 tokens where they shared CUs, 274 on its own ones (235 now; a raised wave
  // priority changed nothing).
  const unsigned alone = p.items > 128 ? 0 : p.per_channel ? DeltaWide<true>::ALONE : DeltaWide<false>::ALONE;
  if (p.per_channel) {
    if (plain) gated_delta_wide_kernel<false, true><<<grid, 256, alone, stream>>>(p);
    else gated_delta_wide_kernel<true, true><<<grid, 256, alone, stream>>>(p);
  } else {
    if (plain) gated_delta_wide_kernel<false, false><<<grid, 256, alone, stream>>>(p);
    else gated_delta_wide_kernel<true, false><<<grid, 256, alone, stream>>>(p);
  }
}

template <int LPC, bool DELTA, bool ONE>
static bool gated_delta_launch(DeltaArgs p, int B, hipStream_t stream) {
  p.ncb = (p.dv + 256 / LPC - 1) / (256 / LPC);
  p.items = B * p.H * p.ncb;
  const dim3 grid((p.items + 7) / 8 * 8);
  const int nr4 = (p.d + 4 * LPC - 1) / (4 * LPC);
  if (nr4 <= 1) gated_delta_kernel<1, LPC, DELTA, ONE><<<grid, 256, 0, stream>>>(p);
  else if (nr4 <= 2) gated_delta_kernel<2, LPC, DELTA, ONE><<<grid, 256, 0, stream>>>(p);
  else if (nr4 <= 4) gated_delta_kernel<4, LPC, DELTA, ONE><<<grid, 256, 0, stream>>>(p);
  else if (nr4 <= 8) gated_delta_kernel<8, LPC, DELTA, ONE><<<grid, 256, 0, stream>>>(p);
  else return false;
  return true;
}

}  // namespace lgs

extern "C" int lgs_delta_prepare(float* qkv, long ld, const float* a, long lda, const float* b, long ldb,
                                 const float* A_log, const float* dt_bias, float* dec, float* beta, float* kq, int T,
                                 int H, int G, int d, int per_channel, float q_scale, float norm_eps, const void* w_a2,
                                 int rank, int a2_f32, int unit, int decay_form, float tau, hipStream_t stream) {
  LGA_CHECK_ARG(qkv && a && dt_bias && dec && kq && T > 0 && (!b || beta), "lgs_delta_prepare: bad arguments");
  LGA_CHECK_ARG((decay_form == 0 && A_log) || (decay_form == 1 && tau > 0.0f),
                "lgs_delta_prepare: decay form 0 needs A_log, form 1 a positive tau");
  LGA_CHECK_ARG(H > 0 && G > 0 && H % G == 0 && d > 0 && ld >= 2L * G * d, "lgs_delta_prepare: bad sizes");
  LGA_CHECK_ARG(!w_a2 || (rank > 0 && rank <= lgs::kMaxRank), "lgs_delta_prepare: inner size of the decay map 1..512");
  lgs::DeltaPrepArgs p{qkv, ld, a, lda, b, ldb, A_log, dt_bias, dec, beta, kq, H, G, d, per_channel ? 1 : 0, q_scale,
                       norm_eps, w_a2, rank, a2_f32, unit ? 1 : 0, decay_form, tau, nullptr, 0, nullptr, 0, 0, 0, nullptr,
                       nullptr, nullptr};
  const int n = per_channel ? H * d : H;
  if (d <= 512 && lgs::prepare_rows_pay(T, H, G, d, per_channel != 0, w_a2 != nullptr)) {
    const int pairs = 4 * (d <= 128 ? 4 : 1);  // of a workgroup
    const long vecs = ((long)T * G + pairs - 1) / pairs;
    const bool map = lgs::lowrank_tiles_fit(a, lda, w_a2, a2_f32, rank);
    const int tokens = map ? lgs::kMapTokens : lgs::kPrepTokens;
    const long decs = ((long)T + tokens - 1) / tokens * ((n + 255) / 256);
    const long betas = b ? ((long)T * H + 255) / 256 : 0;
    if (vecs + decs + betas < (1L << 31)) {
      const unsigned grid = (unsigned)(vecs + decs + betas);
      auto run = [&](auto* kernel) { kernel<<<grid, 256, 0, stream>>>(p, T, (int)vecs, (int)decs); };
      if (map && d <= 128) run(lgs::delta_prepare_rows_kernel<false, 2, true>);
      else if (map) run(lgs::delta_prepare_rows_kernel<false, 8, true>);
      else if (a2_f32 && d <= 128) run(lgs::delta_prepare_rows_kernel<true, 2, false>);
      else if (a2_f32) run(lgs::delta_prepare_rows_kernel<true, 8, false>);
      else if (d <= 128) run(lgs::delta_prepare_rows_kernel<false, 2, false>);
      else run(lgs::delta_prepare_rows_kernel<false, 8, false>);
      LGA_LAUNCH_RETURN();
    }
  }
  // few rows (decode): the decays - with a low-rank second map a product each - spread over workgroups of their own
  const dim3 grid(T, T <= 64 && n > 256 ? 1 + (n + 255) / 256 : 1);
  if (a2_f32) lgs::delta_prepare_kernel<true><<<grid, 256, 0, stream>>>(p);
  else lgs::delta_prepare_kernel<false><<<grid, 256, 0, stream>>>(p);
  LGA_LAUNCH_RETURN();
}

extern "C" int lgs_delta_step_prepare(const float* u, long ldu, const void* conv_w, int conv_f32, int taps,
                                      float* conv_state, const int* seq_slot, const int* seq_pos0, float* qkv,
                                      const float* a, long lda, const float* b, long ldb, const float* A_log,
                                      const float* dt_bias, float* dec, float* beta, float* kq, int B, int H, int G,
                                      int d, int dv, int per_channel, float q_scale, float norm_eps, const void* w_a2,
                                      int rank, int a2_f32, hipStream_t stream) {
  LGA_CHECK_ARG(u && conv_w && conv_state && seq_slot && seq_pos0 && qkv && a && b && A_log && dt_bias && dec && beta &&
                    kq && B > 0,
                "lgs_delta_step_prepare: bad arguments");
  LGA_CHECK_ARG(H > 0 && G > 0 && H % G == 0 && d > 0 && dv > 0 && taps >= 1 && taps <= 16,
                "lgs_delta_step_prepare: bad sizes (taps 1..16)");
  LGA_CHECK_ARG(!w_a2 || (rank > 0 && rank <= lgs::kMaxRank),
                "lgs_delta_step_prepare: inner size of the decay map 1..512");
  const int C = 2 * G * d + H * dv;
  LGA_CHECK_ARG(ldu >= C, "lgs_delta_step_prepare: channels outside the row");
  lgs::DeltaPrepArgs p{qkv, C, a, lda, b, ldb, A_log, dt_bias, dec, beta, kq, H, G, d, per_channel ? 1 : 0, q_scale,
                       norm_eps, w_a2, rank, a2_f32, 1, 0, 1.0f, u, ldu, conv_w, conv_f32, taps, C, conv_state, seq_slot,
                       seq_pos0};
  const int n = per_channel ? H * d : H;
  const dim3 grid(B, G + (H * dv + 255) / 256 + (n + 255) / 256);
  LGA_CHECK_ARG(d <= 512 && grid.y <= 65535, "lgs_delta_step_prepare: key dim <= 512");
  if (conv_f32) {
    if (a2_f32) lgs::delta_step_prepare_kernel<true, true><<<grid, 256, 0, stream>>>(p);
    else lgs::delta_step_prepare_kernel<true, false><<<grid, 256, 0, stream>>>(p);
  } else {
    if (a2_f32) lgs::delta_step_prepare_kernel<false, true><<<grid, 256, 0, stream>>>(p);
    else lgs::delta_step_prepare_kernel<false, false><<<grid, 256, 0, stream>>>(p);
  }
  LGA_LAUNCH_RETURN();
}

static int gated_delta_any(const float* qkv, long ld, const float* dec, const float* beta, const float* kq, float* state,
                           const int* seq_start, const int* seq_slot, const int* seq_pos0, float* out, int B, int H, int G, int d,
                           int dv, int per_channel, int lanes, int plain, bool one, hipStream_t stream) {
  LGA_CHECK_ARG(qkv && dec && (beta || plain) && kq && state && seq_start && seq_slot && seq_pos0 && out,
                "lgs_gated_delta: null pointer");
  LGA_CHECK_ARG(B > 0 && H > 0 && G > 0 && H % G == 0 && d > 0 && d <= 512 && dv > 0,
                "lgs_gated_delta: bad sizes (key dim <= 512)");
  LGA_CHECK_ARG(ld >= 2L * G * d + (long)H * dv, "lgs_gated_delta: q | k | v outside the row");
  LGA_CHECK_ARG((long)B * H * ((dv + 15) / 16) < (1L << 30), "lgs_gated_delta: too many columns");
  lgs::DeltaArgs p{qkv, ld, dec, beta, kq, state, seq_start, seq_slot, seq_pos0, out, H, G, d, dv, per_channel ? 1 : 0,
                   0, 0};
  // lanes per column: more lanes shorten a token's dependent chain and multiply the waves; by default as many as
  // keep the launch within about two waves per SIMD, and at least enough for 32 rows per lane
  int lpc = lanes;
  // Steps of one token take the wide form too, up to its workgroups. us of 128 x 128, wide / ONE with 16 lanes: one sequence of 1 to 16 heads 3.6
  // to 3.9 / 4.1 to 4.5; past 256 workgroups, two to a CU, three of 8 heads 4.7 / 4.3, two of 16 4.9 / 4.3, one of 32 4.8 / 4.3.
  // (even rows: only they gained; rows below 2^24 floats: eight of them are offsets of 32 bits)
  const bool pairs = ld % 2 == 0 && ld < (1 << 24) && ((uintptr_t)qkv | (uintptr_t)dec) % 8 == 0;
  if (lanes == 0 && d == 128 && pairs && (long)B * H * ((dv + 7) / 8) <= lgs::kDeltaWideItems) {
    lgs::gated_delta_wide_launch(p, B, plain != 0, stream);
    LGA_LAUNCH_RETURN();
  }
  if (lpc == 0) {
    const long cols = (long)B * H * dv;
    lpc = cols * 16 / 64 <= 2048 ? 16 : cols * 8 / 64 <= 2048 ? 8 : 4;
    while (lpc > 4 && 4 * lpc > d) lpc >>= 1;
  }
  while (lpc < 16 && d > 32 * lpc) lpc <<= 1;
  bool ok;
  auto go = [&](auto n) {
    constexpr int L = decltype(n)::value;
    if (one) return plain ? lgs::gated_delta_launch<L, false, true>(p, B, stream) : lgs::gated_delta_launch<L, true, true>(p, B, stream);
    return plain ? lgs::gated_delta_launch<L, false, false>(p, B, stream) : lgs::gated_delta_launch<L, true, false>(p, B, stream);
  };
  if (lpc == 4) ok = go(std::integral_constant<int, 4>{});
  else if (lpc == 8) ok = go(std::integral_constant<int, 8>{});
  else if (lpc == 16) ok = go(std::integral_constant<int, 16>{});
  else ok = false;
  LGA_CHECK_ARG(ok, "lgs_gated_delta: lanes per column must be 4, 8 or 16 and cover the key dim");
  LGA_LAUNCH_RETURN();
}

extern "C" int lgs_gated_delta(const float* qkv, long ld, const float* dec, const float* beta, const float* kq,
                               float* state, const int* seq_start, const int* seq_slot, const int* seq_pos0, float* out,
                               int B, int H, int G, int d, int dv, int per_channel, int lanes, int plain,
                               hipStream_t stream) {
  return gated_delta_any(qkv, ld, dec, beta, kq, state, seq_start, seq_slot, seq_pos0, out, B, H, G, d, dv, per_channel, lanes, plain,
                         false, stream);
}

extern "C" int lgs_gated_delta_one(const float* qkv, long ld, const float* dec, const float* beta, const float* kq,
                                   float* state, const int* seq_start, const int* seq_slot, const int* seq_pos0, float* out,
                                   int B, int H, int G, int d, int dv, int per_channel, int lanes, int plain,
                                   hipStream_t stream) {
  return gated_delta_any(qkv, ld, dec, beta, kq, state, seq_start, seq_slot, seq_pos0, out, B, H, G, d, dv, per_channel, lanes, plain,
                         true, stream);
}
