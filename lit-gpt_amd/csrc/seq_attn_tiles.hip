// Prompt attention of the layered models on the bf16 matrix cores, with the results of fp32 products: every fp32
// operand is the exact sum of bf16 summands (the upper 8 bits of its significand, the next 8, the last 8), products of
// bf16 values are exact in fp32, and all sums are fp32. Queries and weights have three summands beside keys and values
// that are bf16 themselves (a cache); keys and values in two summands (16 bits of their significands) meet two of the
// query and three of the weight.
//
// A workgroup of 8 waves takes 32 queries (or 64, 128) of the heads that share one key head; key tiles of 64 positions
// stream through LDS (range-checked LDS-DMA, ST stages: rows past the last visible key arrive as zeros) once for all of
// them. Per 32 keys a wave forms S^T = K Q^T (A: key rows from LDS, B: the query summands in registers), so that a lane
// holds the scores of one query: maximum, normaliser and rescale are its own. The weights' summands are the B operand of
// O^T += V^T P^T as they stand: the transposed LDS reads of V take the keys in the order in which a lane holds them.
// Unless eight (head, map) pairs share the keys, two waves split every key tile and are merged at the end.
//
// Error against float64 beside the thread-per-key form's (rms over the sizes of the tests): 0.5 to 0.9 of it with one map, 0.5
// to 0.85 with two. The two-summand form's operands are less than fp32 (the query's two summands are cut at 16 bits, keys and
// values rounded at 16 or 17, the product of both second summands is left out), in rotated parts too, which the latent form
// multiplies in fp32; but that form rounds queries and weighted latents to bf16: the heads' outputs are 5e-6 to 1.8e-5 off
// float64 here and 1.5e-3 to 3.4e-3 there, with rotated parts that outweigh the others 6e-6 and 1.5e-3.
//
// The two-summand form serves latent attention: expanded keys of 192 and values of 128, 4096 tokens of 16 heads in 372 us
// (205 TFLOP/s of fp32-like products) with 26 us for the summands and 20 for the expansion; the fp32 tiles in the latent
// space took 7.7 ms (2176 operations per pair and head instead of 640, at a sixteenth of the bf16 rate).
//
// Bound by latency inside a wave (scores -> maximum -> exponentials -> weights), then by the matrix cores' rate at three
// times the products that bf16 operands would take.
#include "seq_attn.h"

namespace lgs {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef short i16x8_t __attribute__((ext_vector_type(8)));

constexpr int kTileKeys = 64;
constexpr long kMostRow = 1 << 23;  // elements of a position's keys or values: a tile of them is one buffer (31 bits of bytes)

// 16-byte chunk `ch` of row `row` in an LDS tile of `chunks` a row: permuted so that neither 32 rows' same chunk nor the
// transposed reads meet in a bank
__device__ __forceinline__ int chunk_swizzle(int row, int chunks) {
  return chunks == 8 ? (((row & 3) << 1) | ((row >> 2) & 1)) : (((row & 3) << 2) | ((row >> 2) & 3));
}

// 16 bytes a lane of a buffer into LDS, zeros past its end
__device__ __forceinline__ void tile_dma16(const void* base, int bytes, int off, unsigned char* lds) {
#ifdef __HIP_DEVICE_COMPILE__  // (device builtins: the host pass only type-checks the body)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, bytes, 0x00020000),
                                           (__attribute__((address_space(3))) void*)lds, 16, off, 0, 0, 0);
#endif
}

// the next summands of eight fp32 values as one operand: the upper half of every value, which is taken off it
__device__ __forceinline__ bf16x8_t take_summand(float (&x)[8]) {
  u32x4_t o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t a = __float_as_uint(x[2 * e]), b = __float_as_uint(x[2 * e + 1]);
    o[e] = __builtin_amdgcn_perm(b, a, 0x07060302u);
    x[2 * e] -= __uint_as_float(a & 0xFFFF0000u);
    x[2 * e + 1] -= __uint_as_float(b & 0xFFFF0000u);
  }
  return __builtin_bit_cast(bf16x8_t, o);
}

// e^x for x <= 0: 2^t for the rounded product, times the rounding's own power. 3.6e-8 rms and 1.4e-7 at most off float64,
// where expf has 2.6e-8 and 8.3e-8; whole rows are nearer to float64 than those of the thread-per-key form with expf (0.5 to
// 0.9 of its error over the sizes of the tests), whose scores are one long chain of fp32 sums
__device__ __forceinline__ float exp_neg(float x) {
  const float t = x * 1.44269502f;
  float r = fmaf(x, 1.44269502f, -t);
  r = fmaf(x, 1.92596299e-8f, r);
  const float e = __builtin_amdgcn_exp2f(t);
  return fmaf(e, r * 0.69314718f, e);
}

// tanh x: below 0.625 the odd polynomial of the Cephes library's tanhf, above 1 - 2 e^-2|x| / (1 + e^-2|x|). Errors against
// float64 (rms): 3.6e-8 in [0.625, 1], 1.9e-8 in [1, 3], where tanhf has 3.8e-8 and 1.9e-8. (An infinite x gives NaN, and its
// row goes to attn_row_plain.)
__device__ __forceinline__ float tanh_near(float x) {
  const float z = x * x, y = fabsf(x);
  float p = fmaf(-5.70498872745e-3f, z, 2.06390887954e-2f);
  p = fmaf(p, z, -5.37397155531e-2f);
  p = fmaf(p, z, 1.33314422036e-1f);
  p = fmaf(p, z, -3.33332819422e-1f);
  p = fmaf(p * z, x, x);
  const float e = exp_neg(-2.0f * y), d = 1.0f + e;
  const float r = __builtin_amdgcn_rcpf(d), q = fmaf(-2.0f * e, fmaf(fmaf(-d, r, 1.0f), r, r), 1.0f);
  return y < 0.625f ? p : copysignf(q, x);
}

// 1 / (1 + e^-z) from e^-|z| (3.8e-8 rms for z >= 0, 5.5e-8 below; sigmoid_f 3.8e-8), which is 0 from 120 on (an infinite z has
// no residual in exp_neg; a NaN stays one)
__device__ __forceinline__ float sigmoid_near(float z) {
  const float e = exp_neg(fabsf(z) > 120.0f ? -120.0f : -fabsf(z)), d = 1.0f + e;
  const float r = __builtin_amdgcn_rcpf(d), p = fmaf(fmaf(-d, r, 1.0f), r, r);
  return z >= 0.0f ? p : e * p;
}

// A row of a head whose result is not finite, once more in fp32 by one wave: an infinite operand has no summands (inf - inf)
// and an infinite value or a NaN meets weights that are 0, also those of the keys that its query does not see. A lane scores
// every 64th visible key, then owns DV / 64 columns. Left to itself: about 0.1 ms for 4096 keys; rows of finite operands never
// come here.
template <int DC, int DT, int MAPS, int PARTS, bool SIG>
__device__ __forceinline__ void attn_row_plain(const AttnTileArgs& p, const uint16_t* kbase, const uint16_t* vbase,
                                               const float* q, int h, int qlo, int qpos, int lane, float* out) {
  constexpr int D = DC * 16, DV = DT * 32, C = DV / 64;
  const AttnArgs& a = p.a;
  float o[C], m = -INFINITY, l = 0.0f;
#pragma unroll
  for (int map = 0; map < MAPS; ++map) {
    auto score = [&](int key) {
      const uint16_t* k = kbase + (size_t)min(key, qpos) * p.krow + map * D;
      float s = 0.0f;
#pragma unroll 1
      for (int e = 0; e < D; e += 4) {
        const float4 q4 = *(const float4*)(q + map * D + e);
        const uint2 hi = *(const uint2*)(k + e);
        float x[4] = {bflo(hi.x), bfhi(hi.x), bflo(hi.y), bfhi(hi.y)};
        if (PARTS == 2) {
          const uint2 lo = *(const uint2*)(k + D + e);
          x[0] += bflo(lo.x), x[1] += bfhi(lo.x), x[2] += bflo(lo.y), x[3] += bfhi(lo.y);
        }
        s = fmaf(q4.w, x[3], fmaf(q4.z, x[2], fmaf(q4.y, x[1], fmaf(q4.x, x[0], s))));
      }
      s *= a.scale;
      return a.cap > 0.0f ? a.cap * tanhf(s / a.cap) : s;
    };
    m = -INFINITY, l = 0.0f;
    if (!SIG) {
      for (int k0 = qlo; k0 <= qpos; k0 += 64) {
        const float s = score(k0 + lane);
        m = fmaxf(m, k0 + lane <= qpos ? s : -INFINITY);
      }
      m = wave_max(m);
    }
    float acc[C];
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] = 0.0f;
    for (int k0 = qlo; k0 <= qpos; k0 += 64) {
      const float s = score(k0 + lane);
      float w = 0.0f;
      if (k0 + lane <= qpos) w = SIG ? sigmoid_f(s + a.score_bias[h]) : (m == -INFINITY ? 0.0f : expf(s - m));
      l += w;
      for (int j = 0; j < min(64, qpos - k0 + 1); ++j) {
        const float wj = __shfl(w, j);
        const uint16_t* v = vbase + (size_t)(k0 + j) * p.vrow + lane;
#pragma unroll
        for (int c = 0; c < C; ++c)
          acc[c] = fmaf(wj, PARTS == 2 ? bf2f(v[c * 64]) + bf2f(v[DV + c * 64]) : bf2f(v[c * 64]), acc[c]);
      }
    }
    l = wave_sum(l);
#pragma unroll
    for (int c = 0; c < C; ++c) o[c] = MAPS == 1 ? acc[c] : (map == 0 ? acc[c] / l : o[c] - a.lambda * (acc[c] / l));
  }
  float f = a.post, den = 1.0f;
  if (MAPS == 2) {
    float ss = 0.0f;
#pragma unroll
    for (int c = 0; c < C; ++c) ss = fmaf(o[c], o[c], ss);
    den = sqrtf(wave_sum(ss) / (float)DV + a.eps);
  } else if (!SIG) {
    den = l;
    if (a.sink) {
      const float snk = a.sink[h], top = fmaxf(m, snk), w = m == -INFINITY ? 0.0f : expf(m - top);
      den = l * w + expf(snk - top);
      f *= w;
    }
  }
#pragma unroll
  for (int c = 0; c < C; ++c) out[lane + c * 64] = o[c] / den * f;
}

// DC: 16-wide pieces of one map's key, DT: 32-wide pieces of a value, MAPS: maps per head, PARTS: summands of keys and
// values, SIG: sigmoid weights, ST: stages. grid (B * tiles, key heads * H / (G heads))
template <int DC, int DT, int MAPS, int PARTS, bool SIG, int ST>
__global__ void __launch_bounds__(512) attn_tiles_kernel(AttnTileArgs p) {
  constexpr int CHK = MAPS * PARTS * DC * 2, CHV = PARTS * DT * 4;  // 16-byte chunks per row
  constexpr int STAGE = kTileKeys * 16 * (CHK + CHV);
  constexpr int PU = (CHK + CHV) / 8;  // DMAs per wave and stage (1 KB each)
  constexpr int QP = PARTS == 1 ? 3 : 2, DV = DT * 32;
  static_assert(CHK % 8 == 0 && CHV % 8 == 0 && (CHK == 8 || CHK % 16 == 0) && (CHV == 8 || CHV % 16 == 0), "rows");
  constexpr int kExchange = 4 * 64 * (DT * 16 + 2) * 4, kTurn = 4 * 32 * (DV + 4) * 4;
  constexpr int kLds = ST * STAGE > kExchange ? (ST * STAGE > kTurn ? ST * STAGE : kTurn)
                                              : (kExchange > kTurn ? kExchange : kTurn);
  static_assert(kLds <= kCuLds && (DC != 8 || DT != 4 || MAPS != 1 || PARTS != 1 || kLds == kPromptAttnLds), "LDS");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[kLds];
  const AttnArgs& a = p.a;
  const int tid = threadIdx.x, lane = tid & 63, lq = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nv = p.heads * MAPS, KS = nv == 8 ? 1 : 2, QW = 8 / (nv * KS);
  const int vh = wave % nv, ks = wave / nv % KS, qw = wave / (nv * KS);
  const int map = MAPS == 2 ? vh & 1 : 0;
  const int groups = a.H / p.heads, group = blockIdx.x % groups, at_b = blockIdx.x / groups, B = gridDim.x / groups / a.tiles;
  const int h = group * p.heads + vh / MAPS, g = h / (a.H / a.G);
  const int b = at_b % B, tile = a.tiles - 1 - at_b / B;
  const int rfirst = a.seq_start[b] + tile * 32 * QW, rend = a.seq_start[b + 1];
  if (rfirst >= rend) return;
  const int wgq = min(32 * QW, rend - rfirst);
  const int pos_first = a.seq_pos0[b] + tile * 32 * QW, pos_last = min(pos_first + wgq - 1, a.S - 1);
  auto lowest = [&](int pos) {
    return a.window > 0 ? max(0, pos - a.window + 1) : (a.chunk > 0 ? pos - pos % a.chunk : 0);
  };
  const int kt0 = lowest(pos_first) / kTileKeys, nkt = pos_last / kTileKeys + 1;
  // this lane's query
  const int row = rfirst + qw * 32 + lq;
  const bool live = row < rend;
  const int qpos = live ? pos_first + qw * 32 + lq : -1, qlo = live ? lowest(qpos) : 0;
  // what the wave's queries see in all (positions ascend over the lanes)
  const int nlive = min(32, max(0, rend - rfirst - qw * 32));
  const int wfirst = pos_first + qw * 32, wlast = nlive > 0 ? wfirst + nlive - 1 : -1;
  const int wlo = lowest(wfirst), whi_lo = nlive > 0 ? lowest(wlast) : 0;

  // key and value rows: a buffer per tile that ends after the last visible key (a sequence's rows may exceed one buffer)
  const size_t row0 = p.packed ? (size_t)a.seq_start[b] : (size_t)a.seq_slot[b] * a.S;
  const uint16_t* kbase = p.k + row0 * p.krow + (size_t)g * (MAPS * PARTS * DC * 16);
  const uint16_t* vbase = p.v + row0 * p.vrow + (size_t)g * (PARTS * DV);
  int voff[PU];
#pragma unroll
  for (int i = 0; i < PU; ++i) {
    const int u = wave * PU + i;
    const bool isv = u >= CHK;
    const int idx = (isv ? u - CHK : u) * 64 + lane, n = isv ? CHV : CHK;
    const int r = idx / n, ch = (idx % n) ^ chunk_swizzle(r, n);
    voff[i] = (int)((isv ? p.vrow : p.krow) * 2) * r + ch * 16;
  }
  auto stage = [&](int kt, int buf) {
    const int left = min(pos_last - kt * kTileKeys, kTileKeys - 1);  // the tile's last visible row
    const uint16_t* kat = kbase + (long)kt * kTileKeys * p.krow;
    const uint16_t* vat = vbase + (long)kt * kTileKeys * p.vrow;
    const int kbytes = left < 0 ? 0 : left * (int)p.krow * 2 + CHK * 16, vbytes = left < 0 ? 0 : left * (int)p.vrow * 2 + CHV * 16;
#pragma unroll
    for (int i = 0; i < PU; ++i) {
      const int u = wave * PU + i;
      const bool isv = u >= CHK;
      tile_dma16(isv ? vat : kat, isv ? vbytes : kbytes, voff[i], lds + buf * STAGE + u * 1024);
    }
  };

  bf16x8_t q[QP][DC];
  {
    const float* qr = a.q + (size_t)min(row, rend - 1) * a.ld + ((size_t)h * MAPS + map) * (DC * 16) + 8 * hh;
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      const float4 lo = *(const float4*)(qr + c * 16), hi = *(const float4*)(qr + c * 16 + 4);
      float x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
      for (int s = 0; s < QP; ++s) q[s][c] = take_summand(x);
    }
  }
  // LDS addresses: key row lq; transposed value rows (16-lane group grp, quad qq, pair pp) of the keys that a lane's
  // weights belong to: 4 hh + 0 .. 3 and 8 + 4 hh + 0 .. 3 of 16
  static_assert(MAPS == 1 || (PARTS == 1 && DC == 4), "the second map's chunks are the upper eight of sixteen");
  const int kaddr = lq * (CHK * 16) + 16 * (chunk_swizzle(lq, CHK) ^ (hh | (map * 8)));
  const int qq = (lane & 15) >> 2, pp = lane & 3, grp = lane >> 4;
  const int vr0 = 4 * (grp >> 1) + qq, vr1 = vr0 + 8, vch = 2 * (grp & 1) + (pp >> 1);
  const int vaddr0 = vr0 * (CHV * 16) + 16 * (chunk_swizzle(vr0, CHV) ^ vch) + 8 * (pp & 1);
  const int vaddr1 = vr1 * (CHV * 16) + 16 * (chunk_swizzle(vr1, CHV) ^ vch) + 8 * (pp & 1);
  auto at = [](int addr, int ch) {  // the chunk that is ch (whose bits the lane's own chunk does not have) further
    return (addr ^ (16 * (ch & 15))) + 256 * (ch >> 4);
  };
  f32x16_t o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[t][r] = 0.0f;
  float m = SIG ? 0.0f : -INFINITY, l = 0.0f;  // l: over the keys that this lane holds
  const float bias = SIG ? a.score_bias[h] : 0.0f, inv_cap = a.cap > 0.0f ? 1.0f / a.cap : 0.0f;

  auto keys32 = [&](const unsigned char* K, const unsigned char* V, int k0) {
    f32x16_t s, lo;  // the leading summands' products and the others'
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.0f, lo[r] = 0.0f;
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      const bf16x8_t k = *(const bf16x8_t*)(K + at(kaddr, 2 * c));
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k, q[0][c], s, 0, 0, 0);
      lo = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k, q[1][c], lo, 0, 0, 0);
      if (PARTS == 1) {
        lo = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k, q[QP - 1][c], lo, 0, 0, 0);
      } else {
        const bf16x8_t k1 = *(const bf16x8_t*)(K + at(kaddr, DC * 2 + 2 * c));
        lo = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k1, q[0][c], lo, 0, 0, 0);
      }
    }
    const bool edge = k0 + 31 > wfirst || k0 < whi_lo;  // some query of the wave does not see all of these
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float v = (s[r] + lo[r]) * a.scale;
      if (a.cap > 0.0f) v = a.cap * tanh_near(v * inv_cap);
      if (edge) {
        const int key = k0 + (r & 3) + 8 * (r >> 2) + 4 * hh;
        if (key > qpos || key < qlo) v = -INFINITY;
      }
      s[r] = v;
      if (!SIG) mx = fmaxf(mx, v);
    }
    float mref = 0.0f;
    if (!SIG) {
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
      const float mn = fmaxf(m, mx);
      mref = mn == -INFINITY ? 0.0f : mn;
      if (!__all(mn == m)) {
        const float f = m == -INFINITY ? 0.0f : exp_neg(m - mref);
        l *= f;
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[t][r] *= f;
      }
      m = mn;
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      float w[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = s[8 * kk + e];
        w[e] = v == -INFINITY ? 0.0f : (SIG ? sigmoid_near(v + bias) : exp_neg(v - mref));
        if (!SIG && MAPS == 1) l += w[e];
      }
      // (a difference of two maps, scaled up to unit size, shows what their normalisers lose in one long chain)
      if (MAPS == 2) l += ((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7]));
      bf16x8_t pw[3];
#pragma unroll
      for (int e = 0; e < 3; ++e) pw[e] = take_summand(w);
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int part = 0; part < PARTS; ++part) {
          typedef __attribute__((address_space(3))) i16x4_t lds_i16x4;
          const unsigned char* vk = V + kk * 16 * (CHV * 16);
          const i16x4_t x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(vk + at(vaddr0, part * DT * 4 + t * 4)));
          const i16x4_t y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(vk + at(vaddr1, part * DT * 4 + t * 4)));
          const bf16x8_t vt = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7));
          // The least summands first, then one rounding of the sum so far: 2.4e-7 off float64 with a cap of 3 over 1213 keys,
          // 4.3e-7 with the products one after the other, 4.0e-7 in the thread-per-key form, whose chains are shorter for
          // values of 64. (Of 128 the chain is no worse than that form's: 4.3e-7 and 5.2e-7.)
          if (MAPS == 2 && DT == 2) {
            f32x16_t c;
#pragma unroll
            for (int r = 0; r < 16; ++r) c[r] = 0.0f;
#pragma unroll
            for (int e = 2; e >= 0; --e) c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vt, pw[e], c, 0, 0, 0);
            o[t] += c;
            continue;
          }
#pragma unroll
          for (int e = 0; e < 3 - part; ++e) o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vt, pw[e], o[t], 0, 0, 0);
        }
    }
  };

#pragma unroll
  for (int s = 0; s < ST - 1; ++s) stage(kt0 + s, s);  // (past the last key: zeros)
  int buf = 0;
  for (int kt = kt0; kt < nkt; ++kt) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((ST - 2) * PU) : "memory");
    __builtin_amdgcn_s_barrier();  // tile kt is whole, and no wave reads the one before
    asm volatile("" ::: "memory");
    const unsigned char* K = lds + buf * STAGE;
    const unsigned char* V = lds + buf * STAGE + kTileKeys * 16 * CHK;
    for (int st = ks; st < 2; st += KS) {
      const int k0 = kt * kTileKeys + st * 32;
      if (k0 <= wlast && k0 + 31 >= wlo) keys32(K + st * 32 * (CHK * 16), V + st * 32 * (CHV * 16), k0);
    }
    // (behind the tile's work: the transposed reads wait for every DMA in flight)
    stage(kt + ST - 1, buf == 0 ? ST - 1 : buf - 1);
    buf = buf + 1 == ST ? 0 : buf + 1;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  l += __shfl_xor(l, 32);

  // ---- the two halves of the key tiles (one map), or the two maps
  float* ex = (float*)lds;
  constexpr int EX = 64 * (DT * 16 + 2);
  if (KS == 2) {
    float* mine = ex + (vh + nv * qw) * EX + lane;
    if (ks == 1) {
      mine[0] = m;
      mine[64] = l;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) mine[(2 + t * 16 + r) * 64] = o[t][r];
    }
    __syncthreads();
    if (ks == 0) {
      float fa = 1.0f, fb = 1.0f;
      if (!SIG) {
        const float m2 = mine[0], mn = fmaxf(m, m2), ref = mn == -INFINITY ? 0.0f : mn;
        fa = m == -INFINITY ? 0.0f : exp_neg(m - ref);
        fb = m2 == -INFINITY ? 0.0f : exp_neg(m2 - ref);
        l = l * fa + mine[64] * fb;
        m = mn;
      }
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] = o[t][r] * fa + mine[(2 + t * 16 + r) * 64] * fb;
    }
    __syncthreads();
  }
  bool store = ks == 0;
  if (MAPS == 2) {
    float* mine = ex + (vh / 2 + p.heads * qw) * EX + lane;
    const float inv = 1.0f / l;
    if (store && map == 1) {
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) mine[(t * 16 + r) * 64] = o[t][r] * inv;
    }
    __syncthreads();
    store = store && map == 0;
    if (store) {
      float ss = 0.0f;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          o[t][r] = o[t][r] * inv - a.lambda * mine[(t * 16 + r) * 64];
          ss = fmaf(o[t][r], o[t][r], ss);
        }
      ss += __shfl_xor(ss, 32);
      const float f = a.post / sqrtf(ss / (float)DV + a.eps);
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] *= f;
    }
    __syncthreads();
  } else if (store) {
    float f = a.post;
    if (!SIG) {
      float den = l;
      if (a.sink) {
        const float snk = a.sink[h], top = fmaxf(m, snk);
        const float w = m == -INFINITY ? 0.0f : expf(m - top);
        den = l * w + expf(snk - top);
        f *= w;
      }
      f /= den;
    }
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[t][r] *= f;
  }
  if (!store) return;
  float bad = 0.0f;  // NaN where a result of this lane's query is not finite
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) bad = fmaf(o[t][r], 0.0f, bad);
  const unsigned long long odd = __ballot(live && bad != 0.0f);
  // ---- turned in LDS: a wave writes whole rows of a head
  const int slot = MAPS == 2 ? vh / 2 + p.heads * qw : vh + nv * qw;
  float* turn = ex + slot * 32 * (DV + 4);
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int r = 0; r < 16; r += 4)
      *(float4*)(turn + lq * (DV + 4) + t * 32 + 8 * (r >> 2) + 4 * hh) =
          make_float4(o[t][r], o[t][r + 1], o[t][r + 2], o[t][r + 3]);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  if (odd) {
    for (uint32_t rows = (uint32_t)odd | (uint32_t)(odd >> 32); rows; rows &= rows - 1) {
      const int i = __ffs(rows) - 1;
      const float* q_at = a.q + (size_t)(rfirst + qw * 32 + i) * a.ld + (size_t)h * MAPS * DC * 16;
      attn_row_plain<DC, DT, MAPS, PARTS, SIG>(p, kbase, vbase, q_at, h, lowest(wfirst + i), min(wfirst + i, a.S - 1), lane,
                                               turn + i * (DV + 4));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  constexpr int LANES = DV / 4;  // a lane holds four columns
  for (int i = lane / LANES; i < nlive; i += 64 / LANES) {
    const int c = lane % LANES * 4;
    const float4 got = *(const float4*)(turn + i * (DV + 4) + c);
    float v[4] = {got.x, got.y, got.z, got.w};
    const size_t orow = (size_t)(rfirst + qw * 32 + i);
    if (a.v_freq) {  // turned back by the query's position
      const int hv = DV / 2;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int ce = c + e;
        const bool second = a.interleaved ? (ce & 1) : ce >= hv;
        const int f = a.interleaved ? ce >> 1 : (second ? ce - hv : ce);
        const float other = turn[i * (DV + 4) + (a.interleaved ? ce ^ 1 : (second ? ce - hv : ce + hv))];
        const float mine = e == 0 ? got.x : (e == 1 ? got.y : (e == 2 ? got.z : got.w));
        float sn, cs;
        sincosf((float)(wfirst + i) * a.v_freq[f], &sn, &cs);
        v[e] = second ? mine * cs - other * sn : mine * cs + other * sn;
      }
    }
    if (a.gate) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[e] *= sigmoid_f(a.gate[orow * a.ldg + (a.gate_cols == 1 ? (size_t)h : (size_t)h * DV + c + e)]);
    }
    const size_t to = orow * a.H * DV + (size_t)h * DV + c;
    if (a.out) *(float4*)(a.out + to) = make_float4(v[0], v[1], v[2], v[3]);
    if (a.out16) *(uint2*)(a.out16 + to) = make_uint2(pack2(v[0], v[1]), pack2(v[2], v[3]));
  }
}

// The sizes that have a form, where queries, keys, values and results start on the bytes that it moves at a time, however many
// rows a cache holds; any step with more than one token of a sequence: 9 tokens after 1500 of 16 heads on 4 key heads of 128
// take 75 us here and 158 with a thread per key (seq_attn.hip), 9 of a new sequence 15 and 24, 2048 of one 110 and 634 (51
// GFLOP of bf16 products, 17 of fp32 ones).
bool attn_tiles_fit(const AttnArgs& a, int maps, int parts, int max_len) {
  const bool sized = parts == 2 ? (maps == 1 && a.d == 192 && a.dv == 128)
                                : ((a.dv == 64 || a.dv == 128) && (a.d == 64 || (a.d == 128 && maps == 1)));
  const long row = (long)(parts == 2 ? 2 * a.H : a.G) * (maps * a.d > a.dv ? maps * a.d : a.dv);
  return sized && row <= kMostRow && max_len > 1 && a.pool == 0 && a.ld % 4 == 0 && (uintptr_t)a.q % 16 == 0 &&
         ((uintptr_t)a.cache_k | (uintptr_t)a.cache_v | (uintptr_t)a.out) % 16 == 0 && (uintptr_t)a.out16 % 8 == 0;
}

template <int DC, int DT, int MAPS, int PARTS, int ST>
static int attn_tiles_go(const AttnTileArgs& p, dim3 grid, hipStream_t stream) {
  if (MAPS == 1 && PARTS == 1 && p.a.score_bias)
    attn_tiles_kernel<DC, DT, MAPS, PARTS, MAPS == 1 && PARTS == 1, ST><<<grid, 512, 0, stream>>>(p);
  else
    attn_tiles_kernel<DC, DT, MAPS, PARTS, false, ST><<<grid, 512, 0, stream>>>(p);
  return 0;
}

int attn_tiles_launch(const AttnTileArgs& given, int maps, int parts, int B, int max_len, hipStream_t stream) {
  AttnTileArgs p = given;
  AttnArgs& a = p.a;
  const int share = a.H / a.G;
  p.heads = share % 4 == 0 ? 4 : (share % 2 == 0 ? 2 : 1);
  const int nv = p.heads * maps, qw = nv == 8 ? 1 : 4 / nv;
  a.tiles = (max_len + 32 * qw - 1) / (32 * qw);
  LGA_CHECK_ARG(p.krow <= kMostRow && p.vrow <= kMostRow, "attention: a position's keys or values exceed a buffer");
  LGA_CHECK_ARG((long)B * a.tiles * (a.H / p.heads) < (1L << 31), "attention: too many tiles");
  const dim3 grid((unsigned)(B * a.tiles * (a.H / p.heads)));
  if (parts == 2) return attn_tiles_go<12, 4, 1, 2, 2>(p, grid, stream);
  if (maps == 2) return a.dv == 64 ? attn_tiles_go<4, 2, 2, 1, 3>(p, grid, stream) : attn_tiles_go<4, 4, 2, 1, 3>(p, grid, stream);
  if (a.d == 64) return a.dv == 64 ? attn_tiles_go<4, 2, 1, 1, 3>(p, grid, stream) : attn_tiles_go<4, 4, 1, 1, 3>(p, grid, stream);
  return a.dv == 64 ? attn_tiles_go<8, 2, 1, 1, 3>(p, grid, stream) : attn_tiles_go<8, 4, 1, 1, 3>(p, grid, stream);
}

// keys [T][H][2][d + dr] and values [T][H][2][dv] as two bf16 summands (the nearest bf16 and the nearest to what is left)
// from a row's products kv [T][ld] (H keys of d, then H values of dv) and the rotated part that its heads share, row
// rows[t] of kr. grid (T)
__global__ void __launch_bounds__(256) latent_split_kernel(const float* __restrict__ kv, long ld, const float* __restrict__ kr,
                                                           const int* __restrict__ rows, uint16_t* __restrict__ k,
                                                           uint16_t* __restrict__ v, int H, int d, int dr, int dv) {
  const size_t t = blockIdx.x;
  const float* shared = kr + (size_t)rows[t] * dr;
  auto put = [](uint16_t* hi, uint16_t* lo, const float4 x) {
    const uint32_t a = pack2(x.x, x.y), b = pack2(x.z, x.w);
    auto left = [](float v, float top) { return fabsf(top) == INFINITY ? 0.0f : v - top; };  // (an infinity is its own sum)
    *(uint2*)hi = make_uint2(a, b);
    *(uint2*)lo = make_uint2(pack2(left(x.x, bflo(a)), left(x.y, bfhi(a))), pack2(left(x.z, bflo(b)), left(x.w, bfhi(b))));
  };
  const int dk = d + dr, nk = dk / 4, nv = dv / 4;
  for (int i = threadIdx.x; i < H * nk; i += 256) {
    const int h = i / nk, c = i % nk * 4;
    const float4 x = c < d ? *(const float4*)(kv + t * ld + (size_t)h * d + c) : *(const float4*)(shared + c - d);
    uint16_t* out = k + (t * H + h) * 2 * dk + c;
    put(out, out + dk, x);
  }
  for (int i = threadIdx.x; i < H * nv; i += 256) {
    const int h = i / nv, c = i % nv * 4;
    uint16_t* out = v + (t * H + h) * 2 * dv + c;
    put(out, out + dv, *(const float4*)(kv + t * ld + (size_t)H * d + (size_t)h * dv + c));
  }
}

}  // namespace lgs

extern "C" int lgs_latent_split(const float* kv, long ld, const float* cache_kr, const int* rows, void* k, void* v, int T,
                                int H, int d, int dr, int dv, hipStream_t stream) {
  LGA_CHECK_ARG(kv && cache_kr && rows && k && v && T > 0 && H > 0 && d > 0 && dr >= 0 && dv > 0,
                "lgs_latent_split: bad arguments");
  LGA_CHECK_ARG(d % 4 == 0 && dr % 4 == 0 && dv % 4 == 0 && ld % 4 == 0 && ld >= (long)H * (d + dv) &&
                    ((uintptr_t)kv | (uintptr_t)cache_kr) % 16 == 0 && ((uintptr_t)k | (uintptr_t)v) % 8 == 0,
                "lgs_latent_split: rows in pieces of four values");
  lgs::latent_split_kernel<<<T, 256, 0, stream>>>(kv, ld, cache_kr, rows, (uint16_t*)k, (uint16_t*)v, H, d, dr, dv);
  LGA_LAUNCH_RETURN();
}

extern "C" int lgs_split_attention_fits(int H, int dk, int dv) {
  lgs::AttnArgs a{};
  a.H = a.G = H;
  a.d = dk;
  a.dv = dv;
  return lgs::attn_tiles_fit(a, 1, 2, 2) ? 1 : 0;
}

extern "C" int lgs_split_attention(const float* q, long ld, const void* k, const void* v, const float* sink,
                                   const int* seq_start, const int* seq_slot, const int* seq_pos0, float* out,
                                   void* out_bf16, int B, int max_len, int H, int dk, int dv, float scale, int window,
                                   hipStream_t stream) {
  LGA_CHECK_ARG(q && k && v && seq_start && seq_slot && seq_pos0 && (out || out_bf16), "lgs_split_attention: null pointer");
  LGA_CHECK_ARG(B > 0 && max_len > 1 && H > 0 && window >= 0 && ld >= (long)H * dk, "lgs_split_attention: bad sizes");
  LGA_CHECK_ARG(((uintptr_t)k | (uintptr_t)v) % 16 == 0, "lgs_split_attention: aligned summands");
  lgs::AttnArgs a{};
  a.q = q, a.ld = ld, a.seq_start = seq_start, a.seq_slot = seq_slot, a.seq_pos0 = seq_pos0;
  a.out = out, a.out16 = (uint16_t*)out_bf16;
  a.H = H, a.G = H, a.d = dk, a.dv = dv, a.S = max_len, a.scale = scale, a.post = 1.0f, a.sink = sink, a.window = window;
  LGA_CHECK_ARG(lgs::attn_tiles_fit(a, 1, 2, max_len), "lgs_split_attention: sizes or alignment without a form");
  const lgs::AttnTileArgs t{a, (const uint16_t*)k, (const uint16_t*)v, 2L * H * dk, 2L * H * dv, 1, 0};
  const int rc = lgs::attn_tiles_launch(t, 1, 2, B, max_len, stream);
  if (rc) return rc;
  LGA_LAUNCH_RETURN();
}
