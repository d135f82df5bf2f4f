// Prefill GEMM with weights dequantized in registers: the same products as gemm_q4f.hip (Y = X . bf16(dequant(W))^T with
// bias / residual, and fc_1 || fc_2 + SwiGLU) for prompts whose weight tiles serve few rows; what gemm_q4r.hip leaves of them.
//
// gemm_q4f.hip stages packed weights in LDS, dequantizes them into a bf16 image there and reads fragments back: three
// LDS round trips and a barrier per 64 values of K, which a tile of few rows cannot hide (0.75 us a step). Here a weight
// never passes through LDS. A wave owns 32 rows of W; a lane loads 16 bytes (32 packed values, one scale) of its own
// row per 128 values of K, D blocks ahead in registers, and dequantizes them, to the bits that bnb's dequantize_4bit
// writes, straight into the A operand of v_mfma_f32_16x16x32_bf16. The products' order over K follows what a lane holds:
// instruction m of a block takes values 32 fk + 8 m .. + 7 of each of the four lane groups fk. X (up to 128 rows a tile)
// is shared by the eight waves through LDS (LDS-DMA, source-swizzled, D + 1 buffers), one barrier per 128 values of K.
//
// Ranges of K run side by side until the chip is full; their fp32 partial sums are added in order by a second launch that
// also runs the epilogue.
//
// Bound: up to 64 rows by about 1.7 us per block of 256 rows x 128 values, which neither the dequantization nor the loads'
// width moves (16 x 8192 x 28672 in int4: 46 us, 2.6 TB/s), beyond by the matrix cores' feeding from LDS. Against the LDS
// image, 93 rows of nf4 (N x K): 10240 x 8192 97 -> 43 us, 8192 x 8192 62 -> 39, 8192 x 28672 176 -> 82, 28672 x 8192 with
// SwiGLU 311 -> 150; int4 12288 x 4096 45 -> 29, 4096 x 11008 42 -> 30, 11008 x 4096 with SwiGLU 65 -> 41.
#include "gemm_q4d.h"

namespace lga {
namespace pd {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int BK = 128, NT = 512, NR = 2;  // values of K per block; threads; 16-row pieces of W per wave

struct KArgs {
  Q4dArgs a;
  int mt, nt, splits, per;  // row tiles, column tiles, ranges of K and 128-deep blocks per range
};

// 16 bytes a lane into LDS. Through a buffer resource: behind a flat-encoded load the compiler waits for every load in
// flight wherever it needs one
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, unsigned off, unsigned soff, unsigned char* lds) {
#ifdef __HIP_DEVICE_COMPILE__  // (a device builtin: the host pass only type-checks the body)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, off, soff, 0, 0);
#endif
}
template <int N>  // until at most N of this wave's loads are in flight (the count is a field of the instruction)
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ f32x4_t mfma(bf16x8_t a, bf16x8_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ void cvt_bytes(uint32_t w, float (&f)[4]) {
  asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(f[0]) : "v"(w));
  asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(f[1]) : "v"(w));
  asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(f[2]) : "v"(w));
  asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(f[3]) : "v"(w));
}

// eight packed values -> bf16(value * scale)
template <int FMT>
__device__ __forceinline__ bf16x8_t dequant8(uint32_t w, float s, const float* tab) {
  u32x4 o;
  if (FMT == 0) {  // fma(n, s, -8 s) is exact, rounded once
    const float c = -8.0f * s;
    float fl[4], fh[4];
    cvt_bytes(w & 0x0F0F0F0Fu, fl);
    cvt_bytes((w >> 4) & 0x0F0F0F0Fu, fh);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = pack2(__builtin_fmaf(fl[e], s, c), __builtin_fmaf(fh[e], s, c));
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      o[e] = pack2(__fmul_rn(tab[(w >> (8 * e)) & 0xFu], s), __fmul_rn(tab[(w >> (8 * e + 4)) & 0xFu], s));
  }
  return __builtin_bit_cast(bf16x8_t, o);
}

// FMT 0 int4-g (bf16 scales), 1 codebook (fp32 block maxima). MF: 16-row pieces of X
template <int FMT, bool DUAL, int MF>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2, 2))) gemm_q4d_kernel(KArgs k) {
  const Q4dArgs& a = k.a;
  constexpr int D = 3, NS = D + 1;                          // blocks of 128 values of K ahead; slots
  constexpr int XB = MF * 16 * 256, XP = (MF * 4 + 7) / 8;  // X: bytes of a block; DMAs per wave (1 KB, 4 rows)
  constexpr int WOPS = NR * 2;                              // W: a row's loads of a block are its 16 bytes and the scale
  constexpr int JN = DUAL ? NR / 2 : NR;                    // fragments per matrix
  static_assert((D - 1) * XP + D * WOPS <= 63 && NS * XB + 64 <= 163840, "loads in flight; LDS");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[NS * XB + 64];
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 15, fk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  float* tab = (float*)(lds + NS * XB);
  if (FMT == 1 && tid < 16) tab[tid] = kCode4[a.cb][tid];
  // neighbouring work on one XCD: a column tile's row tiles, then its ranges of K
  const int t = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (t >= k.mt * k.nt * k.splits) return;
  const int m0 = t % k.mt * (MF * 16), split = t / k.mt % k.splits, n0 = t / k.mt / k.splits * (128 * JN);
  const int nb_all = a.K / BK, b0 = split * k.per, b1 = min(nb_all, b0 + k.per);
  const int groups = a.K / a.G, gshift = 31 - __builtin_clz((unsigned)a.G);

  const unsigned char* wp[NR];
  size_t srow[NR];
#pragma unroll
  for (int j = 0; j < NR; ++j) {
    const int n = min(n0 + (wave * JN + j % JN) * 16 + fr, a.N - 1);
    wp[j] = (const unsigned char*)(j < JN ? a.w : a.w2) + (size_t)n * (a.K / 2) + fk * 16;
    srow[j] = (size_t)n * groups;
  }
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.x + (size_t)m0 * a.K), (short)0, min(a.M - m0, MF * 16) * a.K * 2, 0x00020000);
  unsigned xp[XP];
  int xl[XP];
#pragma unroll
  for (int i = 0; i < XP; ++i) {
    const int piece = min(i * 8 + wave, MF * 4 - 1);  // (a surplus DMA repeats the last piece)
    const int r = piece * 4 + (lane >> 4), c = (lane & 15) ^ (r & 15);
    xl[i] = piece * 1024;
    xp[i] = (unsigned)(min(r, a.M - 1 - m0) * a.K + c * 8) * 2;
  }
  u32x4 w[NS][NR];
  uint32_t sc[NS][NR];
  auto fetch = [&](int b, int s) {  // block b (past the range: its last, never used) into slot s; X before W, as the waits count
    const int bb = min(b, b1 - 1);
#pragma unroll
    for (int i = 0; i < XP; ++i) dma16(xr, xp[i], bb * (BK * 2), lds + s * XB + xl[i]);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < NR; ++j) w[s][j] = *(const u32x4*)(wp[j] + (size_t)bb * (BK / 2));
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      const void* sp = j < JN ? a.sc : a.sc2;
      const size_t si = srow[j] + ((bb * BK + fk * 32) >> gshift);
      sc[s][j] = FMT == 0 ? ((const uint16_t*)sp)[si] : ((const uint32_t*)sp)[si];
    }
  };
  f32x4_t acc[NR][MF];
#pragma unroll
  for (int j = 0; j < NR; ++j)
#pragma unroll
    for (int i = 0; i < MF; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto block = [&](int s) {
    const unsigned char* X = lds + s * XB + fr * 256;
    bf16x8_t xf[2][MF];  // the fragments of the next 32 values are read while these are used
    auto frags = [&](int m, bf16x8_t (&f)[MF]) {
#pragma unroll
      for (int i = 0; i < MF; ++i)
        f[i] = *(const bf16x8_t*)(X + i * 4096 + 16 * ((fk * 4 + m) ^ fr));
    };
    frags(0, xf[0]);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      bf16x8_t wf[NR];
#pragma unroll
      for (int j = 0; j < NR; ++j)
        wf[j] = dequant8<FMT>(w[s][j][m], __uint_as_float(FMT == 0 ? sc[s][j] << 16 : sc[s][j]), tab);
      if (m < 3) frags(m + 1, xf[(m + 1) & 1]);
#pragma unroll
      for (int i = 0; i < MF; ++i)
#pragma unroll
        for (int j = 0; j < NR; ++j) acc[j][i] = mfma(wf[j], xf[m & 1][i], acc[j][i]);
    }
  };
#pragma unroll
  for (int s = 0; s < D; ++s) {
    fetch(b0 + s, s);
    asm volatile("" ::: "memory");
  }
  for (int b = b0; b < b1; b += NS) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if (b + s < b1) {
        wait_vm<(D - 1) * XP + D * WOPS>();  // X of block b + s is here: later loads may be in flight
        __builtin_amdgcn_s_barrier();        // ... for every wave, and nobody reads the block before it
        asm volatile("" ::: "memory");
        fetch(b + s + D, (s + D) % NS);
        block(s);
      }
    }
  }
  wait_vm<0>();  // no DMA may outlive the workgroup's LDS

  // a lane holds columns 4 fk .. + 3 of fragment j for row fr of piece i
  const size_t ldy = a.ldy ? a.ldy : a.N;
#pragma unroll
  for (int j = 0; j < JN; ++j) {
    const int n = n0 + (wave * JN + j) * 16 + fk * 4;
    if (n >= a.N) continue;
#pragma unroll
    for (int i = 0; i < MF; ++i) {
      const int m = m0 + i * 16 + fr;
      if (m >= a.M) continue;
      if (k.splits > 1) {
        float* p = a.slabs + ((size_t)split * (DUAL ? 2 : 1) * a.M + m) * a.N + n;
        *(f32x4_t*)p = acc[j][i];
        if (DUAL) *(f32x4_t*)(p + (size_t)a.M * a.N) = acc[NR - JN + j][i];
      } else if (DUAL) {
        *(uint2*)(a.y + m * ldy + n) = q4d_swiglu(acc[j][i], acc[NR - JN + j][i]);
      } else {
        q4d_store(a, m, n, ldy, acc[j][i]);
      }
    }
  }
}

// the ranges of K in order, then the epilogue; a thread takes four columns of a row
template <bool DUAL>
__global__ void __launch_bounds__(256) q4d_sum_kernel(Q4dArgs a, int splits) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x, n4 = a.N / 4;
  if (i >= (size_t)a.M * n4) return;
  const int m = (int)(i / n4), n = (int)(i % n4) * 4;
  const size_t plane = (size_t)a.M * a.N, step = plane * (DUAL ? 2 : 1);
  const float* p = a.slabs + (size_t)m * a.N + n;
  f32x4_t s = *(const f32x4_t*)p, s2 = {0.f, 0.f, 0.f, 0.f};
  if (DUAL) s2 = *(const f32x4_t*)(p + plane);
#pragma unroll 4
  for (int z = 1; z < splits; ++z) {
    s += *(const f32x4_t*)(p + z * step);
    if (DUAL) s2 += *(const f32x4_t*)(p + z * step + plane);
  }
  const size_t ldy = a.ldy ? a.ldy : a.N;
  if (DUAL) *(uint2*)(a.y + m * ldy + n) = q4d_swiglu(s, s2);
  else q4d_store(a, m, n, ldy, s);
}

}  // namespace pd

void q4d_sum(const Q4dArgs& a, int splits, bool dual, hipStream_t stream) {
  const unsigned grid = (unsigned)(((size_t)a.M * a.N / 4 + 255) / 256);
  if (dual) pd::q4d_sum_kernel<true><<<grid, 256, 0, stream>>>(a, splits);
  else pd::q4d_sum_kernel<false><<<grid, 256, 0, stream>>>(a, splits);
}

namespace pd {

template <int FMT, bool DUAL, int MF>
static int go(KArgs k, hipStream_t stream) {
  const unsigned work = (unsigned)(k.mt * k.nt * k.splits);
  gemm_q4d_kernel<FMT, DUAL, MF><<<(work + 7) / 8 * 8, NT, 0, stream>>>(k);
  if (k.splits > 1) q4d_sum(k.a, k.splits, DUAL, stream);
  return 0;
}

template <int FMT, bool DUAL>
static int go_rows(const KArgs& k, int mf, hipStream_t stream) {
  switch (mf) {
    case 1: return go<FMT, DUAL, 1>(k, stream);
    case 2: return go<FMT, DUAL, 2>(k, stream);
    case 4: return go<FMT, DUAL, 4>(k, stream);
    case 6: return go<FMT, DUAL, 6>(k, stream);
    default: return go<FMT, DUAL, 8>(k, stream);
  }
}

}  // namespace pd

// Which products come here, of those that gemm_q4r.hip leaves (q4r_plan: up to 96 rows) or has no aligned scales for (us here / on
// the LDS image's tiles; NK = N x K of one matrix):
//   up to 32 rows   all but NK <= 2^24, where two launches are not repaid (int4 16 x 4096 x 4096: 18 / 15)
//   up to 96 rows   all (int4 64 x 4096 x 4096: 19 / 23)
//   up to 128 rows  beyond 2^24 (int4 4096 x 4096: 31 / 26; 12288 x 4096: 37 / 42); SwiGLU from 2^26 (int4 11008 x 4096:
//                   68 / 64, 28672 x 8192: 159 / 268)
//   up to 256 rows  one matrix up to 2^27 of at most 16384 columns (nf4 200 x 8192 x 8192: 56 / 71; 16384 x 4096: 56 / 70,
//                   16384 x 8192: 95 / 101; 20480 x 4096: 83 / 70, 28672 x 4096: 84 / 74, 50000 x 2048: 90 / 73; 8192 x
//                   28672: 156 / 160, int4 142 / 148 at 160): the 256-row tiles read larger weights once, and more
//                   columns give them more than half a round of the chip without ranges of K
Q4dPlan q4d_plan(int M, int N, int K, bool dual) {
  Q4dPlan p{0, 0, 0, 0, 0};
  const size_t nk = (size_t)N * K, one = 1;
  if (K % pd::BK != 0 || M > 256) return p;
  if (M > 128 && (dual || N > 16384 || nk > one << 27)) return p;
  if (M > 96 && M <= 128 && nk <= one << (dual ? 26 : 24)) return p;
  if (M <= 32 && nk <= one << 24) return p;
  p.mf = M <= 16 ? 1 : (M <= 32 ? 2 : (M <= 64 ? 4 : (M <= 96 ? 6 : 8)));
  p.mt = (M + p.mf * 16 - 1) / (p.mf * 16);
  const int cols = 128 * (dual ? 1 : 2), nb = K / pd::BK;
  p.nt = (N + cols - 1) / cols;
  // ranges of K: rounds of 256 workgroups (two to a CU are no faster: 16 x 10240 x 8192 24 us with 240, 28 with 480) times
  // their blocks and a start of about four blocks' time, and the second launch with its traffic, in thousandths of a block
  long best = 0;
  for (int s = 1; s <= 16 && (s == 1 || nb / s >= 2); ++s) {
    const int per = (nb + s - 1) / s, used = (nb + per - 1) / per;
    const long cost = ((long)p.mt * p.nt * used + 255) / 256 * (per + 4) * 1000 +
                      (used > 1 ? 3000 + (long)M * N * (dual ? 2 : 1) * used / 1000 : 0);
    if (s == 1 || cost < best) best = cost, p.splits = used, p.per = per;
  }
  return p;
}

size_t q4d_workspace(const Q4dPlan& p, int M, int N, bool dual) {
  return p.splits > 1 ? 4096 + (size_t)p.splits * (dual ? 2 : 1) * M * N * 4 : 0;
}

int q4d_run(const Q4dArgs& a, const Q4dPlan& p, int kernel_fmt, bool dual, hipStream_t stream) {
  const pd::KArgs k{a, p.mt, p.nt, p.splits, p.per};
  switch (kernel_fmt * 2 + (dual ? 1 : 0)) {
    case 0: pd::go_rows<0, false>(k, p.mf, stream); break;
    case 1: pd::go_rows<0, true>(k, p.mf, stream); break;
    case 2: pd::go_rows<1, false>(k, p.mf, stream); break;
    default: pd::go_rows<1, true>(k, p.mf, stream); break;
  }
  LGA_LAUNCH_RETURN();
}

int preload_gemm_q4d() {
  using namespace pd;
  int bad = 0;
#define LGA_PRE(F, D)                                                                                    \
  bad += preload(gemm_q4d_kernel<F, D, 1>) + preload(gemm_q4d_kernel<F, D, 2>) +                         \
         preload(gemm_q4d_kernel<F, D, 4>) + preload(gemm_q4d_kernel<F, D, 6>) + preload(gemm_q4d_kernel<F, D, 8>)
  LGA_PRE(0, false);
  LGA_PRE(0, true);
  LGA_PRE(1, false);
  LGA_PRE(1, true);
#undef LGA_PRE
  return bad + preload(q4d_sum_kernel<false>) + preload(q4d_sum_kernel<true>);
}

}  // namespace lga
