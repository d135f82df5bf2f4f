// Prefill GEMM with 4-bit weights: the products of gemm_q4d.hip (Y = X . bf16(dequant(W))^T with bias / residual, and fc_1 ||
// fc_2 + SwiGLU) where a tile of weights serves 128 to 256 rows, and most of those where it serves 32 to 96.
//
// A workgroup of four waves makes 256 columns (SwiGLU: 128 of each matrix) of 32 FN rows; a wave 64 columns of all its rows:
// 2 x FN accumulators of v_mfma_f32_32x32x16_bf16 with the weights as the A operand, so that no weight is dequantized
// twice. X reaches LDS as in gemm_tiles.h: whole 128-byte lines, a ring of RX steps of 64 values, one barrier a step, whose last
// 16 values' operands are in registers by then. Packed weights reach LDS 64 bytes of a row at a time (two steps' worth), a wave's
// own rows only, so that no barrier is theirs; a lane takes 16 bytes of its row a step and dequantizes eight of its 32 values,
// to the bits that bnb's dequantize_4bit writes, between the matrix instructions of the 16 values of K before. The products'
// order over K follows what a lane holds: instruction m of a step takes values 8 m .. + 7 and 32 + 8 m .. + 7. (Weights loaded
// straight into registers cost 64 separate addresses a load: 930 of 5600 clocks a pair of steps, scales two at a time 700.)
//
// Up to 96 rows a wave has too few matrix instructions to stand its 410 others of a pair of steps between (one each five
// clocks while a wave is alone on its SIMD, half as many while two are): a second group of four waves takes the other half of
// the workgroup's range of K, with buffers of its own, and hands its sums over in LDS. 93 rows of nf4 28672 x 8192 with SwiGLU:
// one group 135 us, two workgroups of one group each on a CU and halves of K through memory 137, two groups 124.
#include "gemm_q4d.h"

#include <algorithm>

namespace lga {
namespace pr {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

struct KArgs {
  Q4dArgs a;
  int mt, nt, splits, per;  // tiles over rows and columns, ranges of K and pairs of steps (128 values) per range
};

// 16 bytes a lane into LDS. Through a buffer resource: behind a flat-encoded load the compiler waits for every load in
// flight wherever it needs one
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, unsigned off, unsigned soff, unsigned char* lds) {
#ifdef __HIP_DEVICE_COMPILE__  // (a device builtin: the host pass only type-checks the body)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, off, soff, 0, 0);
#endif
}
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack(float lo, float hi) {  // v_cvt_pk_bf16_f32
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), bf16x2));
}

// Eight packed values of one row -> bf16(value * scale), in eight parts that stand between matrix instructions. A wave alone
// on its SIMD issues an instruction of any kind every five clocks, six to a matrix instruction's 32; what stands closer in
// one place costs its full time.
template <int FMT>
struct Dequant;
template <>
struct Dequant<0> {  // int4-g: fma(n, s, -8 s) is exact, rounded once
  uint32_t lo, hi;
  float a, b;
  u32x4 o;
  template <int P>
  __device__ __forceinline__ void part(uint32_t w, float s, const unsigned char*) {
    const float c = -8.0f * s;
    // (opaque, or hipcc would extract each nibble anew)
    if constexpr (P == 0) {
      lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;
      asm("" : "+v"(lo), "+v"(hi));
    }
    if constexpr (P == 1) a = (float)(lo & 0xFF), b = (float)(hi & 0xFF), a = __builtin_fmaf(a, s, c);
    if constexpr (P == 2) b = __builtin_fmaf(b, s, c), o[0] = pack(a, b), a = (float)(lo >> 8 & 0xFF);
    if constexpr (P == 3) b = (float)(hi >> 8 & 0xFF), a = __builtin_fmaf(a, s, c), b = __builtin_fmaf(b, s, c);
    if constexpr (P == 4) o[1] = pack(a, b), a = (float)(lo >> 16 & 0xFF), b = (float)(hi >> 16 & 0xFF);
    if constexpr (P == 5) a = __builtin_fmaf(a, s, c), b = __builtin_fmaf(b, s, c), o[2] = pack(a, b);
    if constexpr (P == 6) a = (float)(lo >> 24), b = (float)(hi >> 24), a = __builtin_fmaf(a, s, c);
    if constexpr (P == 7) b = __builtin_fmaf(b, s, c), o[3] = pack(a, b);
  }
};
template <>
struct Dequant<1> {  // codebook in LDS, fp32 product: the lookups first, the products when they are back
  uint32_t lo, hi;  // the nibbles times four, a byte each
  float l[4], h[4];
  u32x4 o;
  template <int P>
  __device__ __forceinline__ void part(uint32_t w, float s, const unsigned char* tab) {
    auto look = [&](uint32_t b, int e) { return *(const float*)(tab + (b >> (8 * e) & 0xFF)); };
    if constexpr (P == 0) {
      lo = w << 2 & 0x3C3C3C3Cu;
      asm("" : "+v"(lo));
      l[0] = look(lo, 0);
    }
    if constexpr (P == 1) l[1] = look(lo, 1), l[2] = look(lo, 2);
    if constexpr (P == 2) {
      l[3] = look(lo, 3);
      hi = w >> 2 & 0x3C3C3C3Cu;
      asm("" : "+v"(hi));
      h[0] = look(hi, 0);
    }
    if constexpr (P == 3) h[1] = look(hi, 1), h[2] = look(hi, 2), h[3] = look(hi, 3);
    if constexpr (P >= 4) o[P - 4] = pack(__fmul_rn(l[P - 4], s), __fmul_rn(h[P - 4], s));
  }
};

template <int FN>
struct Tile {
  static constexpr int KW = FN < 4 ? 2 : 1;                                              // groups of four waves: halves of K
  static constexpr int RX = FN == 8 ? 3 : (FN == 6 ? 5 : (FN == 4 ? 6 : (FN == 3 ? 3 : 4)));  // X: steps of 64 values in LDS
  static constexpr int XB = FN * 4096, WB = 16384, OFF_W = RX * XB, GROUP = OFF_W + 2 * WB, OFF_TAB = KW * GROUP, LDS = OFF_TAB + 64;
  static_assert(LDS <= 163840, "LDS");
  // loads younger than X of step k + 1 at the barrier of step k: what the steps since its own have issued (X, and the scales of
  // a pair in its first step, its weights in its second)
  static constexpr int later(int k) {
    int n = 0;
    for (int j = k + 3 - RX; j <= k; ++j) n += FN + (j % 2 != 0 ? 4 : 1);
    return n;
  }
  static_assert(later(8) <= 63 && later(9) <= 63, "loads in flight are counted in six bits");
};

// FMT 0 int4-g (bf16 scales), 1 codebook (fp32 block maxima)
template <int FMT, bool DUAL, int FN>
__global__ void __launch_bounds__(256 * Tile<FN>::KW, Tile<FN>::KW) gemm_q4r_kernel(KArgs k) {
  using T = Tile<FN>;
  constexpr int RX = T::RX, XB = T::XB, KW = T::KW, E = 2 * FN;
  __shared__ __attribute__((aligned(1024))) unsigned char lds_all[T::LDS];
  const Q4dArgs& a = k.a;
  const int tid = threadIdx.x, lane = tid & 63, l31 = lane & 31, hi = lane >> 5;
  const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave_all & 3, kg = wave_all >> 2;
  unsigned char* lds = lds_all + kg * T::GROUP;
  const unsigned char* tab = lds_all + T::OFF_TAB;
  if (FMT == 1 && tid < 16) ((float*)tab)[tid] = kCode4[a.cb][tid];
  // an XCD takes neighbouring tiles: of a column's weights those of up to eight row tiles, range after range
  int t = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int per = k.nt * k.mt, split = t / per;
  if (split >= k.splits) return;
  t -= split * per;
  const int g = t / (8 * k.nt), gm = min(8, k.mt - g * 8);
  t -= g * 8 * k.nt;
  const int m0 = (g * 8 + t % gm) * (FN * 32), n0 = t / gm * (DUAL ? 128 : 256);
  const int range = min(a.K / 128 - split * k.per, k.per), most = (range + KW - 1) / KW;  // pairs of steps; a group's at most
  const int p0 = split * k.per + kg * most, np = kg == 0 ? most : range - most, nk = 2 * np;  // this group's, from p0 on
  const int groups = a.K / a.G, gshift = 31 - __builtin_clz((unsigned)a.G);

  // this wave's 64 rows of weights: of one matrix, or 32 of each; rows past the end repeat the last one (never stored)
  const int nw = n0 + wave * (DUAL ? 32 : 64);
  auto row_of = [&](int r) { return min(nw + (DUAL ? r % 32 : r), a.N - 1); };
  auto rsrc = [&](const void* w) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)((const unsigned char*)w + (size_t)n0 * (a.K / 2)), (short)0,
                                             min(a.N - n0, 256) * (a.K / 2), 0x00020000);
  };
  const __amdgpu_buffer_rsrc_t wr = rsrc(a.w), wr2 = rsrc(DUAL ? a.w2 : a.w);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.x + (size_t)m0 * a.K), (short)0, min(a.M - m0, FN * 32) * a.K * 2, 0x00020000);
  unsigned xp[FN], wp[4];
#pragma unroll
  for (int i = 0; i < FN; ++i) {
    int r, c;
    gemm_dma_at(wave * FN + i, lane, &r, &c);
    xp[i] = (unsigned)(min(r, a.M - 1 - m0) * a.K + c * 8) * 2;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {  // 16 rows of 64 bytes, swizzled for fragments read without bank conflicts
    const int r = i * 16 + (lane >> 2);
    wp[i] = (unsigned)((row_of(r) - n0) * (a.K / 2) + 16 * ((lane & 3) ^ (r >> 1 & 3)));
  }
  // (past the range the last step and pair again, never used: the count of loads in flight is the same everywhere)
  auto dma_x = [&](int i, int st, int slot) {
    dma16(xr, xp[i], (p0 * 128 + min(st, nk - 1) * 64) * 2, lds + slot * XB + (wave * FN + i) * 1024);
  };
  auto dma_w = [&](int i, int p) {
    dma16(DUAL && i >= 2 ? wr2 : wr, wp[i], (p0 + min(p, np - 1)) * 64, lds + T::OFF_W + (p & 1) * T::WB + wave * 4096 + i * 1024);
  };
  // lane's row of scales: row lane of this wave's 64. The two of a pair of steps lie in one aligned pair of the matrix's
  // scales (groups of 64: two; wider ones: the same one twice); N % 8 == 0 keeps the last one's in bounds
  typedef uint32_t scales_t __attribute__((ext_vector_type(FMT == 0 ? 1 : 2)));
  const unsigned char* sp = (const unsigned char*)(DUAL && hi ? a.sc2 : a.sc);
  const size_t srow = (size_t)row_of(lane) * groups;
  auto scale_at = [&](int p, int st) { return srow + (size_t)(((p0 + min(p, np - 1)) * 128 + st * 64) >> gshift); };
  scales_t sraw;
  auto fetch_scales = [&](int p) { sraw = *(const scales_t*)(sp + (scale_at(p, 0) >> 1) * sizeof(scales_t)); };
  float sc[2][2];  // [step of the pair][fragment]
  auto spread_scales = [&](int p, int st, float (&out)[2]) {  // lanes 0 .. 31's to all lanes, and lanes 32 .. 63's
    const bool odd = scale_at(p, st) & 1;
    const uint32_t v = FMT == 0 ? (odd ? sraw[0] & 0xFFFF0000u : sraw[0] << 16) : (odd ? sraw[FMT] : sraw[0]);
    const auto both = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    out[0] = __uint_as_float(both[0]), out[1] = __uint_as_float(both[1]);
  };
  u32x4 w[2][2];  // [step of the pair][fragment]: 32 packed values of lane's row
  const int w_at = T::OFF_W + wave * 4096 + l31 * 64, w_sw = l31 >> 1 & 3;
  auto read_w = [&](int p, int st, int i) {
    w[st][i] = *(const u32x4*)(lds + (p & 1) * T::WB + w_at + i * 2048 + 16 * ((st * 2 + hi) ^ w_sw));
  };
  struct Frags {
    gemm_bf16x8 w[2], x[FN];
  };
  const int x_at = l31 * 128 + 16 * ((hi * 4) ^ (l31 & 7));
  auto read_x = [&](Frags& f, int j, int slot, int m) {
    f.x[j] = *(const gemm_bf16x8*)(lds + slot * XB + (x_at ^ (16 * m)) + j * 4096);
  };

  f32x16_t acc[2][FN];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  fetch_scales(0);
#pragma unroll
  for (int i = 0; i < 4; ++i) dma_w(i, 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) dma_w(i, 1);
#pragma unroll
  for (int s = 0; s < RX - 1; ++s)
#pragma unroll
    for (int i = 0; i < FN; ++i) dma_x(i, s, s);
  gemm_wait_vm<0>();  // (all of it: the counts below hold for loads issued inside the loop)
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the codebook)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  Frags f[2];
#pragma unroll
  for (int j = 0; j < FN; ++j) read_x(f[0], j, 0, 0);
#pragma unroll
  for (int st = 0; st < 2; ++st) spread_scales(0, st, sc[st]);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    read_w(0, 0, i);
    Dequant<FMT> d;
    auto all = [&](auto self, auto p) {
      constexpr int P = decltype(p)::value;
      if constexpr (P < 8) {
        d.template part<P>(w[0][i][0], sc[0][i], tab);
        self(self, std::integral_constant<int, P + 1>{});
      }
    };
    all(all, std::integral_constant<int, 0>{});
    f[0].w[i] = __builtin_bit_cast(gemm_bf16x8, d.o);
  }
  int slot = 0, free_slot = RX - 1;  // X buffers: of this step, and the one that the last barrier freed
  // A pair of steps: eight times the matrix instructions of 16 values of K; among them the next 16 values' X fragments and
  // weights are made, and X, weights and scales of later steps set on their way
  for (int p = 0; p < np; ++p) {
    float sn[2][2];
    auto substep = [&](auto self, auto qv) {
      constexpr int q = decltype(qv)::value, st = q / 4, m = q % 4;
      constexpr int nst = (q + 1) / 4 % 2, nm = (q + 1) % 4;  // the next 16 values
      const int next = slot + 1 == RX ? 0 : slot + 1;
      if constexpr (m == 3) {
        gemm_wait_vm<T::later(8 + st)>();    // this wave's part of the next step's X has landed, ...
        __builtin_amdgcn_s_waitcnt(0xC07F);  // ... and it has read all that it reads of this one's
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      // (one wait for all reads of the 16 values of K before, not one per fragment: lgkmcnt(0))
      if constexpr (FMT == 0 && m != 3) __builtin_amdgcn_s_waitcnt(0xC07F);
      if constexpr (q == 6) gemm_wait_vm<2 * FN + 5>();  // the next pair's weights: since then two steps' X, these scales, the pair's after
      if constexpr (q == 7) sc[0][0] = sn[0][0], sc[0][1] = sn[0][1], sc[1][0] = sn[1][0], sc[1][1] = sn[1][1];
      __builtin_amdgcn_sched_barrier(0);
      const Frags& c = f[q & 1];
      Frags& n = f[(q + 1) & 1];
      const int rs = m == 3 ? next : slot;
      Dequant<FMT> d[2];
      auto element = [&](auto eself, auto ev) {
        constexpr int e = decltype(ev)::value;
        if constexpr (e < E) {
          acc[e % 2][e / 2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c.w[e % 2], c.x[e / 2], acc[e % 2][e / 2], 0, 0, 0);
          // (one wait for each row's lookups, not one per product)
          if constexpr (FMT == 1 && e == FN) __builtin_amdgcn_s_waitcnt(0xC07F | 8 << 8);        // the other row's 8 behind
          if constexpr (FMT == 1 && e == FN + FN / 2) __builtin_amdgcn_s_waitcnt(0xC07F | FN / 2 << 8);  // X behind
          // X beside the products of looked-up values, or else ahead of the loads
          constexpr int x = FMT == 1 ? e - FN : e, l = FMT == 1 || FN < 3 ? e : (FN == 3 ? e - 2 : e - FN);
          if constexpr (x >= 0 && x < FN) read_x(n, x, rs, nm);
          // lookups of both rows, then their products; without lookups row after row
          constexpr int HALF = FMT == 1 ? 4 : 8, lo = 16 * e / E, up = 16 * (e + 1) / E;
          auto parts = [&](auto pself, auto pv) {
            constexpr int P = decltype(pv)::value;
            if constexpr (P < up) {
              constexpr int round = P / (2 * HALF), i = P / HALF % 2, part = round * HALF + P % HALF;
              d[i].template part<part>(w[nst][i][nm], sc[nst][i], tab);
              pself(pself, std::integral_constant<int, P + 1>{});
            }
          };
          parts(parts, std::integral_constant<int, lo>{});
          if constexpr (q == 0 && l == 0) fetch_scales(p + 1);
          if constexpr (q == 4 && FN > 1 && l >= 0 && l < 4) dma_w(l, p + 2);
          if constexpr (q == 4 && FN == 1) dma_w(2 * e, p + 2), dma_w(2 * e + 1, p + 2);
          if constexpr (m == 1 && l >= 0 && l < FN) dma_x(l, 2 * p + st + RX - 1, free_slot);
          if constexpr (m == 2 && l >= 0 && l < 2) read_w(p + st, 1 - st, l);
          if constexpr (q == 6 && FN > 1 && (l == 2 || l == 3)) spread_scales(p + 1, l - 2, sn[l - 2]);
          if constexpr (q == 6 && FN == 1) spread_scales(p + 1, e, sn[e]);
          __builtin_amdgcn_sched_barrier(0);
          eself(eself, std::integral_constant<int, e + 1>{});
        }
      };
      element(element, std::integral_constant<int, 0>{});
      n.w[0] = __builtin_bit_cast(gemm_bf16x8, d[0].o), n.w[1] = __builtin_bit_cast(gemm_bf16x8, d[1].o);
      if constexpr (m == 3) free_slot = slot, slot = next;
      if constexpr (q < 7) self(self, std::integral_constant<int, q + 1>{});
    };
    substep(substep, std::integral_constant<int, 0>{});
  }
  gemm_wait_vm<0>();  // no DMA may outlive the workgroup's LDS

  if constexpr (KW > 1) {  // group 1's sums meet group 0's in LDS
    static_assert(FN * 32768 <= T::LDS, "sums of a group");
    if (np < most) {  // (a group with a pair less: the other's barriers)
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_s_barrier();
    }
    __syncthreads();
    f32x4_t* sums = (f32x4_t*)(lds_all + wave * (FN * 8192)) + lane;
    if (kg != 0) {
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            sums[((j * 2 + i) * 4 + e) * 64] =
                f32x4_t{acc[i][j][e * 4], acc[i][j][e * 4 + 1], acc[i][j][e * 4 + 2], acc[i][j][e * 4 + 3]};
    }
    __syncthreads();
    if (kg != 0) return;
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const f32x4_t o = sums[((j * 2 + i) * 4 + e) * 64];
#pragma unroll
          for (int c = 0; c < 4; ++c) acc[i][j][e * 4 + c] += o[c];
        }
  }
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int m = m0 + j * 32 + l31;
#pragma unroll
    for (int i = 0; i < (DUAL ? 1 : 2); ++i)
      q4d_store_fragment<DUAL>(a, acc[i][j], acc[1][j], m, nw + i * 32, hi, split, k.splits);
  }
}

template <int FMT, bool DUAL, int FN>
static void go(KArgs k, hipStream_t stream) {
  const unsigned work = (unsigned)(k.mt * k.nt * k.splits);
  gemm_q4r_kernel<FMT, DUAL, FN><<<(work + 7) / 8 * 8, 256 * Tile<FN>::KW, 0, stream>>>(k);
  if (k.splits > 1) q4d_sum(k.a, k.splits, DUAL, stream);
}
template <int FMT, bool DUAL>
static void go_rows(const KArgs& k, int fn, hipStream_t stream) {
  if (fn == 8) go<FMT, DUAL, 8>(k, stream);
  else if (fn == 6) go<FMT, DUAL, 6>(k, stream);
  else if (fn == 4) go<FMT, DUAL, 4>(k, stream);
  else if (fn == 3) go<FMT, DUAL, 3>(k, stream);
  else if (fn == 2) go<FMT, DUAL, 2>(k, stream);
  else go<FMT, DUAL, 1>(k, stream);
}

}  // namespace pr

// Rounds of 256 workgroups times their pairs of steps (128 values of K), at the clock of a full chip or, with few workgroups, a
// higher one, and their start and end; several ranges of K cost a second launch and the traffic of their sums, at a copy's rate. Of
// 462 products of 16 to 2048 rows of twelve matrices the choice is 1.1 % from the fastest of up to ten forms and ranges in the
// mean, and the ranges of the forms that stood here before 2.5 % (nf4 517 rows of 4096 x 11008 77 / 69 us, int4 400 of 8192 x
// 28672 217 / 195; int4 128 of 11008 x 4096 with SwiGLU 39.0 / 40.7). us of a pair for 256, 192 and 128 rows, measured on 256
// workgroups of K 4096: int4 2.93, 2.30, 1.75 (4740, 3870, 3140 clocks, of which 4096, 3072, 2048 of matrix instructions),
// codebooks 3.22, 2.67, 2.12 (5560, 5050, 4470: sixteen more instructions per eight weights); for 96, 64 and 32 rows from whole
// products of 86 to 240 workgroups.
// us on gemm_q4f.hip's tiles / here, int4 with weights from memory: 2048 rows of 12288 x 4096 209 / 197, 4096 x 4096 75 / 68,
// 11008 x 4096 with SwiGLU 374 / 311, 4096 x 11008 194 / 171; 517 rows 118 / 65, 71 / 37, 194 / 126, 126 / 70; 300 rows 70 / 56,
// -, 122 / 76, 90 / 49; nf4 2048 rows 233 / 212, 82 / 82, 429 / 341, 209 / 202.
// Up to 128 rows against gemm_q4d.hip's form, or the tiles where that is not taken, weights from memory:
//   97 .. 128      int4 128 rows 11008 x 4096 with SwiGLU 63 / 42, 4096 x 11008 35 / 30, 4096 x 4096 28 / 22: all here
//   33 .. 96       nf4 93 rows 28672 x 8192 with SwiGLU 150 / 124, 8192 x 28672 84 / 71; int4 64 rows 12288 x 4096 25.5 / 24.1, 11008 x
//                  4096 with SwiGLU 37 / 33. One matrix of up to 8192 columns between 2^24 and 2^26 values stays there: int4 80
//                  rows 5120 x 5120 26.1 / 27.1, 8192 x 4096 24.2 / 28.3, 4096 x 8192 25.8 / 29.4, nf4 24.6 / 27.3 and 25.8 / 28.4
//                  (4096 x 4096 23.5 / 22.1 and 24.2 / 23.2); up to 64 rows so do smaller ones of codebooks (4096 x 4096 21 / 22).
//                  And so do 8192 columns, whose partial sums it writes faster than those of 8064 (16.1 for 18.0 us, not
//                  explained): int4 48 rows, K 1536 11.6 / 15.6, with SwiGLU 14.9 / 19.6 (7168: 14.4 / 13.9, 18.0 / 18.1)
//   2 .. 32        int4 4096 x 4096 19.6 / 14.6, 11008 x 4096 with SwiGLU 32 / 28, nf4 28672 x 8192 with SwiGLU 108 / 98; 4096 x 11008
//                  20.1 / 21.1, nf4 10240 x 8192 28.9 / 30.0: beyond 2^24 values one matrix stays there, and with SwiGLU one of up
//                  to 8192 columns and 2^26 values: int4 16 rows 4096 x 8192 21.5 / 24.3, 8192 x 8192 31.8 / 34.7, 4096 x 11008
//                  24.8 / 26.4, nf4 24.0 / 25.0, 36.3 / 36.9, 28.4 / 30.4
Q4rPlan q4r_plan(int M, int N, int K, bool dual, int kernel_fmt, bool ranges) {
  Q4rPlan p{0, 0, 0, 0, 0};
  // up to 16 ranges, and up to 128 MB of their sums
  const size_t plane = (size_t)(dual ? 2 : 1) * M * N * 4;
  const int most = ranges ? (int)std::max<size_t>(std::min<size_t>(((size_t)128 << 20) / plane, 16), 1) : 1;
  const size_t nk = (size_t)N * K, one = 1;
  if (K % 128 != 0) return p;
  const bool middle = N <= 8192 && nk > one << 24;  // columns by columns of K
  if (M <= 32 && (dual ? middle && nk <= one << 26 : nk > one << 24)) return p;
  if (!dual && M > 32 && M <= 64 && kernel_fmt == 1 && nk < one << 26) return p;
  if (!dual && M > 32 && M <= 96 && middle && nk < one << 26) return p;
  if (N == 8192 && K >= 1536 && K <= 2560 && M > 32 && M <= (dual ? 64 : 96)) return p;
  const int cols = dual ? 128 : 256, np = K / 128;
  p.nt = (N + cols - 1) / cols;
  constexpr int forms[] = {8, 6, 4, 3, 2, 1};
  const float pair_us[2][6] = {{2.93f, 2.30f, 1.75f, 1.65f, 1.40f, 1.05f}, {3.22f, 2.67f, 2.12f, 1.85f, 1.55f, 1.42f}};
  const float fast_us[2][6] = {{1.97f, 1.61f, 1.31f, 1.12f, 0.97f, 0.90f}, {2.32f, 2.10f, 1.86f, 1.40f, 1.28f, 1.19f}};
  float best = 0.0f;
  for (int i = 0; i < 6; ++i) {
    const int fn = forms[i], mt = (M + fn * 32 - 1) / (fn * 32);
    const float slow = pair_us[kernel_fmt][i], fast = fast_us[kernel_fmt][i], ends = fn < 4 ? 4.0f : 2.0f + fn;
    for (int s = 1; s <= most && (s == 1 || np / s >= 2); ++s) {
      const int per = (np + s - 1) / s, used = (np + per - 1) / per;
      if (fn < 4 && np - per * (used - 1) < 2) continue;  // (a pair for each half)
      const float rounds = (float)((long)mt * p.nt * used) / 256.0f, whole = floorf(rounds);
      float us = whole * (per * slow + ends);
      if (rounds > whole) us += per * fmaxf(fast, slow * (0.3f + 0.7f * (rounds - whole))) + ends;
      if (used > 1) us += 2.0f + 0.25f * used + (float)plane * (used + 1) / 4.75e6f;
      if (p.fn == 0 || us < best) best = us, p.fn = fn, p.mt = mt, p.splits = used, p.per = per;
    }
  }
  return p;
}

size_t q4r_workspace(const Q4rPlan& p, int M, int N, bool dual) {
  return p.splits > 1 ? 4096 + (size_t)p.splits * (dual ? 2 : 1) * M * N * 4 : 0;
}

int q4r_run(const Q4dArgs& a, const Q4rPlan& p, int kernel_fmt, bool dual, hipStream_t stream) {
  const pr::KArgs k{a, p.mt, p.nt, p.splits, p.per};
  switch (kernel_fmt * 2 + (dual ? 1 : 0)) {
    case 0: pr::go_rows<0, false>(k, p.fn, stream); break;
    case 1: pr::go_rows<0, true>(k, p.fn, stream); break;
    case 2: pr::go_rows<1, false>(k, p.fn, stream); break;
    default: pr::go_rows<1, true>(k, p.fn, stream); break;
  }
  LGA_LAUNCH_RETURN();
}

int preload_gemm_q4r() {
  using namespace pr;
  int bad = 0;
#define LGA_PRE(F, D) \
  bad += preload(gemm_q4r_kernel<F, D, 1>) + preload(gemm_q4r_kernel<F, D, 2>) + preload(gemm_q4r_kernel<F, D, 3>) + \
         preload(gemm_q4r_kernel<F, D, 4>) + preload(gemm_q4r_kernel<F, D, 6>) + preload(gemm_q4r_kernel<F, D, 8>)
  LGA_PRE(0, false);
  LGA_PRE(0, true);
  LGA_PRE(1, false);
  LGA_PRE(1, true);
#undef LGA_PRE
  return bad;
}

}  // namespace lga
