// The large products of the layered models' prompts: Y (+)= act(A W^T + bias) with A and W in bf16, sums in fp32, on the
// pipelined tiles of gemm_tiles.h.
#include "seq_gemm.h"

#include "gemm_tiles.h"

namespace lgs {

using lga::GemmTile;
using lga::f32x16_t;
using lga::gemm_tile;

// grouped rows: the batch whose tiles hold number t, the batches' tiles counted side by side over the lanes; t becomes the
// number inside the batch
template <int ROWS>
__device__ __forceinline__ bool gemm_group(const int* z_start, int batch, int nt, int lane, int* t_at, int* z_at) {
  int t = *t_at, z = 0;
  bool found = false;
  for (int e0 = 0; e0 < batch && !found; e0 += 64) {
    const int e = e0 + lane;
    const int rows = e < batch ? z_start[e + 1] - z_start[e] : 0;
    const int own = (rows + ROWS - 1) / ROWS * nt;
    int upto = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(upto, o);
      if (lane >= o) upto += v;
    }
    const unsigned long long past = __ballot(upto > t);
    if (past) {
      const int l = __ffsll(past) - 1;
      z = e0 + l;
      t -= __shfl(upto - own, l);
      found = true;
    } else {
      t -= __shfl(upto, 63);
    }
  }
  if (!found) return false;
  z = __builtin_amdgcn_readfirstlane(z);
  t = __builtin_amdgcn_readfirstlane(t);
  *t_at = t;
  *z_at = z;
  return true;
}

// Bound by the matrix cores' feeding: without its DMAs the 256 x 256 form runs 1.3 times as fast, without its fragment
// reads 1.1 times, without both at the matrix cores' rate (2.1 PFLOP/s). Results go straight to memory, past the caches
// (a lane's rows in 128-byte pieces): turning them in LDS into longer pieces cost 14 us a tile.
//
// Workgroup b runs on XCD b % 8, and an XCD takes neighbouring tiles, whose rows of A and W its L2 then holds.
template <int WM, int WN, int FM, int FN, int BK, int ST>
__global__ void __launch_bounds__(WM* WN * 64) gemm_kernel(LinArgs p, int mt, int nt, int batch) {
  using T = GemmTile<WM, WN, FM, FN, BK, ST>;
  constexpr int P = T::P;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[ST * T::STAGE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int t = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  int z = 0, split = 0, r_lo = 0, Mz = p.M, m, n;
  if (p.z_start) {
    if (!gemm_group<T::BM>(p.z_start, batch, nt, lane, &t, &z)) return;
    r_lo = p.z_start[z];
    Mz = p.z_start[z + 1] - r_lo;
    const int mz = (Mz + T::BM - 1) / T::BM;
    m = t % mz;
    n = t / mz;
  } else {
    const int per = mt * nt;
    const int which = t / per;
    if (which >= batch * p.ksplit) return;
    if (p.ksplit > 1) split = which;
    else z = which;
    t -= which * per;
    const int g = t / (8 * nt), gm = min(8, mt - g * 8);  // groups of up to 8 row tiles
    t -= g * 8 * nt;
    m = g * 8 + t % gm;
    n = t / gm;
  }
  const int m0 = m * T::BM, n0 = n * T::BN;
  int nk = p.K / BK, k0 = 0;
  if (p.ksplit > 1) {  // (kper counts 64 values of K)
    k0 = split * p.kper * T::RPL;
    nk = min(nk - k0, p.kper * T::RPL);
  }
  // DMA sources: lane -> LDS row lane / 8 of the piece, the 16-byte chunk of it that the swizzle places at lane % 8
  const unsigned char* src[P];
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int piece = wave * P + i;
    const bool of_a = piece < T::BM / T::ROWS;  // (wave-uniform)
    int r, c;
    lga::gemm_dma_at<BK>((of_a ? piece : piece - T::BM / T::ROWS) * 8 + (lane >> 3), lane, &r, &c);
    if (of_a) {
      const int lr = r_lo + min(m0 + r, Mz - 1);  // rows past the end repeat the last one (never stored)
      src[i] = (const unsigned char*)(p.a16 + (size_t)z * p.sa + (size_t)(p.a_rows ? p.a_rows[lr] : lr) * p.lda);
    } else {
      src[i] = (const unsigned char*)((const uint16_t*)p.w + (size_t)z * p.sw + (size_t)min(n0 + r, p.N - 1) * p.K);
    }
    src[i] += (size_t)k0 * (BK * 2) + c * 16;
  }
  f32x16_t acc[FM][FN];
  gemm_tile<WM, WN, FM, FN, BK, ST>(lds, src, nk, wave, lane, acc);
  const int wm = wave % WM, wn = wave / WM, l31 = lane & 31, hi = lane >> 5;
  // a lane holds column l31 of a fragment and its rows 8 (e / 4) + 4 hi + e % 4
  const int row0 = m0 + wm * FM * 32 + hi * 4, col0 = n0 + wn * FN * 32 + l31;
  auto each = [&](auto&& put) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int r = i * 32 + (e >> 2) * 8 + (e & 3);
        if (row0 + r < Mz)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            if (col0 + j * 32 < p.N) put(r, j, acc[i][j][e]);
      }
  };
  if (p.ksplit > 1) {
    float* y = p.part + ((size_t)split * p.M + row0) * p.N + col0;
    each([&](int r, int j, float v) { y[(long)r * p.N + j * 32] = v; });
    return;
  }
  float bias[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) bias[j] = p.bias ? p.bias[min(col0 + j * 32, p.N - 1)] : 0.0f;
  const long at = (long)z * p.sy + (long)(r_lo + row0) * p.ldy + col0;
  if (p.act != kActNone) {  // (few products have one: a loop that keeps the code small)
    each([&](int r, int j, float v) {
      v = act_f(p.act, v + bias[j]);
      const long o = at + (long)r * p.ldy + j * 32;
      if (p.y16) p.y16[o] = f2bf(v);
      else p.y[o] = p.accumulate ? p.y[o] + v : v;
    });
  } else if (p.y16) {
    each([&](int r, int j, float v) { p.y16[at + (long)r * p.ldy + j * 32] = f2bf(v + bias[j]); });
  } else if (p.accumulate) {
    each([&](int r, int j, float v) { p.y[at + (long)r * p.ldy + j * 32] += v + bias[j]; });
  } else {
    each([&](int r, int j, float v) { __builtin_nontemporal_store(v + bias[j], p.y + at + (long)r * p.ldy + j * 32); });
  }
}

template <int WM, int WN, int FM, int FN, int BK, int ST>
static int gemm_go(const LinArgs& p, int batch, hipStream_t stream) {
  using T = GemmTile<WM, WN, FM, FN, BK, ST>;
  const int mt = (p.M + T::BM - 1) / T::BM, nt = (p.N + T::BN - 1) / T::BN;
  const long tiles = p.z_start ? (long)(mt + batch) * nt : (long)mt * nt * batch * p.ksplit;
  LGA_CHECK_ARG(tiles < (1L << 30), "lgs_linear: too many tiles");
  gemm_kernel<WM, WN, FM, FN, BK, ST><<<(unsigned)((tiles + 7) / 8 * 8), T::NT, 0, stream>>>(p, mt, nt, batch);
  return 0;
}

// act(gate) * up with the gate's and the up's rows of W in turn as the tile's A, 32 of each: the pair of a column meets in
// one lane, which has four neighbouring columns of a row and stores them rounded to bf16. Two passes over fp32 results of
// twice the width and a launch less than the product and its unit apart, whose bits it gives: 511 us for 2407 rows, twice
// 11008 columns and K 4096 in a model's prompt, where the two took 497 and 82.
template <int WM, int WN, int FM, int FN, int BK, int ST, bool CLAMPED>
__global__ void __launch_bounds__(WM* WN * 64) gemm_glu_kernel(LinArgs p, GluForm f, int mt, int nt, int batch) {
  using T = GemmTile<WM, WN, FM, FN, BK, ST>;
  constexpr int P = T::P;
  static_assert(FM % 2 == 0, "fragments of the two matrices in pairs");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[ST * T::STAGE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int t = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  int z = 0, r_lo = 0, Mz = p.M, m, n;
  if (p.z_start) {
    if (!gemm_group<T::BN>(p.z_start, batch, nt, lane, &t, &z)) return;
    r_lo = p.z_start[z];
    Mz = p.z_start[z + 1] - r_lo;
    const int mz = (Mz + T::BN - 1) / T::BN;
    m = t % mz, n = t / mz;
  } else {
    if (t >= mt * nt) return;
    const int g = t / (8 * nt), gm = min(8, mt - g * 8);  // groups of up to 8 row tiles
    t -= g * 8 * nt;
    m = g * 8 + t % gm, n = t / gm;
  }
  const int m0 = m * T::BN, n0 = n * (T::BM / 2);
  const unsigned char* src[P];
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int piece = wave * P + i;
    const bool of_w = piece < T::BM / T::ROWS;  // (wave-uniform)
    int r, c;
    lga::gemm_dma_at<BK>((of_w ? piece : piece - T::BM / T::ROWS) * 8 + (lane >> 3), lane, &r, &c);
    if (of_w) {  // columns past the end repeat the last one (never stored)
      const int col = min(n0 + r / 64 * 32 + r % 32, p.N - 1);
      src[i] = (const unsigned char*)((const uint16_t*)p.w + (size_t)z * p.sw + (r / 32 % 2 ? f.up : 0) + (size_t)col * p.K);
    } else {
      const int lr = r_lo + min(m0 + r, Mz - 1);
      src[i] = (const unsigned char*)(p.a16 + (size_t)(p.a_rows ? p.a_rows[lr] : lr) * p.lda);
    }
    src[i] += c * 16;
  }
  f32x16_t acc[FM][FN];
  gemm_tile<WM, WN, FM, FN, BK, ST>(lds, src, p.K / BK, wave, lane, acc);
  const int wm = wave % WM, wn = wave / WM, l31 = lane & 31, hi = lane >> 5;
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int row = m0 + (wn * FN + j) * 32 + l31;
    if (row >= Mz) continue;
#pragma unroll
    for (int i = 0; i < FM; i += 2)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int col = n0 + (wm * FM + i) * 16 + q * 8 + hi * 4;
        if (col >= p.N) continue;
        uint32_t o[2];
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          const float a = glu_f<CLAMPED>(f, acc[i][j][q * 4 + e], acc[i + 1][j][q * 4 + e]);
          const float b = glu_f<CLAMPED>(f, acc[i][j][q * 4 + e + 1], acc[i + 1][j][q * 4 + e + 1]);
          o[e / 2] = (uint32_t)f2bf(a) | (uint32_t)f2bf(b) << 16;
        }
        *(uint2*)(p.y16 + (size_t)(r_lo + row) * p.ldy + col) = make_uint2(o[0], o[1]);
      }
  }
}

template <int WM, int WN, int FM, int FN, int BK, int ST>
static int glu_go(const LinArgs& p, const GluForm& f, int batch, hipStream_t stream) {
  using T = GemmTile<WM, WN, FM, FN, BK, ST>;
  const int mt = (p.M + T::BN - 1) / T::BN, nt = (p.N + T::BM / 2 - 1) / (T::BM / 2);
  const long tiles = p.z_start ? (long)(mt + batch) * nt : (long)mt * nt;
  LGA_CHECK_ARG(tiles < (1L << 30), "lgs_linear_glu: too many tiles");
  const unsigned grid = (unsigned)((tiles + 7) / 8 * 8);
  if (f.clamped) gemm_glu_kernel<WM, WN, FM, FN, BK, ST, true><<<grid, T::NT, 0, stream>>>(p, f, mt, nt, batch);
  else gemm_glu_kernel<WM, WN, FM, FN, BK, ST, false><<<grid, T::NT, 0, stream>>>(p, f, mt, nt, batch);
  return 0;
}

int gemm_glu_launch(const LinArgs& p, const GluForm& f, int batch, hipStream_t stream) {
#define LGS_CASE(I, SLOTS, US, ...) \
  case I: return glu_go<__VA_ARGS__>(p, f, batch, stream);
  switch (lga::gemm_tile_plan(p.M, 2 * p.N, p.K, batch, p.z_start != nullptr, 1, true).tile) { LGA_GEMM_FORMS(LGS_CASE) }
#undef LGS_CASE
  lga_set_error("lgs_linear_glu: no such form");
  return (int)hipErrorInvalidValue;
}

GemmPlan gemm_plan(int M, int N, int K, int batch, bool grouped, int ksplit) {
  if (grouped && gemm_few_rows(M, batch)) return GemmPlan{-1, 1};
  return lga::gemm_tile_plan(M, N, K, batch, grouped, ksplit);
}

int gemm_launch(const LinArgs& p, const GemmPlan& plan, int batch, hipStream_t stream) {
#define LGS_CASE(I, SLOTS, US, ...) \
  case I: return gemm_go<__VA_ARGS__>(p, batch, stream);
  switch (plan.tile) { LGA_GEMM_FORMS(LGS_CASE) }
#undef LGS_CASE
  lga_set_error("lgs_linear: no such form");
  return (int)hipErrorInvalidValue;
}

}  // namespace lgs
