// Prompt products with bf16 weights, Y = X W^T with bias / residual, and fc_1 || fc_2 + SwiGLU, on the pipelined tiles of
// gemm_tiles.h. The weights are the tile's A: two lanes then hold eight neighbouring columns of one row of Y, four each, swap halves
// and store 16 bytes, and for SwiGLU a wave's fragments alternate between the two matrices, so that the pair of a column
// meets in one lane.
//
// Bound as the tiles are; with few rows by the weights on their way from memory. With weights from memory, us on stages of 32
// values / here: of 517 rows (N x K) 12288 x 4096 70 / 65, 4096 x 4096 36 / 35, 4096 x 11008 68 / 71, 11008 x 4096 with
// SwiGLU 131 / 119; of 2048 rows 12288 x 4096 195 / 178, 4096 x 11008 181 / 162, 6144 x 4096 with SwiGLU 209 / 192.
#include "gemm_q4d.h"
#include "gemm_tiles.h"

namespace lga {

struct BfArgs {
  Q4dArgs a;
  int nt, splits, kper;  // tiles over columns; ranges of K of kper stages of 64 values
};

// the tile at rows m0 .. and columns n0 .. of range `split`
template <int WM, int WN, int FM, int FN, int RA, int RB, bool DUAL>
__device__ __forceinline__ void bf16_rows(const BfArgs& k, unsigned char* lds, int split, int m0, int n0) {
  using T = GemmTile<WM, WN, FM, FN, RA, RB>;
  static_assert(!DUAL || FM % 2 == 0, "fragments of the two matrices in pairs");
  const Q4dArgs& a = k.a;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int k0 = split * k.kper, nk = min(a.K / 64 - k0, k.kper);
  const unsigned char *src_w[T::PA], *src_x[T::PB];
  int r, c;
#pragma unroll
  for (int i = 0; i < T::PA; ++i) {  // columns past the end repeat the last one (never stored)
    gemm_dma_at(wave * T::PA + i, lane, &r, &c);
    const int n = DUAL ? r / 64 * 32 + r % 32 : r;
    const void* w = DUAL && r / 32 % 2 ? a.w2 : a.w;
    src_w[i] = (const unsigned char*)((const uint16_t*)w + (size_t)min(n0 + n, a.N - 1) * a.K) + (size_t)k0 * 128 + c * 16;
  }
#pragma unroll
  for (int i = 0; i < T::PB; ++i) {
    gemm_dma_at(wave * T::PB + i, lane, &r, &c);
    src_x[i] = (const unsigned char*)(a.x + (size_t)min(m0 + r, a.M - 1) * a.K) + (size_t)k0 * 128 + c * 16;
  }
  f32x16_t acc[FM][FN];
  gemm_tile<WM, WN, FM, FN, RA, RB>(lds, src_w, src_x, nk, wave, lane, acc);
  const int wm = wave % WM, wn = wave / WM, l31 = lane & 31, hi = lane >> 5;
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int m = m0 + (wn * FN + j) * 32 + l31;
#pragma unroll
    for (int i = 0; i < FM; i += DUAL ? 2 : 1)
      q4d_store_fragment<DUAL>(a, acc[i][j], acc[i + (DUAL ? 1 : 0)][j], m, n0 + (wm * FM + i) * (DUAL ? 16 : 32), hi, split, k.splits);
  }
}

template <int WM, int WN, int FM, int FN, int MOST, bool DUAL, int F = FN - 1>
__device__ __forceinline__ void bf16_short(const BfArgs& k, unsigned char* lds, int split, int m0, int n0, int frags) {
  if constexpr (F > 0) {
    using S = GemmShort<WM, WN, FM, F, MOST>;
    if (frags == F) bf16_rows<WM, WN, FM, F, S::RA, S::RB, DUAL>(k, lds, split, m0, n0);
    else bf16_short<WM, WN, FM, FN, MOST, DUAL, F - 1>(k, lds, split, m0, n0, frags);
  }
}

// (an XCD takes neighbouring tiles: of a column's weights those of up to eight row tiles, range after range. All of a column's on
// one XCD: 517 x 12288 x 4096 with weights from memory 70 -> 62 us)
template <int WM, int WN, int FM, int FN, int RA, int RB, bool DUAL>
__global__ void __launch_bounds__(WM* WN * 64) gemm_bf16_kernel(BfArgs k) {
  using T = GemmTile<WM, WN, FM, FN, RA, RB>;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[FN > 1 ? kGemmLds<T> : T::LDS];
  GemmAt at;
  if (!gemm_at<T::BN, WN * 32>(k.a.M, k.nt, k.splits, &at)) return;
  const int m0 = at.m * T::BN, n0 = at.n * (DUAL ? T::BM / 2 : T::BM), frags = (k.a.M - m0 + WN * 32 - 1) / (WN * 32);
  if (frags >= FN) bf16_rows<WM, WN, FM, FN, RA, RB, DUAL>(k, lds, at.which, m0, n0);
  else bf16_short<WM, WN, FM, FN, kGemmLds<T>, DUAL>(k, lds, at.which, m0, n0, frags);
}

template <int WM, int WN, int FM, int FN, int RA, int RB>
static void bf16_go(BfArgs k, bool dual, hipStream_t stream) {
  using T = GemmTile<WM, WN, FM, FN, RA, RB>;
  const int bn = dual ? T::BM / 2 : T::BM;
  k.nt = (k.a.N + bn - 1) / bn;
  const unsigned grid = gemm_grid((long)k.nt * ((k.a.M + T::BN - 1) / T::BN) * k.splits);
  if constexpr (FM % 2 == 0) {
    if (dual) gemm_bf16_kernel<WM, WN, FM, FN, RA, RB, true><<<grid, T::NT, 0, stream>>>(k);
  }
  if (!dual) gemm_bf16_kernel<WM, WN, FM, FN, RA, RB, false><<<grid, T::NT, 0, stream>>>(k);
}

// All products but those of few rows and small weights, where a launch over ranges of K and one that adds them are not repaid
// (us here / on gemm_q4f.hip's tiles): 16 x 4096 x 4096 20 / 14, 16 x 4096 x 11008 26 / 23, against 38 / 39 for 8192 x 8192
// (2^26). More than 1024 rows that fill the chip keep K whole.
GemmPlan bf16_plan(int M, int N, int K, bool dual) {
  const long cols = dual ? 2L * N : N;
  if (M <= 32 && cols * K < 1L << 26) return GemmPlan{-1, 1};
  const bool full = M > 1024 && (M + 255) / 256 * (cols / 128) >= 256;
  return gemm_tile_plan(M, (int)cols, K, 1, false, full ? 1 : 0, kGemmRowsB | (dual ? kGemmPairs : 0));
}

// (its number among the forms, and behind eight bits the ranges of K; -1: not on these tiles)
extern "C" int lga_bf16_gemm_form(int M, int N, int K, int swiglu) {
  if (M <= 0 || N <= 0 || K <= 0) return -1;
  const GemmPlan p = bf16_plan(M, N, K, swiglu != 0);
  return p.tile < 0 ? -1 : p.tile | p.ksplit << 8;
}

size_t bf16_workspace(const GemmPlan& p, int M, int N, bool dual) {
  return p.ksplit > 1 ? 4096 + (size_t)p.ksplit * (dual ? 2 : 1) * M * N * 4 : 0;
}

int bf16_run(const Q4dArgs& a, const GemmPlan& p, bool dual, hipStream_t stream) {
  const int steps = a.K / 64, kper = (steps + p.ksplit - 1) / p.ksplit;
  const BfArgs k{a, 0, (steps + kper - 1) / kper, kper};
  switch (p.tile) {
#define LGA_CASE(I, SLOTS, US, FAST, ROUND, ...) \
  case I: bf16_go<__VA_ARGS__>(k, dual, stream); break;
    LGA_GEMM_FORMS(LGA_CASE)
#undef LGA_CASE
  }
  if (k.splits > 1) q4d_sum(a, k.splits, dual, stream);
  LGA_LAUNCH_RETURN();
}

template <int WM, int WN, int FM, int FN, int RA, int RB>
static int bf16_preload() {
  int bad = preload(gemm_bf16_kernel<WM, WN, FM, FN, RA, RB, false>);
  if constexpr (FM % 2 == 0) bad += preload(gemm_bf16_kernel<WM, WN, FM, FN, RA, RB, true>);
  return bad;
}
int preload_gemm_bf16() {
  int bad = 0;
#define LGA_PRE(I, SLOTS, US, FAST, ROUND, ...) bad += bf16_preload<__VA_ARGS__>();
  LGA_GEMM_FORMS(LGA_PRE)
#undef LGA_PRE
  return bad;
}

}  // namespace lga
