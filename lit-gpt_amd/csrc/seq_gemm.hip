// The large products of the layered models' prompts: Y (+)= act(A W^T + bias) with A and W in bf16, sums in fp32, on the
// pipelined tiles of gemm_tiles.h.
#include "seq_gemm.h"

#include <algorithm>

#include "gemm_tiles.h"

namespace lgs {

using lga::GemmTile;
using lga::f32x16_t;
using lga::gemm_tile;

// grouped rows: this workgroup's tile, z its batch and m, n its place inside it, a short one beside the whole ones of its columns
// (false: none is left). The batches' tiles are
// counted side by side over the lanes, and every XCD takes an eighth of those that there are: the grid is the largest number that the
// groups' sizes allow, of which a third stayed empty and with it the last XCDs (16 groups of 512 rows of 2 x 1408 x 2048: 3 rounds on 5
// XCDs instead of 2 on all, 216 -> 125 us).
template <int ROWS>
__device__ __forceinline__ bool gemm_group(const int* z_start, int batch, int nt, int lane, lga::GemmAt* o) {
  auto count = [&](int e, int* mt) {  // batch e's *mt row tiles, and the tiles of those of this lane and of all before it
    *mt = e < batch ? (z_start[e + 1] - z_start[e] + ROWS - 1) / ROWS : 0;
    int upto = *mt * nt;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int u = __shfl_up(upto, d);
      if (lane >= d) upto += u;
    }
    return upto;
  };
  int total = 0, mt, t;
  for (int e0 = 0; e0 < batch; e0 += 64) total += __shfl(count(e0 + lane, &mt), 63);
  if (!lga::gemm_xcd(total, 0, &t)) return false;
  for (int e0 = 0; e0 < batch; e0 += 64) {
    const int upto = count(e0 + lane, &mt);
    const unsigned long long past = __ballot(upto > t);
    if (past) {
      const int at = __ffsll(past) - 1;
      t = __builtin_amdgcn_readfirstlane(t - __shfl(upto - mt * nt, at));
      mt = __builtin_amdgcn_readfirstlane(__shfl(mt, at));
      o->which = __builtin_amdgcn_readfirstlane(e0 + at);
      o->m = t % mt, o->n = t / mt;
      return true;
    }
    t -= __shfl(upto, 63);
  }
  return false;
}

// an activation on more accumulators than these is code past what the compiler unrolls (it then keeps them in memory)
template <int FM, int FN>
constexpr bool kActsFit = FM * FN <= 8;

// Bound by the matrix cores and the power that they take (gemm_tiles.h); start, end and the results of a round of 256 x 256
// tiles cost 15 us, of 256 x 128 8. Results go straight to memory, past the caches (a lane's rows in 128-byte pieces):
// turning them in LDS into longer pieces cost 14 us a tile.
//
// The tile at rows m0 .. of batch z, whose list has Mz rows from r_lo on, and columns n0 ..
template <int WM, int WN, int FM, int FN, int RA, int RB, bool SHORT, bool ACTS>
__device__ __forceinline__ void gemm_rows(const LinArgs& p, unsigned char* lds, int z, int split, int r_lo, int Mz, int m0, int n0) {
  using T = GemmTile<WM, WN, FM, FN, RA, RB>;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int nk = p.K / 64, k0 = 0;
  if (p.ksplit > 1) {
    k0 = split * p.kper;
    nk = min(nk - k0, p.kper);
  }
  const unsigned char *src_a[T::PA], *src_w[T::PB];
  int r, c;
#pragma unroll
  for (int i = 0; i < T::PA; ++i) {
    lga::gemm_dma_at(wave * T::PA + i, lane, &r, &c);
    const int lr = r_lo + min(m0 + r, Mz - 1);  // rows past the end repeat the last one (never stored)
    src_a[i] = (const unsigned char*)(p.a16 + (size_t)z * p.sa + (size_t)(p.a_rows ? p.a_rows[lr] : lr) * p.lda) +
               (size_t)k0 * 128 + c * 16;
  }
#pragma unroll
  for (int i = 0; i < T::PB; ++i) {
    lga::gemm_dma_at(wave * T::PB + i, lane, &r, &c);
    src_w[i] = (const unsigned char*)((const uint16_t*)p.w + (size_t)z * p.sw + (size_t)min(n0 + r, p.N - 1) * p.K) +
               (size_t)k0 * 128 + c * 16;
  }
  f32x16_t acc[FM][FN];
  gemm_tile<WM, WN, FM, FN, RA, RB>(lds, src_a, src_w, nk, wave, lane, acc);
  // a lane holds column l31 of a fragment and its rows 8 (e / 4) + 4 hi + e % 4: the wave's rows and columns begin at
  // (mw, nw); a row's address is the wave's, a lane's place in it 32 bits
  const int wm = wave % WM, wn = wave / WM, l31 = lane & 31, hi = lane >> 5;
  const int mw = m0 + wm * FM * 32, nw = n0 + wn * FN * 32;
  const bool inside = mw + FM * 32 <= Mz && nw + FN * 32 <= p.N;
  // y: (mw, nw). R rows of a fragment at a time: the old values of sums on their way together, then the results, then the stores.
  // (More, and all accumulators are fetched ahead, into memory; row by row, the latency of a load or an activation stands
  // between any two rows.)
  constexpr int FEW = FM * FN > 12 ? 1 : 4;
  auto each = [&](auto in, auto sums, auto past, auto rows_at_once, auto* y, long ld, auto&& make) __attribute__((always_inline)) {
    constexpr bool IN = decltype(in)::value, SUMS = decltype(sums)::value;
    constexpr int R = decltype(rows_at_once)::value;
    const unsigned at = (unsigned)(hi * 4 * (int)ld + l31);
    const int rows = Mz - 1 - mw - hi * 4, cols = p.N - 1 - nw - l31;  // a lane's last ones
    if constexpr (!SUMS) lga::wait_loads();
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int q = 0; q < 16; q += R) {
        const int r0 = i * 32 + q / 4 * 8 + q % 4;
        float old[R][FN];
        std::remove_reference_t<decltype(*y)> v[R][FN];
        if constexpr (SUMS) {
#pragma unroll
          for (int e = 0; e < R; ++e)
#pragma unroll
            for (int j = 0; j < FN; ++j)  // (past the end the last ones, not used)
              old[e][j] = IN ? (y + (long)(r0 + e) * ld + j * 32)[at] : y[(long)(min(r0 + e, rows) + hi * 4) * ld + l31 + min(j * 32, cols)];
        }
#pragma unroll
        for (int e = 0; e < R; ++e)
#pragma unroll
          for (int j = 0; j < FN; ++j) v[e][j] = make(j, acc[i][j][q + e], SUMS ? old[e][j] : 0.0f);
#pragma unroll
        for (int e = 0; e < R; ++e) {
          auto* row = y + (long)(r0 + e) * ld;
          if (IN || r0 + e <= rows)
#pragma unroll
            for (int j = 0; j < FN; ++j)
              if (IN || j * 32 <= cols) {
                if constexpr (decltype(past)::value) __builtin_nontemporal_store(v[e][j], row + j * 32 + at);
                else (row + j * 32)[at] = v[e][j];
              }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
  };
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  constexpr std::integral_constant<int, 1> one{};
  constexpr std::integral_constant<int, FEW> few{};
  auto put = [&](auto sums, auto past, auto n, auto* y, long ld, auto&& make) __attribute__((always_inline)) {
    if constexpr (!SHORT) {
      if (inside) return each(yes, sums, past, n, y, ld, make);
    }
    each(no, sums, past, n, y, ld, make);
  };
  if (p.ksplit > 1) {
    put(no, no, one, p.part + ((size_t)split * p.M + mw) * p.N + nw, p.N, [](int, float v, float) { return v; });
    return;
  }
  float bias[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) bias[j] = p.bias ? p.bias[min(nw + l31 + j * 32, p.N - 1)] : 0.0f;
  // (here and at each list of stores: or, in tiles that rows or columns end in, every store waits for the one before. us: 1000 rows of
  // 6288 x 2048 36.3 / 29.6, 1500 52.0 / 41.6, of 4096 x 4096 53.8 / 49.7, 2407 of 2048 x 2048 29.4 / 25.1; 16 groups of 512 rows of 1024
  // x 1024 41.5 / 29.4)
  lga::wait_loads(bias);
  const long at = (long)z * p.sy + (long)(r_lo + mw) * p.ldy + nw;
  if (ACTS && p.act != kActNone) {
    if constexpr (ACTS) {
      // (a loop of its own for each activation: a choice per result keeps them from standing among one another. Into sums: 2084 rows of
      // 3159 x 256, silu, 46.1 -> 33.8 us, 832 of 9600 x 1408 97 -> 77.7, 264 of 20528 x 1152 59.7 -> 46.2)
      auto act = [&](auto kind) __attribute__((always_inline)) {
        auto f = [&](int j, float v, float) { return act_f(decltype(kind)::value, v + bias[j]); };
        if (p.y16) each(no, no, no, few, p.y16 + at, p.ldy, [&](int j, float v, float) { return f2bf(f(j, v, 0.0f)); });
        else if (p.accumulate) each(no, yes, no, few, p.y + at, p.ldy, [&](int j, float v, float old) {
#pragma clang fp contract(off)
          return old + f(j, v, 0.0f);
        });
        else each(no, no, no, few, p.y + at, p.ldy, f);
      };
      if (p.act == kActRelu2) act(std::integral_constant<int, kActRelu2>{});
      else if (p.act == kActGeluTanh) act(std::integral_constant<int, kActGeluTanh>{});
      else if (p.act == kActSilu) act(std::integral_constant<int, kActSilu>{});
      else act(std::integral_constant<int, kActSigmoid>{});
    }
  } else if (p.y16) {
    put(no, no, one, p.y16 + at, p.ldy, [&](int j, float v, float) { return f2bf(v + bias[j]); });
  } else if (p.accumulate) {
    put(yes, no, few, p.y + at, p.ldy, [&](int j, float v, float old) { return old + (v + bias[j]); });
  } else {
    put(no, yes, one, p.y + at, p.ldy, [&](int j, float v, float) { return v + bias[j]; });
  }
}

// f: fragments along the rows that have one, FM and less
template <int WM, int WN, int FM, int FN, int MOST, int F = FM - 1>
__device__ __forceinline__ void gemm_short(const LinArgs& p, unsigned char* lds, int z, int split, int r_lo, int Mz, int m0, int n0, int f) {
  if constexpr (F > 0) {
    using S = lga::GemmShort<WM, WN, F, FN, MOST>;
    if (f == F) gemm_rows<WM, WN, F, FN, S::RA, S::RB, true, kActsFit<FM, FN>>(p, lds, z, split, r_lo, Mz, m0, n0);
    else gemm_short<WM, WN, FM, FN, MOST, F - 1>(p, lds, z, split, r_lo, Mz, m0, n0, f);
  }
}

template <int WM, int WN, int FM, int FN, int RA, int RB>
__global__ void __launch_bounds__(WM* WN * 64) gemm_kernel(LinArgs p, int nt, int batch) {
  using T = GemmTile<WM, WN, FM, FN, RA, RB>;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[FM > 1 ? lga::kGemmLds<T> : T::LDS];
  lga::GemmAt at;
  int z = 0, split = 0, r_lo = 0, Mz = p.M;
  if (p.z_start) {
    if (!gemm_group<T::BM>(p.z_start, batch, nt, threadIdx.x & 63, &at)) return;
    z = at.which;
    r_lo = p.z_start[z];
    Mz = p.z_start[z + 1] - r_lo;
  } else {
    if (!lga::gemm_at<T::BM, WM * 32>(Mz, nt, batch * p.ksplit, &at)) return;
    if (p.ksplit > 1) split = at.which;
    else z = at.which;
  }
  const int m0 = at.m * T::BM, n0 = at.n * T::BN, f = (Mz - m0 + WM * 32 - 1) / (WM * 32);
  if (f >= FM) gemm_rows<WM, WN, FM, FN, RA, RB, false, kActsFit<FM, FN>>(p, lds, z, split, r_lo, Mz, m0, n0);
  else gemm_short<WM, WN, FM, FN, lga::kGemmLds<T>>(p, lds, z, split, r_lo, Mz, m0, n0, f);
}

template <int WM, int WN, int FM, int FN, int RA, int RB>
static int gemm_go(const LinArgs& p, int batch, hipStream_t stream) {
  using T = GemmTile<WM, WN, FM, FN, RA, RB>;
  const long mt = (p.M + T::BM - 1) / T::BM, nt = (p.N + T::BN - 1) / T::BN;
  const long tiles = p.z_start ? (mt + batch) * nt : mt * nt * batch * p.ksplit;
  LGA_CHECK_ARG(tiles < (1L << 30), "lgs_linear: too many tiles");
  gemm_kernel<WM, WN, FM, FN, RA, RB><<<lga::gemm_grid(tiles), T::NT, 0, stream>>>(p, (int)nt, batch);
  return 0;
}

// act(gate) * up with the gate's and the up's rows of W in turn as the tile's A, 32 of each: the pair of a column meets in
// one lane, which has four neighbouring columns of a row and stores them rounded to bf16. Two passes over fp32 results of
// twice the width and a launch less than the product and its unit apart, whose bits it gives: 403 us for 2407 rows, twice
// 11008 columns and K 4096 in a model's prompt (511 on stages of 32 values of K).
template <int WM, int WN, int FM, int FN, int RA, int RB, bool CLAMPED>
__device__ __forceinline__ void glu_rows(const LinArgs& p, const GluForm& f, unsigned char* lds, int z, int r_lo, int Mz, int m0, int n0) {
  using T = GemmTile<WM, WN, FM, FN, RA, RB>;
  static_assert(FM % 2 == 0, "fragments of the two matrices in pairs");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned char *src_w[T::PA], *src_x[T::PB];
  int r, c;
#pragma unroll
  for (int i = 0; i < T::PA; ++i) {  // columns past the end repeat the last one (never stored)
    lga::gemm_dma_at(wave * T::PA + i, lane, &r, &c);
    const int col = min(n0 + r / 64 * 32 + r % 32, p.N - 1);
    src_w[i] = (const unsigned char*)((const uint16_t*)p.w + (size_t)z * p.sw + (r / 32 % 2 ? f.up : 0) + (size_t)col * p.K) + c * 16;
  }
#pragma unroll
  for (int i = 0; i < T::PB; ++i) {
    lga::gemm_dma_at(wave * T::PB + i, lane, &r, &c);
    const int lr = r_lo + min(m0 + r, Mz - 1);
    src_x[i] = (const unsigned char*)(p.a16 + (size_t)(p.a_rows ? p.a_rows[lr] : lr) * p.lda) + c * 16;
  }
  f32x16_t acc[FM][FN];
  gemm_tile<WM, WN, FM, FN, RA, RB>(lds, src_w, src_x, p.K / 64, wave, lane, acc);
  const int wm = wave % WM, wn = wave / WM, l31 = lane & 31, hi = lane >> 5;
  auto store = [&](auto&& unit) {
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
            const float a = unit(acc[i][j][q * 4 + e], acc[i + 1][j][q * 4 + e]);
            const float b = unit(acc[i][j][q * 4 + e + 1], acc[i + 1][j][q * 4 + e + 1]);
            o[e / 2] = (uint32_t)f2bf(a) | (uint32_t)f2bf(b) << 16;
          }
          *(uint2*)(p.y16 + (size_t)(r_lo + row) * p.ldy + col) = make_uint2(o[0], o[1]);
        }
    }
  };
  // the unit that gated models have gets code of its own: a choice per result costs 18 us a round of 256 x 256 tiles
  if (CLAMPED || f.act != kActSilu) store([&](float g, float u) { return glu_f<CLAMPED>(f, g, u); });
  else store([](float g, float u) { return act_f(kActSilu, g) * u; });
}

template <int WM, int WN, int FM, int FN, int MOST, bool CLAMPED, int F = FN - 1>
__device__ __forceinline__ void glu_short(const LinArgs& p, const GluForm& f, unsigned char* lds, int z, int r_lo, int Mz, int m0, int n0,
                                          int frags) {
  if constexpr (F > 0) {
    using S = lga::GemmShort<WM, WN, FM, F, MOST>;
    if (frags == F) glu_rows<WM, WN, FM, F, S::RA, S::RB, CLAMPED>(p, f, lds, z, r_lo, Mz, m0, n0);
    else glu_short<WM, WN, FM, FN, MOST, CLAMPED, F - 1>(p, f, lds, z, r_lo, Mz, m0, n0, frags);
  }
}

template <int WM, int WN, int FM, int FN, int RA, int RB, bool CLAMPED>
__global__ void __launch_bounds__(WM* WN * 64) gemm_glu_kernel(LinArgs p, GluForm f, int nt, int batch) {
  using T = GemmTile<WM, WN, FM, FN, RA, RB>;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[FN > 1 ? lga::kGemmLds<T> : T::LDS];
  lga::GemmAt at;
  int z = 0, r_lo = 0, Mz = p.M;
  if (p.z_start) {
    if (!gemm_group<T::BN>(p.z_start, batch, nt, threadIdx.x & 63, &at)) return;
    z = at.which;
    r_lo = p.z_start[z];
    Mz = p.z_start[z + 1] - r_lo;
  } else if (!lga::gemm_at<T::BN, WN * 32>(Mz, nt, 1, &at)) {
    return;
  }
  const int m0 = at.m * T::BN, n0 = at.n * (T::BM / 2), frags = (Mz - m0 + WN * 32 - 1) / (WN * 32);
  if (frags >= FN) glu_rows<WM, WN, FM, FN, RA, RB, CLAMPED>(p, f, lds, z, r_lo, Mz, m0, n0);
  else glu_short<WM, WN, FM, FN, lga::kGemmLds<T>, CLAMPED>(p, f, lds, z, r_lo, Mz, m0, n0, frags);
}

template <int WM, int WN, int FM, int FN, int RA, int RB>
static int glu_go(const LinArgs& p, const GluForm& f, int batch, hipStream_t stream) {
  using T = GemmTile<WM, WN, FM, FN, RA, RB>;
  const long mt = (p.M + T::BN - 1) / T::BN, nt = (p.N + T::BM / 2 - 1) / (T::BM / 2);
  const long tiles = p.z_start ? (mt + batch) * nt : mt * nt;
  LGA_CHECK_ARG(tiles < (1L << 30), "lgs_linear_glu: too many tiles");
  const unsigned grid = lga::gemm_grid(tiles);
  if (f.clamped) gemm_glu_kernel<WM, WN, FM, FN, RA, RB, true><<<grid, T::NT, 0, stream>>>(p, f, (int)nt, batch);
  else gemm_glu_kernel<WM, WN, FM, FN, RA, RB, false><<<grid, T::NT, 0, stream>>>(p, f, (int)nt, batch);
  return 0;
}

GemmPlan gemm_glu_plan(int M, int n, int K, int batch, bool grouped) {
  return lga::gemm_tile_plan(M, 2 * n, K, batch, grouped, 1, lga::kGemmRowsB | lga::kGemmPairs);
}

int gemm_glu_launch(const LinArgs& p, const GluForm& f, int batch, hipStream_t stream) {
#define LGS_CASE(I, SLOTS, US, FAST, ROUND, ...)                                     \
  case I:                                                                            \
    if constexpr (lga::kGemmForms[I].fm % 2 == 0) return glu_go<__VA_ARGS__>(p, f, batch, stream); \
    break;
  const GemmPlan plan = gemm_glu_plan(p.M, p.N, p.K, batch, p.z_start != nullptr);
  switch (plan.tile) { LGA_GEMM_FORMS(LGS_CASE) }
#undef LGS_CASE
  lga_set_error("lgs_linear_glu: no such form");
  return (int)hipErrorInvalidValue;
}

GemmPlan gemm_plan(int M, int N, int K, int batch, bool grouped, int ksplit, int act, bool sums) {
  if (grouped && gemm_few_rows(M, batch)) return GemmPlan{-1, 1};
  return lga::gemm_tile_plan(M, N, K, batch, grouped, ksplit, (act != kActNone ? lga::kGemmActs : 0) | (sums ? lga::kGemmSums : 0));
}

int gemm_launch(const LinArgs& p, const GemmPlan& plan, int batch, hipStream_t stream) {
#define LGS_CASE(I, SLOTS, US, FAST, ROUND, ...) \
  case I: return gemm_go<__VA_ARGS__>(p, batch, stream);
  switch (plan.tile) { LGA_GEMM_FORMS(LGS_CASE) }
#undef LGS_CASE
  lga_set_error("lgs_linear: no such form");
  return (int)hipErrorInvalidValue;
}

// 32 rows and up to 32 columns by one wave, eight steps ahead: a router's logits, whole in K. The sums are those of the tiles above, to the
// same bits, but there are more workgroups and none of their waves works on columns that are not there. Bound by the latency of a step.
// us, the tiles of 64 x 128 / here: 2048 x 18 x 2048 13.8 / 10.4 (in a model's prompt 16.4 / 12.0), 4096 x 16 x 2048 14.0 / 10.8, 2407 x 16
// x 4096 23.0 / 17.2, 300 x 32 x 1024 8.7 / 6.7; past 8192 rows both have work for the chip (16000 x 18 x 2048 16.3 / 17.7), the rows of
// all batches together (4 of 8192 x 32 x 64 4.8 / 6.1, 64 of 512 x 16 x 512 9.1 / 12.7), or 16384 where there are few batches or K is short
// (8 of 2048 x 16 x 2048 15.3 / 13.9, 16 of 1024 15.4 / 14.4, 64 of 256 x 16 x 512 6.9 / 5.2; x 32 x 1024 9.9 / 13.0). With the operands
// in registers as the instructions take them 9.9 and 16.0, but only for K a multiple of 512.
__global__ void __launch_bounds__(64) gemm_narrow_kernel(LinArgs p) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds[GemmTile<1, 1, 1, 1, 8, 8>::LDS];
  gemm_rows<1, 1, 1, 1, 8, 8, true, true>(p, lds, blockIdx.y, 0, 0, p.M, blockIdx.x * 32, 0);
}

bool gemm_narrow(const LinArgs& p, int batch, hipStream_t stream) {
  const long rows = (long)p.M * batch;
  const bool idle = p.M <= 8192 && (rows <= 8192 || (rows <= 16384 && (batch <= 16 || p.K <= 512)));
  if (p.N > 32 || !idle || p.K % 64 != 0 || p.ksplit > 1 || p.z_start) return false;
  gemm_narrow_kernel<<<dim3((p.M + 31) / 32, batch), 64, 0, stream>>>(p);
  return true;
}

}  // namespace lgs
