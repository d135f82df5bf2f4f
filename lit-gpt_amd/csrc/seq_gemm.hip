// The large products of the layered models' prompts: Y (+)= act(A W^T + bias) with A and W in bf16, sums in fp32.
//
// A tile of BM x BN outputs belongs to one workgroup of WM x WN waves; a wave holds FM x FN accumulators of
// v_mfma_f32_32x32x16_bf16. A and W reach LDS by LDS-DMA (global_load_lds, 16 bytes a lane, source-swizzled so that
// fragments are read without bank conflicts) in ST stages of BK values of K. Per 16 values of K a wave reads FM + FN
// fragments for FM * FN matrix instructions; the fragments of the next 16 are read while these run, across the stages
// too: the one barrier of a stage stands before its last 16 values' matrix instructions, whose operands are in
// registers by then, and the buffer that it frees is refilled between the matrix instructions that follow.
#include "seq_gemm.h"

#include <cmath>

namespace lgs {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

__device__ __forceinline__ void gemm_dma16(const void* src, unsigned char* lds) {
  __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}
template <int N>  // until at most N of this wave's DMAs are in flight (the count is a field of the instruction)
__device__ __forceinline__ void gemm_wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <int WM, int WN, int FM, int FN, int BK, int ST>
struct GemmTile {
  static_assert(BK == 32 || BK == 64, "a row of a stage is half or all of a 128-byte LDS row");
  static constexpr int BM = WM * FM * 32, BN = WN * FN * 32, NW = WM * WN, NT = NW * 64;
  static constexpr int RPL = 64 / BK;                     // matrix rows per LDS row
  static constexpr int STAGE = (BM + BN) / RPL * 128;     // bytes
  static constexpr int ROWS = 8 * RPL;                    // matrix rows per DMA of a wave (1 KB)
  static constexpr int P = (BM + BN) / ROWS / NW;         // DMAs per wave and stage
  static constexpr int H = (P + 1) / 2;                   // ... of these ahead of the next barrier but one
  static_assert((BM + BN) % (ROWS * NW) == 0 && BM % ROWS == 0 && ST >= 2, "every wave issues the same number of DMAs");
  static_assert((ST - 1) * P <= 63, "DMAs in flight are counted in six bits");
  static_assert(ST * STAGE <= 163840, "LDS");
};

// Bound by the matrix cores' feeding: without its DMAs the 256 x 256 form runs 1.3 times as fast, without its fragment
// reads 1.1 times, without both at the matrix cores' rate (2.1 PFLOP/s). Results go straight to memory, past the caches
// (a lane's rows in 128-byte pieces): turning them in LDS into longer pieces cost 14 us a tile.
//
// Workgroup b runs on XCD b % 8, and an XCD takes neighbouring tiles, whose rows of A and W its L2 then holds.
template <int WM, int WN, int FM, int FN, int BK, int ST>
__global__ void __launch_bounds__(WM* WN * 64) gemm_kernel(LinArgs p, int mt, int nt, int batch) {
  using T = GemmTile<WM, WN, FM, FN, BK, ST>;
  constexpr int P = T::P, H = T::H;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[ST * T::STAGE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int t = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  int z = 0, split = 0, r_lo = 0, Mz = p.M, m, n;
  if (p.z_start) {  // grouped: the batch whose tiles hold number t, the batches' tiles counted side by side over the lanes
    bool found = false;
    for (int e0 = 0; e0 < batch && !found; e0 += 64) {
      const int e = e0 + lane;
      const int rows = e < batch ? p.z_start[e + 1] - p.z_start[e] : 0;
      const int own = (rows + T::BM - 1) / T::BM * nt;
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
    if (!found) return;
    z = __builtin_amdgcn_readfirstlane(z);
    t = __builtin_amdgcn_readfirstlane(t);
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
    const int R = (of_a ? piece : piece - T::BM / T::ROWS) * 8 + (lane >> 3);
    const int lc = (lane & 7) ^ (R & 7);
    const int r = BK == 64 ? R : 2 * R + (lc >> 2), c = BK == 64 ? lc : lc & 3;
    if (of_a) {
      const int lr = r_lo + min(m0 + r, Mz - 1);  // rows past the end repeat the last one (never stored)
      src[i] = (const unsigned char*)(p.a16 + (size_t)z * p.sa + (size_t)(p.a_rows ? p.a_rows[lr] : lr) * p.lda);
    } else {
      src[i] = (const unsigned char*)((const uint16_t*)p.w + (size_t)z * p.sw + (size_t)min(n0 + r, p.N - 1) * p.K);
    }
    src[i] += (size_t)k0 * (BK * 2) + c * 16;
  }
  // Past the last stage the last one is fetched again into a buffer that nobody reads: the count of DMAs in flight is
  // the same at every barrier, and no branch stands around them.
  auto stage = [&](int k, int buf, int from, int to) {
    const size_t at = (size_t)min(k, nk - 1) * (BK * 2);
#pragma unroll
    for (int i = 0; i < P; ++i)
      if (i >= from && i < to) gemm_dma16(src[i] + at, lds + buf * T::STAGE + (wave * P + i) * 1024);
  };
  const int wm = wave % WM, wn = wave / WM;
  const int l31 = lane & 31, hi = lane >> 5;
  // row l31 of a fragment, chunk hi: its LDS row and swizzled chunk; chunk 2 s + hi lies at that address ^ 32 s
  const int lrow = l31 / T::RPL;
  const int sw = lrow * 128 + 16 * (((l31 % T::RPL) * 4 + hi) ^ (lrow & 7));
  const int abase = wm * FM * 32 / T::RPL * 128 + sw, bbase = (T::BM + wn * FN * 32) / T::RPL * 128 + sw;
  struct Frags {
    bf16x8_t a[FM], b[FN];
  };
  auto read = [&](int buf, int s, Frags& f) {
    const unsigned char* A = lds + buf * T::STAGE + (abase ^ (32 * s));
    const unsigned char* B = lds + buf * T::STAGE + (bbase ^ (32 * s));
#pragma unroll
    for (int j = 0; j < FN; ++j) f.b[j] = *(const bf16x8_t*)(B + j * (4096 / T::RPL));
#pragma unroll
    for (int i = 0; i < FM; ++i) f.a[i] = *(const bf16x8_t*)(A + i * (4096 / T::RPL));
  };
  f32x16_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  auto mma = [&](const Frags& f) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[i], f.b[j], acc[i][j], 0, 0, 0);
  };
  // after every matrix instruction two reads of the next fragments, after every second a DMA
#define LGS_WEAVE(DMAS)                                                \
  do {                                                                 \
    int rd_ = 0, dma_ = 0;                                             \
    _Pragma("unroll") for (int e_ = 0; e_ < FM * FN; ++e_) {           \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);               \
      _Pragma("unroll") for (int q_ = 0; q_ < 2; ++q_)                 \
        if (rd_ < FM + FN) {                                           \
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);           \
          ++rd_;                                                       \
        }                                                              \
      if (e_ % 2 == 1 && dma_ < (DMAS)) {                              \
        __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);             \
        ++dma_;                                                        \
      }                                                                \
    }                                                                  \
  } while (0)
#pragma unroll
  for (int s = 0; s < ST; ++s) stage(s, s, 0, P);
  gemm_wait_vm<(ST - 1) * P>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  Frags f0, f1;
  read(0, 0, f0);
  int buf = 0, last = ST - 1;  // the buffers of stages k and k - 1
  for (int k = 0; k < nk; ++k) {
    __builtin_amdgcn_sched_barrier(0);
    read(buf, 1, f1);
    stage(k - 1 + ST, last, H, P);  // (first pass: the second half of the last stage of the lead once more)
    mma(f0);
    LGS_WEAVE(P - H);
    if constexpr (BK == 64) {
      __builtin_amdgcn_sched_barrier(0);
      read(buf, 2, f0);
      mma(f1);
      LGS_WEAVE(0);
      __builtin_amdgcn_sched_barrier(0);
      read(buf, 3, f1);
      mma(f0);
      LGS_WEAVE(0);
    }
    __builtin_amdgcn_sched_barrier(0);
    const int next = buf + 1 == ST ? 0 : buf + 1;
    gemm_wait_vm<(ST - 2) * P>();                       // this wave's part of stage k + 1 has landed,
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // and it has read all that it reads of stage k
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    read(next, 0, f0);  // (past the last stage: the repeated one, never used)
    stage(k + ST, buf, 0, H);
    mma(f1);
    LGS_WEAVE(H);
    last = buf;
    buf = next;
  }
#undef LGS_WEAVE
  gemm_wait_vm<0>();  // no DMA may outlive the workgroup's LDS
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

// The tile forms, and what a stage of 64 values of K costs a full chip of their workgroups, measured on products of
// 2048 x 2048 x 2048 to 2407 x 22016 x 4096: a tile of 256 x 256 runs 1.80 us per 64 values (1190 TFLOP/s, 0.79 of
// what a large matrix product reaches on this card), of 256 x 128 1.02, of 128 x 128 0.63 alone on a compute unit and
// 1.14 for two, of 64 x 128 0.43. The larger tile moves fewer bytes per product, the smaller ones fill the chip when
// rows or columns are few. A workgroup's start and end cost about 3 us.
struct GemmForm {
  int bm, bn, slots;  // slots: workgroups of the whole chip at a time
  float step_us;
};
static const GemmForm kForms[] = {{256, 256, 256, 1.80f}, {256, 128, 256, 1.02f}, {128, 128, 512, 1.14f},
                                  {128, 128, 256, 0.63f}, {64, 128, 256, 0.43f}};

// Rounds of workgroups times what one takes; several ranges of K cost a second launch that reads them all. E.g.
// 2048 x 2048 x 5632: 256 tiles of 128 x 128 in one round, 55 us (64 of 256 x 256: 131); 128 x 4096 x 4096: 64 tiles of
// 64 x 128 in four ranges of K, 16 us (whole: 41); before these tiles 126 and 86 us.
GemmPlan gemm_plan(int M, int N, int K, int batch, bool grouped, int ksplit) {
  GemmPlan best{-1, 1};
  if (K % 64 != 0 || M <= 0) return best;
  const int steps = K / 64;
  float best_us = 0.0f;
  for (int f = 0; f < (int)(sizeof(kForms) / sizeof(kForms[0])); ++f) {
    const GemmForm& t = kForms[f];
    const float nt = (float)((N + t.bn - 1) / t.bn);
    // a range of the list ends somewhere in its last tile
    const float mt = grouped ? (float)M / t.bm + 0.5f * batch : (float)((M + t.bm - 1) / t.bm) * batch;
    const int s_lo = ksplit > 0 ? ksplit : 1, s_hi = ksplit > 0 ? ksplit : (batch > 1 || grouped ? 1 : 16);
    for (int s = s_lo; s <= s_hi && (s == s_lo || steps / s >= 4); ++s) {
      const int per = (steps + s - 1) / s;
      const float rounds = ceilf(mt * nt * (float)((steps + per - 1) / per) / (float)t.slots);
      float us = rounds * (per * t.step_us + 3.0f);
      if (s > 1) us += 5.0f + (float)M * N * 4.0f * (2 * s + 1) / 3.0e6f;
      if (best.tile < 0 || us < best_us) {
        best_us = us;
        best = GemmPlan{f, s};
      }
    }
  }
  return best;
}

int gemm_launch(const LinArgs& p, const GemmPlan& plan, int batch, hipStream_t stream) {
  switch (plan.tile) {
    case 0: return gemm_go<2, 4, 4, 2, 32, 5>(p, batch, stream);
    case 1: return gemm_go<4, 2, 2, 2, 64, 3>(p, batch, stream);
    case 2: return gemm_go<2, 2, 2, 2, 64, 2>(p, batch, stream);
    case 3: return gemm_go<2, 4, 2, 1, 64, 4>(p, batch, stream);
    default: return gemm_go<1, 4, 2, 1, 64, 4>(p, batch, stream);
  }
}

}  // namespace lgs
