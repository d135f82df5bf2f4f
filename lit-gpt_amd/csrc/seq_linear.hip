// Linear layers, embedding and RMS norms of the layered models: fp32 activations, bf16 or fp32 weights.
//
//   lgs_linear     Y[z] (+)= act(A[z] W[z]^T + bias): one entry point for every projection. Up to 8 rows run a streaming
//                  GEMV (a wave per pair of output columns, 16-B weight loads, fp32 sums); more rows run the
//                  pipelined tiles of seq_gemm.hip (A a producer's bf16 copy, K a multiple of 64, aligned rows), 128x128
//                  tiles of v_mfma_f32_16x16x32_bf16 (other bf16 products; an fp32 A is rounded to bf16 while it is
//                  staged into LDS) or 64x64 fp32 FMA tiles (fp32 weights). `batch` with strides runs per-head products (the
//                  latent attention's absorbed key and value maps); `z_start` / `a_rows` make it a grouped product
//                  over row ranges of a sorted list (sparse experts during a prompt).
//   lgs_embed      x[t] = table[token[t]] * scale
//   lgs_rmsnorm    y = x / sqrt(mean(x^2) + eps) * (offset + w), rows with strides (whole rows, or heads)
#include <algorithm>

#include "seq_gemm.h"
#include "seq_rows.h"

namespace lgs {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------------------------------------ GEMV, M <= 8
// R output columns per wave: 4 for tall matrices (more loads in flight per lane), fewer for short ones (more waves)
// KS 4: short and deep matrices; the four waves of a workgroup share its R columns, each a quarter of K
// AHEAD: the weights of four passes over K on their way together, for few columns a wave, whose time is trips to memory. us without /
// with, weights from memory: 1024 x 8192 11.4 / 9.7, 2048 x 4096 8.0 / 7.7, two rows 12.3 / 8.9, 11264 x 2048 13.0 / 12.0; where more
// waves stand side by side the registers cost more of them than the trips take: 3584 x 4096 9.2 / 9.8 (3072: 8.8 / 8.9), 4088 x 8192
// 17.5 / 18.9, 22016 x 4096 38.8 / 41.6; and passes past a short row's end cost theirs: 2048 x 1024 3.5 / 3.6, 8192 x 1024 5.8 / 6.5,
// 16376 x 1536 12.3 / 12.9. The row's own values come pass by pass, behind the weights.
template <bool WF32, int MT, int R, int KS, bool AHEAD>
__global__ void __launch_bounds__(256) lin_gemv_kernel(LinArgs p) {
  __shared__ float shared_acc[KS > 1 ? 4 * MT * R : 1];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int z = blockIdx.y;
  const int n0 = (KS > 1 ? blockIdx.x : blockIdx.x * 4 + wave) * R;
  if (n0 >= p.N) return;
  const int kl = KS > 1 ? wave * 64 + lane : lane;  // this lane's place in a pass over K
  const float* a = p.a + (size_t)z * p.sa;
  const size_t wbase = (size_t)z * p.sw;
  float acc[MT][R];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int r = 0; r < R; ++r) acc[m][r] = 0.0f;
  const int K = p.K;
  const bool vec = (K % 8 == 0) && (p.lda % 4 == 0) && (((uintptr_t)a) % 16 == 0) && (p.sw % 8 == 0) &&
                   (((uintptr_t)p.w) % 16 == 0);
  int rows[R];
  float bias[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    rows[r] = min(n0 + r, p.N - 1);
    bias[r] = p.bias ? p.bias[rows[r]] : 0.0f;
  }
  auto add = [&](int k, const float (&wv)[R][8]) {  // eight values of K of every row and column
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      if (m < p.M) {
        const float* ar = a + (size_t)m * p.lda + k;
        const float4 lo = *(const float4*)ar, hi = *(const float4*)(ar + 4);
        const float av[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float x = aop<WF32>(av[e]);
#pragma unroll
          for (int r = 0; r < R; ++r) acc[m][r] = fmaf(x, wv[r][e], acc[m][r]);
        }
      }
    }
  };
  auto spread = [](const uint4& q, float (&v)[8]) {
    v[0] = bflo(q.x); v[1] = bfhi(q.x); v[2] = bflo(q.y); v[3] = bfhi(q.y);
    v[4] = bflo(q.z); v[5] = bfhi(q.z); v[6] = bflo(q.w); v[7] = bfhi(q.w);
  };
  if (vec && AHEAD) {
    static_assert(!AHEAD || (!WF32 && KS == 1), "bf16 weights, a wave per column");
    constexpr int U = 4;
    for (int k0 = kl * 8; k0 < K; k0 += 512 * U) {
      uint4 q[U][R];
      // (a lane past the end loads its row's last values and does not use them: behind a branch a load waits for those before it)
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int r = 0; r < R; ++r)
          q[u][r] = *(const uint4*)((const uint16_t*)p.w + wbase + (size_t)rows[r] * K + min(k0 + u * 512, K - 8));
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (k0 + u * 512 >= K) break;
        float wv[R][8];
#pragma unroll
        for (int r = 0; r < R; ++r) spread(q[u][r], wv[r]);
        add(k0 + u * 512, wv);
      }
    }
  } else if (vec) {
#pragma unroll 2
    for (int k = kl * 8; k < K; k += 512 * KS) {
      float wv[R][8];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const size_t off = wbase + (size_t)rows[r] * K + k;
        if (WF32) {
          const float4 lo = *(const float4*)((const float*)p.w + off), hi = *(const float4*)((const float*)p.w + off + 4);
          wv[r][0] = lo.x; wv[r][1] = lo.y; wv[r][2] = lo.z; wv[r][3] = lo.w;
          wv[r][4] = hi.x; wv[r][5] = hi.y; wv[r][6] = hi.z; wv[r][7] = hi.w;
        } else {
          spread(*(const uint4*)((const uint16_t*)p.w + off), wv[r]);
        }
      }
      add(k, wv);
    }
  } else {
    for (int k = kl; k < K; k += 64 * KS) {
      float wv[R];
#pragma unroll
      for (int r = 0; r < R; ++r) wv[r] = wload<WF32>(p.w, wbase + (size_t)rows[r] * K + k);
#pragma unroll
      for (int m = 0; m < MT; ++m)
        if (m < p.M) {
          const float x = aop<WF32>(a[(size_t)m * p.lda + k]);
#pragma unroll
          for (int r = 0; r < R; ++r) acc[m][r] = fmaf(x, wv[r], acc[m][r]);
        }
    }
  }
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float s = wave_sum(acc[m][r]);
      if (KS > 1) {
        if (lane == 0) shared_acc[(wave * MT + m) * R + r] = s;
        continue;
      }
      if (lane == 0 && m < p.M && n0 + r < p.N) {
        float* yp = p.y + (size_t)z * p.sy + (size_t)m * p.ldy + n0 + r;
        const float v = act_f(p.act, s + bias[r]);
        *yp = p.accumulate ? *yp + v : v;
      }
    }
  if (KS > 1) {
    __syncthreads();
    const int m = threadIdx.x / R, r = threadIdx.x % R;
    if (m < MT && m < p.M && n0 + r < p.N) {
      const float* q = shared_acc + m * R + r;
      const float s = (q[0] + q[MT * R]) + (q[2 * MT * R] + q[3 * MT * R]);
      float* yp = p.y + (size_t)z * p.sy + (size_t)m * p.ldy + n0 + r;
      const float v = act_f(p.act, s + (p.bias ? p.bias[n0 + r] : 0.0f));
      *yp = p.accumulate ? *yp + v : v;
    }
  }
}

static bool gemv_deep(long columns, int K) { return columns <= 512 && K >= 1024; }  // few columns: four waves per column

// One row's gated unit in its input product's launch: a wave makes a gate column and the up column beside it, in lin_gemv_kernel's
// order (but that of few columns: gemv_deep), and the unit of the two. us, product and unit / here: 2 x 520 columns of 2048 values
// 5.9 / 4.1, 2 x 5632 14.2 / 11.8, of 4096 values 24.8 / 20.0, 2 x 11008 41.1 / 36.2, of 8192 75.0 / 70.5.
template <bool AHEAD, bool CLAMPED>
__global__ void __launch_bounds__(256) lin_glu_row_kernel(const float* __restrict__ a, const uint16_t* __restrict__ w, GluForm f,
                                                          float* __restrict__ y, int n, int K) {
  const int col = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (col >= n) return;
  const uint16_t* rows[2] = {w + (size_t)col * K, w + f.up + (size_t)col * K};
  float acc[2] = {0.0f, 0.0f};
  constexpr int U = AHEAD ? 4 : 2;
  for (int k0 = lane * 8; k0 < K; k0 += 512 * U) {
    uint4 q[U][2];  // (past the end: the row's last values, not used)
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int r = 0; r < 2; ++r) q[u][r] = *(const uint4*)(rows[r] + min(k0 + u * 512, K - 8));
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * 512;
      if (k >= K) break;
      const float4 lo = *(const float4*)(a + k), hi = *(const float4*)(a + k + 4);
      const float av[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const uint4 v = q[u][r];
        const float wv[8] = {bflo(v.x), bfhi(v.x), bflo(v.y), bfhi(v.y), bflo(v.z), bfhi(v.z), bflo(v.w), bfhi(v.w)};
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[r] = fmaf(aop<false>(av[e]), wv[e], acc[r]);
      }
    }
  }
  const float g = wave_sum(acc[0]), u = wave_sum(acc[1]);
  if (lane == 0) y[col] = glu_f<CLAMPED>(f, g, u);
}

// seq_rows.h's products, finished here
// (32 columns: registers for three workgroups a compute unit, as many as their LDS allows. Two, 8 x 21660 x 128: 5.9 -> 8.0 us)
template <int NR, int KW, int MR, int RB, bool ONE>
__global__ void __launch_bounds__(KW * 64, NR == 2 && RB == 1 ? 3 : 1) lin_rows_kernel(LinArgs p) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds[RowsTile<NR, KW, MR, RB>::LDS];
  const int tid = threadIdx.x, lane = tid & 63, l15 = lane & 15, q4 = lane >> 4;
  const int z = blockIdx.y, n0 = blockIdx.x * (16 * NR);
  const uint16_t* w = (const uint16_t*)p.w + (size_t)z * p.sw;
  rows_products<NR, KW, MR, RB, ONE>(lds, [&](int r) { return w + (size_t)min(n0 + r, p.N - 1) * p.K; }, p.a + (size_t)z * p.sa,
                                     p.lda, p.M, p.K);
  if (tid >= NR * 64 || l15 >= p.M) return;
  const int j = NR > 1 ? __builtin_amdgcn_readfirstlane(tid >> 6) : 0;
  const rows_f32x4 v = rows_sum<NR, KW>(lds, j, lane);
  float* y = p.y + (size_t)z * p.sy + (size_t)l15 * p.ldy;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int n = n0 + j * 16 + q4 * 4 + r;
    if (n >= p.N) continue;
    const float o = act_f(p.act, v[r] + (p.bias ? p.bias[n] : 0.0f));
    y[n] = p.accumulate ? y[n] + o : o;
  }
}
// 16 columns a workgroup; 32, which read A half as often, for more than four rows where their workgroups end together: many, or one a
// compute unit (us of 16 / 32 columns: 8 x 32000 x 2048 31.3 / 30.2, x 22016 x 4096 40.6 / 37.6, x 6288 x 2048 9.8 / 9.0, x 4608 x 4096
// 13.0 / 11.5, x 8192 x 2048 9.5 / 10.2, x 4096 x 4096 9.3 / 13.4, x 5120 x 1024 5.4 / 5.8; 3 x 32000 x 4096 48.2 / 50.8). Below 4096 columns
// eight waves share K.
template <int NR, int KW, int MR, bool ONE>
static void lin_rows_go(const LinArgs& p, int batch, hipStream_t stream) {
  const dim3 grid((p.N + 16 * NR - 1) / (16 * NR), batch);
  if constexpr (KW == 4) {
    if ((long)grid.x * batch <= 256) return lin_rows_kernel<NR, KW, MR, 2, ONE><<<grid, KW * 64, 0, stream>>>(p);
  }
  lin_rows_kernel<NR, KW, MR, 1, ONE><<<grid, KW * 64, 0, stream>>>(p);
}
template <int NR, int KW>
static void lin_rows_go(const LinArgs& p, int batch, hipStream_t stream) {
  if (rows_one(p.K)) (p.M > 4 ? lin_rows_go<NR, KW, 8, true> : lin_rows_go<NR, KW, 4, true>)(p, batch, stream);
  else (p.M > 4 ? lin_rows_go<NR, KW, 8, false> : lin_rows_go<NR, KW, 4, false>)(p, batch, stream);
}

// What they gain on a lane's sums (lin_gemv_kernel; us there / here): 5 to 8 rows always (8 x 64 x 512 5.5 / 3.1, 5 x 1024 x 4096 15.3 / 7.2),
// four but of few columns and long rows (4 x 1024 x 2048 7.4 / 4.4, x 20608 x 2048 34.3 / 18.8; x 256 x 2048 4.1 / 4.0, x 256 x 4096 5.4 /
// 4.9), two and three of long rows (2 x 2048 x 4096 9.0 / 7.9, 3 x 1024 x 4096 11.4 / 6.6; 3 x 512 x 8192 8.9 / 9.3), one of longer rows and few
// columns (1 x 2048 x 5632 10.0 / 9.2, x 3072 x 8192 15.7 / 12.3; x 512 x 5632 5.0 / 7.4, x 2048 x 2048 5.2 / 5.4). Two and three shorter
// rows (2 x 8192 x 2048 12.6 / 9.1) keep the bits that each has alone, and two of large matrices whose rows lie a multiple of 16 KB apart,
// in the same channels of memory, go faster side by side (2 x 16384 x 8192 55.4 / 57.8, x 14336 x 16384 91 / 104; x 11008 x 8192 39.8 /
// 37.3, x 14336 x 11008 76 / 65). Of short rows: 5 x 2048 x 128 3.5 / 3.3, 4 x 512 x 128 4.0 / 3.2, of 16 heads 8 x 512 x 128 9.3 / 4.0.
// columns: of all batches
static bool lin_rows_pay(int M, long columns, int K) {
  if (K % 128 != 0 || M > 8) return false;
  if (M == 1) return K > 4096 && columns > 512 && columns < 4096;
  if (M == 2 && K % 8192 == 0 && columns > 12288) return false;
  if (M <= 3) return K >= 4096 && columns > 512;
  return M > 4 || columns > 512 || K < 1024;
}

// ------------------------------------------------------------------------------------------------ MFMA tiles
constexpr int BM = 128, BN = 128, BK = 64;
constexpr int TILE_BYTES = BM * BK * 2;
__device__ __forceinline__ int swz(int row, int chunk) { return row * 128 + 16 * (chunk ^ (row & 7)); }

// VEC: K % 8 == 0 and 16-B aligned rows of A and W (vector loads); otherwise element loads with k guards.
// A16: A arrives as bf16 (half the operand traffic of the fp32 stream; the same values the fp32 path would round to)
// NARROW: up to 32 columns, those of a router
template <bool VEC, bool A16, bool NARROW>
__global__ void __launch_bounds__(256) lin_mfma_kernel(LinArgs p) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[2 * 2 * TILE_BYTES];  // [buf][A|W]
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int wm = wave >> 1, wn = wave & 1;
  const int z = p.ksplit > 1 ? 0 : blockIdx.z;
  const int r_lo = p.z_start ? p.z_start[z] : 0;
  const int Mz = p.z_start ? p.z_start[z + 1] - r_lo : p.M;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  if (m0 >= Mz) return;
  const float* abase = A16 ? nullptr : p.a + (size_t)z * p.sa;
  const uint16_t* abase16 = A16 ? p.a16 + (size_t)z * p.sa : nullptr;
  const uint16_t* wbase = (const uint16_t*)p.w + (size_t)z * p.sw;
  const int K = p.K;
  int kt_lo = 0, nk = (K + BK - 1) / BK;
  if (p.ksplit > 1) {
    kt_lo = blockIdx.z * p.kper;
    nk = min(nk, kt_lo + p.kper);
  }
  const int t_row = tid >> 1, t_half = tid & 1;
  const int lr = r_lo + min(m0 + t_row, Mz - 1);  // rows past the end repeat the last one (never stored)
  const size_t arow_off = (size_t)(p.a_rows ? p.a_rows[lr] : lr) * p.lda;
  const float* arow = abase + arow_off;
  const uint16_t* arow16 = abase16 + arow_off;
  const uint16_t* wrow = wbase + (size_t)min(n0 + t_row, p.N - 1) * K;

  uint4 areg[4], wreg[4];
  auto gload = [&](int kt) {
    const int k0 = kt * BK + t_half * 32;
    if (VEC) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int k = k0 + c * 8;
        if (k < K) {
          if (A16) {
            areg[c] = *(const uint4*)(arow16 + k);
          } else {
            const float4 lo = *(const float4*)(arow + k), hi = *(const float4*)(arow + k + 4);
            areg[c] = make_uint4(pack2(lo.x, lo.y), pack2(lo.z, lo.w), pack2(hi.x, hi.y), pack2(hi.z, hi.w));
          }
          wreg[c] = *(const uint4*)(wrow + k);
        } else {
          areg[c] = make_uint4(0, 0, 0, 0);
          wreg[c] = make_uint4(0, 0, 0, 0);
        }
      }
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        uint32_t av[4], wv[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int k = k0 + c * 8 + 2 * e;
          const uint32_t w0 = k < K ? wrow[k] : 0, w1 = k + 1 < K ? wrow[k + 1] : 0;
          if (A16) {
            const uint32_t b0 = k < K ? arow16[k] : 0, b1 = k + 1 < K ? arow16[k + 1] : 0;
            av[e] = b0 | (b1 << 16);
          } else {
            const float a0 = k < K ? arow[k] : 0.0f, a1 = k + 1 < K ? arow[k + 1] : 0.0f;
            av[e] = pack2(a0, a1);
          }
          wv[e] = w0 | (w1 << 16);
        }
        areg[c] = make_uint4(av[0], av[1], av[2], av[3]);
        wreg[c] = make_uint4(wv[0], wv[1], wv[2], wv[3]);
      }
    }
  };
  auto lstore = [&](int buf) {
    unsigned char* A = lds + buf * (2 * TILE_BYTES);
    unsigned char* B = A + TILE_BYTES;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      *(uint4*)(A + swz(t_row, t_half * 4 + c)) = areg[c];
      *(uint4*)(B + swz(t_row, t_half * 4 + c)) = wreg[c];
    }
  };

  f32x4_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  gload(kt_lo);
  lstore(0);
  __syncthreads();
  const int fr = lane & 15, fk = lane >> 4;
  for (int kt = kt_lo; kt < nk; ++kt) {
    const int cur = (kt - kt_lo) & 1;
    if (kt + 1 < nk) gload(kt + 1);
    const unsigned char* A = lds + cur * (2 * TILE_BYTES);
    const unsigned char* B = A + TILE_BYTES;
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      bf16x8_t af[4], bfr[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        af[i] = *(const bf16x8_t*)(A + swz(wm * 64 + i * 16 + fr, sub * 4 + fk));
        bfr[i] = *(const bf16x8_t*)(B + swz(wn * 64 + i * 16 + fr, sub * 4 + fk));
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0);
    }
    if (kt + 1 < nk) lstore(cur ^ 1);
    __syncthreads();
  }

  if constexpr (NARROW) {  // as the accumulators lie, and only those that hold columns
    if (wn > 0) return;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int n = j * 16 + fr;
      if (n >= p.N) continue;
      const float bias = p.bias ? p.bias[n] : 0.0f;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m0 + wm * 64 + i * 16 + fk * 4 + r;
          if (m >= Mz) continue;
          if (p.ksplit > 1) {
            p.part[((size_t)blockIdx.z * p.M + m) * p.N + n] = acc[i][j][r];
            continue;
          }
          const size_t at = (size_t)z * p.sy + (size_t)(r_lo + m) * p.ldy + n;
          const float v = act_f(p.act, acc[i][j][r] + bias);
          if (p.y16) p.y16[at] = f2bf(v);
          else p.y[at] = p.accumulate ? p.y[at] + v : v;
        }
    }
    return;
  }
  // a wave turns 32 rows of its 64 x 64 results at a time in LDS of its own and stores them four columns a lane, 256 bytes of a row
  // together (as the accumulators lie, 64: 2048 x 2048 x 64, all of it results, 22.0 -> 13.4 us; of a few columns most of that would be work
  // for none, us turned / as they lie: 1725 x 16 x 512 into sums 25.0 / 19.1, 2048 x 16 x 2048 60.5 / 54.6, 300 x 18 x
  // 2048 61.0 / 58.3, 58 x 16 x 64 8.7 / 6.5, 1211 x 20 x 64 9.5 / 11.0; of 19 to 31 columns that do not lie in fours, 118 products into
  // sums 1.03 in the mean and up to 1.12, 1530 x 27 x 384 26.2 / 24.2, others the same)
  constexpr int RS = 68;
  float* turned = (float*)(lds + wave * 16384);
  const int c4 = fr * 4, n = n0 + wn * 64 + c4, cols = p.N - n;
  const bool split = p.ksplit > 1;
  float* out = split ? p.part + ((size_t)blockIdx.z * p.M) * p.N : p.y + ((size_t)z * p.sy + (size_t)r_lo * p.ldy);
  uint16_t* out16 = split || !p.y16 ? nullptr : p.y16 + ((size_t)z * p.sy + (size_t)r_lo * p.ldy);
  const size_t ld = split ? p.N : p.ldy;
  const bool four = cols >= 4 && ld % 4 == 0 && (out16 ? (uintptr_t)out16 % 8 == 0 : (uintptr_t)out % 16 == 0);
  float bias[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) bias[e] = p.bias && !split ? p.bias[min(n + e, p.N - 1)] : 0.0f;
  lga::wait_loads(bias);  // (or every store waits for the one before)
#pragma unroll
  for (int part = 0; part < 2; ++part) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) turned[(i * 16 + fk * 4 + r) * RS + j * 16 + fr] = acc[part * 2 + i][j][r];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int m = m0 + wm * 64 + part * 32 + q * 4 + fk;
      float4 v = *(const float4*)(turned + (q * 4 + fk) * RS + c4);
      if (m >= Mz || cols <= 0) continue;
      const size_t at = (size_t)m * ld + n;
      float* f = (float*)&v;
      if (!split) {
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = act_f(p.act, f[e] + bias[e]);
        if (p.accumulate && !out16) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (e < cols) f[e] = out[at + e] + f[e];
        }
      }
      if (out16) {
        if (four) *(uint2*)(out16 + at) = make_uint2(pack2(f[0], f[1]), pack2(f[2], f[3]));
        else
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (e < cols) out16[at + e] = f2bf(f[e]);
      } else if (four) {
        *(float4*)(out + at) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (e < cols) out[at + e] = f[e];
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// the ranges of K in ascending order, then bias, activation and place as the tiles would. grid (ceil(N / 256), M)
__global__ void __launch_bounds__(256) lin_sum_kernel(LinArgs p) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  const size_t m = blockIdx.y;
  if (n >= p.N) return;
  float s = 0.0f;
#pragma unroll 4
  for (int z = 0; z < p.ksplit; ++z) s += p.part[((size_t)z * p.M + m) * p.N + n];
  const float v = act_f(p.act, s + (p.bias ? p.bias[n] : 0.0f));
  const size_t at = m * p.ldy + n;
  if (p.y16) p.y16[at] = f2bf(v);
  else p.y[at] = p.accumulate ? p.y[at] + v : v;
}

// ------------------------------------------------------------------------------------------------ fp32 tiles
// 64x64 outputs per workgroup, 16 deep; thread (ty, tx) owns rows ty + 16 i and columns tx + 16 j; k ascending
template <bool WF32>
__global__ void __launch_bounds__(256) lin_fma_kernel(LinArgs p) {
  __shared__ float As[16][65];
  __shared__ float Ws[16][65];
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  const int z = blockIdx.z;
  const int r_lo = p.z_start ? p.z_start[z] : 0;
  const int Mz = p.z_start ? p.z_start[z + 1] - r_lo : p.M;
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  if (m0 >= Mz) return;
  const float* abase = p.a + (size_t)z * p.sa;
  const size_t wz = (size_t)z * p.sw;
  const int K = p.K;
  // staging: thread loads column k = tid & 15 of rows (tid >> 4) + 16 i
  const int sk = tid & 15, sr = tid >> 4;
  const float* arows[4];
  size_t wrows[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int lr = r_lo + min(m0 + sr + 16 * i, Mz - 1);
    arows[i] = abase + (size_t)(p.a_rows ? p.a_rows[lr] : lr) * p.lda;
    wrows[i] = wz + (size_t)min(n0 + sr + 16 * i, p.N - 1) * K;
  }
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.0f;
  for (int k0 = 0; k0 < K; k0 += 16) {
    const int k = k0 + sk;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      As[sk][sr + 16 * i] = k < K ? aop<WF32>(arows[i][k]) : 0.0f;
      Ws[sk][sr + 16 * i] = k < K ? wload<WF32>(p.w, wrows[i] + k) : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      float av[4], wv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        av[i] = As[kk][ty + 16 * i];
        wv[i] = Ws[kk][tx + 16 * i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(av[i], wv[j], acc[i][j]);
    }
    __syncthreads();
  }
  float* ybase = p.y + (size_t)z * p.sy;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty + 16 * i;
    if (m >= Mz) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx + 16 * j;
      if (n >= p.N) continue;
      float* yp = ybase + (size_t)(r_lo + m) * p.ldy + n;
      const float v = act_f(p.act, acc[i][j] + (p.bias ? p.bias[n] : 0.0f));
      *yp = p.accumulate ? *yp + v : v;
    }
  }
}

// ------------------------------------------------------------------------------------------------ row kernels
// (grid (T, parts of a row), as embed_grid has it)
template <bool WF32>
__global__ void __launch_bounds__(256) embed_kernel(const int* __restrict__ tok, const void* __restrict__ table,
                                                    float* __restrict__ x, int W, int vocab, float scale) {
  const int t = blockIdx.x;
  int id = tok[t];
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);  // the host validates ids; never read out of bounds
  for (int i = blockIdx.y * 256 + threadIdx.x; i < W; i += gridDim.y * 256)
    x[(size_t)t * W + i] = wload<WF32>(table, (size_t)id * W + i) * scale;
}

// x[t] = table[tok[t]] * scale + ptable[pos[t]] (a learned position vector, not scaled); x16: optional rounded copy
template <bool WF32>
__global__ void __launch_bounds__(256) embed_pos_kernel(const int* __restrict__ tok, const int* __restrict__ pos,
                                                        const void* __restrict__ table, const void* __restrict__ ptable,
                                                        float* __restrict__ x, uint16_t* __restrict__ x16, int W, int vocab,
                                                        int positions, float scale) {
  const int t = blockIdx.x;
  int id = tok[t], ps = pos[t];
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);  // the host validates ids and positions
  ps = ps < 0 ? 0 : (ps >= positions ? positions - 1 : ps);
  for (int i = blockIdx.y * 256 + threadIdx.x; i < W; i += gridDim.y * 256) {
    const float v = fmaf(wload<WF32>(table, (size_t)id * W + i), scale, wload<WF32>(ptable, (size_t)ps * W + i));
    x[(size_t)t * W + i] = v;
    if (x16) x16[(size_t)t * W + i] = f2bf(v);
  }
}

// Layer norm of a sublayer's output joining the residual: x[r] (+)= mult * ((y - mean) / sqrt(var + eps) * w + b),
// var = mean of the squared deviations (two passes over the row, which stays in registers up to 256 * CPT columns).
// x16: optional copy of the new x rounded to bf16 (the next product's operand). grid (rows). Bound by latency for few rows:
// 8 rows of 2048 take 4.7 us (8.0 with weights, bias and residual loaded after the sums). AHEAD: those are on their way
// before the sums; not for rows of which the registers hold less than half (3000 rows of 11008: 95 us, 80 without).
template <int CPT, bool AHEAD>
__global__ void __launch_bounds__(256) layernorm_kernel(const float* __restrict__ y, const float* __restrict__ w,
                                                        const float* __restrict__ b, float eps, float mult, int accumulate,
                                                        float* __restrict__ x, uint16_t* __restrict__ x16, int n) {
  __shared__ float red[4];
  const size_t r = blockIdx.x;
  const float* yr = y + r * n;
  float v[CPT], wv[CPT], bv[CPT], xv[CPT];
  float s = 0.0f;
#pragma unroll
  for (int e = 0; e < CPT; ++e) {
    const int i = min((int)threadIdx.x + 256 * e, n - 1);
    v[e] = yr[i];
    if (!AHEAD) continue;
    wv[e] = w[i];
    bv[e] = b ? b[i] : 0.0f;
    xv[e] = accumulate ? x[r * n + i] : 0.0f;
  }
#pragma unroll
  for (int e = 0; e < CPT; ++e) {
    if ((int)threadIdx.x + 256 * e >= n) v[e] = 0.0f;
    s += v[e];
  }
  for (int i = threadIdx.x + 256 * CPT; i < n; i += 256) s += yr[i];
  const float mean = block_sum_256(s, red) / (float)n;
  float q = 0.0f;
#pragma unroll
  for (int e = 0; e < CPT; ++e) {
    const float dlt = threadIdx.x + 256 * e < n ? v[e] - mean : 0.0f;
    q = fmaf(dlt, dlt, q);
  }
  for (int i = threadIdx.x + 256 * CPT; i < n; i += 256) {
    const float dlt = yr[i] - mean;
    q = fmaf(dlt, dlt, q);
  }
  const float rstd = 1.0f / sqrtf(block_sum_256(q, red) / (float)n + eps);
  auto put = [&](int i, float val, float wi, float bi, float xi) {
#pragma clang fp contract(off)  // (product and sum rounded apart, accumulating or not)
    float o = mult * fmaf((val - mean) * rstd, wi, bi);
    if (accumulate) o += xi;
    x[r * n + i] = o;
    if (x16) x16[r * n + i] = f2bf(o);
  };
#pragma unroll
  for (int e = 0; e < CPT; ++e) {
    const int i = threadIdx.x + 256 * e;
    if (i >= n) continue;
    if (AHEAD) put(i, v[e], wv[e], bv[e], xv[e]);
    else put(i, v[e], w[i], b ? b[i] : 0.0f, accumulate ? x[r * n + i] : 0.0f);
  }
  for (int i = threadIdx.x + 256 * CPT; i < n; i += 256)
    put(i, yr[i], w[i], b ? b[i] : 0.0f, accumulate ? x[r * n + i] : 0.0f);
}

// z <- cap * tanh(z / cap)
__global__ void __launch_bounds__(256) softcap_kernel(float* __restrict__ z, size_t n, float cap) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) z[i] = cap * tanhf(z[i] / cap);
}

// grid (rows, groups): group g of row r is x[r * ldx + g * n .. + n); weight (may be null) is indexed within a group. A row's first
// 256 CPT columns and their weights are loaded ahead of the sum: few rows are a trip to memory each way (one row of 2048 4.0
// us with the row read again and the weights behind the sum, 2.6 here; 2407 rows of 4096 24.5 / 12.7)
template <int CPT>
__global__ void __launch_bounds__(256) rmsnorm_kernel(const float* __restrict__ x, long ldx, const float* __restrict__ w,
                                                      float offset, float eps, float* __restrict__ y, long ldy, int n,
                                                      uint16_t* __restrict__ y16) {
  __shared__ float red[4];
  const float* xr = x + (size_t)blockIdx.x * ldx + (size_t)blockIdx.y * n;
  float* yr = y + (size_t)blockIdx.x * ldy + (size_t)blockIdx.y * n;
  float ss = 0.0f, r[CPT], g[CPT];
#pragma unroll
  for (int e = 0; e < CPT; ++e) {
    const int i = min((int)threadIdx.x + 256 * e, n - 1);
    r[e] = xr[i];
    g[e] = w ? w[i] : 0.0f;
  }
#pragma unroll
  for (int e = 0; e < CPT; ++e)
    if ((int)threadIdx.x + 256 * e < n) ss = fmaf(r[e], r[e], ss);
  for (int i = threadIdx.x + 256 * CPT; i < n; i += 256) ss = fmaf(xr[i], xr[i], ss);
  ss = block_sum_256(ss, red);
  const float rstd = 1.0f / sqrtf(ss / (float)n + eps);
  uint16_t* yb = y16 ? y16 + (size_t)blockIdx.x * ldy + (size_t)blockIdx.y * n : nullptr;
  auto put = [&](int i, float x_, float g_) {
    const float v = x_ * rstd * (w ? offset + g_ : 1.0f);
    yr[i] = v;
    if (yb) yb[i] = f2bf(v);  // the rounded copy the matrix cores read
  };
#pragma unroll
  for (int e = 0; e < CPT; ++e)
    if ((int)threadIdx.x + 256 * e < n) put(threadIdx.x + 256 * e, r[e], g[e]);
  for (int i = threadIdx.x + 256 * CPT; i < n; i += 256) put(i, xr[i], w ? w[i] : 0.0f);
}

// y[i] = x[rows[i]] (row gather of the positions whose logits are asked for)
__global__ void __launch_bounds__(256) gather_rows_kernel(const float* __restrict__ x, const int* __restrict__ rows,
                                                          float* __restrict__ y, int W) {
  const size_t src = (size_t)rows[blockIdx.x] * W, dst = (size_t)blockIdx.x * W;
  for (int i = threadIdx.x; i < W; i += 256) y[dst + i] = x[src + i];
}

}  // namespace lgs

extern "C" int lgs_linear(const void* a_any, long lda, long stride_a, const void* w, int w_f32, long stride_w, void* y_any,
                          long ldy, long stride_y, int M, int N, int K, int batch, int accumulate, int act,
                          const int* a_rows, const int* z_start, int a_bf16, int y_bf16, const float* bias, float* part,
                          int ksplit, hipStream_t stream) {
  const float* a = (const float*)a_any;  // (bf16 when a_bf16)
  float* y = (float*)y_any;              // (bf16 when y_bf16)
  LGA_CHECK_ARG(a && w && y, "lgs_linear: null pointer");
  LGA_CHECK_ARG(!a_bf16 || (!w_f32 && (M > 8 || z_start || a_rows)),
                "lgs_linear: a bf16 A operand goes with bf16 weights on the MFMA tiles (more than 8 rows)");
  LGA_CHECK_ARG(M > 0 && N > 0 && K > 0 && batch > 0 && batch <= 65535, "lgs_linear: bad sizes");
  LGA_CHECK_ARG(lda >= K && ldy >= N, "lgs_linear: row strides shorter than the rows");
  LGA_CHECK_ARG(act >= 0 && act <= lgs::kActSigmoid, "lgs_linear: unknown activation");
  LGA_CHECK_ARG(!y_bf16 || (!w_f32 && !accumulate && (M > 8 || z_start || a_rows)),
                "lgs_linear: a bf16 result comes from the MFMA tiles (bf16 weights, more than 8 rows, no accumulate)");
  lgs::LinArgs p{a, lda, stride_a, w, stride_w, y, ldy, stride_y, M, N, K, accumulate, act, a_rows, z_start,
                 a_bf16 ? (const uint16_t*)a : nullptr, y_bf16 ? (uint16_t*)y : nullptr, bias, nullptr, 1, 0};
  LGA_CHECK_ARG(ksplit >= 1 && (ksplit == 1 || (part && !w_f32 && batch == 1 && !z_start && !a_rows && M > 8 && M <= 65535)),
                "lgs_linear: K is split for one plain product on the MFMA tiles, with a workspace");
  // A row's bits are not those that it has alone: lin_gemv_kernel adds in another order
  if (!z_start && !a_rows && !w_f32 && lgs::lin_rows_pay(M, (long)N * batch, K) && lda % 4 == 0 && stride_a % 4 == 0 &&
      stride_w % 8 == 0 && ((uintptr_t)a | (uintptr_t)w) % 16 == 0) {
    if (N < 4096) lgs::lin_rows_go<1, 8>(p, batch, stream);
    else if (M > 4 && (N >= 16384 || (N > 4096 && N < 8192 && K >= 2048))) lgs::lin_rows_go<2, 4>(p, batch, stream);
    else lgs::lin_rows_go<1, 4>(p, batch, stream);
    LGA_LAUNCH_RETURN();
  }
  if (M <= 8 && !z_start && !a_rows) {
    const int R = N >= 16384 ? 4 : (N >= 4096 ? 2 : 1);
    const bool deep = lgs::gemv_deep((long)N * batch, K);
    const dim3 grid(deep ? N : (N + 4 * R - 1) / (4 * R), batch);
#define LGS_GEMV_R(MT, RR, KS)                                                                 \
  do {                                                                                         \
    if (w_f32) lgs::lin_gemv_kernel<true, MT, RR, KS, false><<<grid, 256, 0, stream>>>(p);     \
    else lgs::lin_gemv_kernel<false, MT, RR, KS, false><<<grid, 256, 0, stream>>>(p);          \
  } while (0)
#define LGS_GEMV(MT)                       \
  do {                                     \
    if (R == 4) LGS_GEMV_R(MT, 4, 1);      \
    else if (R == 2) LGS_GEMV_R(MT, 2, 1); \
    else if (deep) LGS_GEMV_R(MT, 1, 4);   \
    else LGS_GEMV_R(MT, 1, 1);             \
  } while (0)
    const bool ahead = M == 2 ? R == 1 && K >= 1024 : M == 1 && (R == 1 ? N <= 3072 && K >= 1536 : R == 2 && K > 1536 && K <= 2048);
    if (!w_f32 && !deep && ahead) {
      if (R == 2) lgs::lin_gemv_kernel<false, 1, 2, 1, true><<<grid, 256, 0, stream>>>(p);
      else if (M == 1) lgs::lin_gemv_kernel<false, 1, 1, 1, true><<<grid, 256, 0, stream>>>(p);
      else lgs::lin_gemv_kernel<false, 2, 1, 1, true><<<grid, 256, 0, stream>>>(p);
      LGA_LAUNCH_RETURN();
    }
    if (M == 1) LGS_GEMV(1);
    else if (M == 2) LGS_GEMV(2);
    else if (M <= 4) LGS_GEMV(4);
    else LGS_GEMV(8);
#undef LGS_GEMV
#undef LGS_GEMV_R
    LGA_LAUNCH_RETURN();
  }
  if (w_f32) {
    const dim3 grid((N + 63) / 64, (M + 63) / 64, batch);
    LGA_CHECK_ARG(grid.y <= 65535, "lgs_linear: too many rows");
    lgs::lin_fma_kernel<true><<<grid, 256, 0, stream>>>(p);
    LGA_LAUNCH_RETURN();
  }
  const int am = a_bf16 ? 8 : 4;  // elements per 16 bytes of A
  const bool vec = K % 8 == 0 && lda % am == 0 && stride_a % am == 0 && stride_w % 8 == 0 && (uintptr_t)a % 16 == 0 &&
                   (uintptr_t)w % 16 == 0;
  if (ksplit > 1) {
    const int nk = (K + lgs::BK - 1) / lgs::BK;
    p.part = part;
    p.kper = (nk + ksplit - 1) / ksplit;
    p.ksplit = (nk + p.kper - 1) / p.kper;  // (no empty range)
  }
  if (a_bf16 && vec && std::max(ldy, (long)N) < (1L << 28)) {  // (a lane's place in four rows of Y: 32 bits)
    if (lgs::gemm_narrow(p, batch, stream)) LGA_LAUNCH_RETURN();
    const lgs::GemmPlan plan = lgs::gemm_plan(M, N, K, batch, z_start != nullptr, p.ksplit, act, accumulate != 0);
    if (plan.tile >= 0) {
      const int rc = lgs::gemm_launch(p, plan, batch, stream);
      if (rc) return rc;
      if (p.ksplit > 1) lgs::lin_sum_kernel<<<dim3((N + 255) / 256, M), 256, 0, stream>>>(p);
      LGA_LAUNCH_RETURN();
    }
  }
  const dim3 grid((N + lgs::BN - 1) / lgs::BN, (M + lgs::BM - 1) / lgs::BM, p.ksplit > 1 ? p.ksplit : batch);
  LGA_CHECK_ARG(grid.y <= 65535, "lgs_linear: too many rows");
#define LGS_MFMA(NARROW)                                                                    \
  do {                                                                                      \
    if (a_bf16 && vec) lgs::lin_mfma_kernel<true, true, NARROW><<<grid, 256, 0, stream>>>(p); \
    else if (a_bf16) lgs::lin_mfma_kernel<false, true, NARROW><<<grid, 256, 0, stream>>>(p); \
    else if (vec) lgs::lin_mfma_kernel<true, false, NARROW><<<grid, 256, 0, stream>>>(p);   \
    else lgs::lin_mfma_kernel<false, false, NARROW><<<grid, 256, 0, stream>>>(p);           \
  } while (0)
  if (N <= 18 || (N < 32 && (p.ksplit > 1 ? N : ldy) % 4 != 0)) LGS_MFMA(true);
  else LGS_MFMA(false);
#undef LGS_MFMA
  if (p.ksplit > 1) lgs::lin_sum_kernel<<<dim3((N + 255) / 256, M), 256, 0, stream>>>(p);
  LGA_LAUNCH_RETURN();
}

static bool glu_served(int M, int n, int K) {
  return M > 8 && n >= 32 && n % 4 == 0 && n <= (1 << 29) && K > 0 && K % 64 == 0;
}
// whether a product of M rows (the sizes of all its groups; groups 0: one plain product) on gate | up of n columns each is best
// made by lgs_linear_glu: not where the plain product is better made in ranges of K, or on the tiles for few rows of many groups
extern "C" int lgs_linear_glu_fits(int M, int n, int K, int groups) {
  if (!glu_served(M, n, K)) return 0;
  return (groups > 0 ? !lgs::gemm_few_rows(M, groups) : lgs::gemm_plan(M, 2 * n, K, 1, false, 0).ksplit == 1) ? 1 : 0;
}

extern "C" int lgs_linear_glu(const void* a, long lda, const void* w, long stride_w, long up_rows, void* y, long ldy, int M,
                              int n, int K, int batch, const int* a_rows, const int* z_start, int act, int clamped,
                              float alpha, float limit, float shift, hipStream_t stream) {
  LGA_CHECK_ARG(a && w && y, "lgs_linear_glu: null pointer");
  LGA_CHECK_ARG(glu_served(M, n, K), "lgs_linear_glu: not one of its sizes");
  LGA_CHECK_ARG(batch > 0 && batch <= 65535 && (batch == 1 || z_start), "lgs_linear_glu: batches are groups of rows");
  LGA_CHECK_ARG(lda >= K && ldy >= n && up_rows >= n, "lgs_linear_glu: row strides shorter than the rows");
  LGA_CHECK_ARG(act >= 0 && act <= lgs::kActSigmoid, "lgs_linear_glu: unknown activation");
  LGA_CHECK_ARG(((uintptr_t)a | (uintptr_t)w) % 16 == 0 && (uintptr_t)y % 8 == 0 && lda % 8 == 0 && stride_w % 8 == 0 &&
                    ldy % 4 == 0,
                "lgs_linear_glu: rows of A and W start on 16 bytes, of Y on 8");
  lgs::LinArgs p{nullptr, lda, 0, w, stride_w, nullptr, ldy, 0, M, n, K, 0, act, a_rows, z_start, (const uint16_t*)a,
                 (uint16_t*)y, nullptr, nullptr, 1, 0};
  const lgs::GluForm f{clamped, act, alpha, limit, shift, (size_t)up_rows * K};
  const int rc = lgs::gemm_glu_launch(p, f, batch, stream);
  if (rc) return rc;
  LGA_LAUNCH_RETURN();
}

extern "C" int lgs_linear_glu_row_fits(int columns, int K) { return columns > 0 && K > 0 && K % 8 == 0 && !lgs::gemv_deep(columns, K) && !lgs::lin_rows_pay(1, columns, K) ? 1 : 0; }

extern "C" int lgs_linear_glu_row(const float* a, const void* w, long up_rows, float* y, int n, int K, int act, int clamped,
                                  float alpha, float limit, float shift, hipStream_t stream) {
  LGA_CHECK_ARG(a && w && y && n > 0 && K > 0 && up_rows >= n, "lgs_linear_glu_row: bad arguments");
  LGA_CHECK_ARG(act >= 0 && act <= lgs::kActSigmoid, "lgs_linear_glu_row: unknown activation");
  LGA_CHECK_ARG(K % 8 == 0 && ((uintptr_t)a | (uintptr_t)w) % 16 == 0, "lgs_linear_glu_row: rows of eight values, 16-byte alignment");
  const lgs::GluForm f{clamped, act, alpha, limit, shift, (size_t)up_rows * K};
  const unsigned grid = (unsigned)((n + 3) / 4);
  const uint16_t* m = (const uint16_t*)w;
  if (K <= 2048) {  // (as lin_gemv_kernel's two columns a wave)
    if (clamped) lgs::lin_glu_row_kernel<true, true><<<grid, 256, 0, stream>>>(a, m, f, y, n, K);
    else lgs::lin_glu_row_kernel<true, false><<<grid, 256, 0, stream>>>(a, m, f, y, n, K);
  } else {
    if (clamped) lgs::lin_glu_row_kernel<false, true><<<grid, 256, 0, stream>>>(a, m, f, y, n, K);
    else lgs::lin_glu_row_kernel<false, false><<<grid, 256, 0, stream>>>(a, m, f, y, n, K);
  }
  LGA_LAUNCH_RETURN();
}

// ranges of K that a plain product of a bf16 A on bf16 weights is best made in (1: as one)
extern "C" int lgs_linear_ksplit(int M, int N, int K) {
  return M > 8 && M <= 65535 && N > 0 && K > 0 ? lgs::gemm_plan(M, N, K, 1, false, 0).ksplit : 1;
}
// the tile (LGA_GEMM_FORMS) that such a product is made with, by ksplit ranges of K or (gated) with its unit; -1: none of them
extern "C" int lgs_linear_form(int M, int N, int K, int batch, int grouped, int ksplit, int act, int gated) {
  if (M <= 8 || N <= 0 || K <= 0 || batch <= 0 || ksplit <= 0) return -1;
  if (gated) return glu_served(M, N, K) ? lgs::gemm_glu_plan(M, N, K, batch, grouped != 0).tile : -1;
  return lgs::gemm_plan(M, N, K, batch, grouped != 0, ksplit, act).tile;
}

extern "C" int lgs_embed(const int* tokens, const void* table, int w_f32, float scale, float* x, int T, int W,
                         int vocab, hipStream_t stream) {
  LGA_CHECK_ARG(tokens && table && x && T > 0 && W > 0 && vocab > 0, "lgs_embed: bad arguments");
  if (w_f32) lgs::embed_kernel<true><<<lgs::embed_grid(T, W), 256, 0, stream>>>(tokens, table, x, W, vocab, scale);
  else lgs::embed_kernel<false><<<lgs::embed_grid(T, W), 256, 0, stream>>>(tokens, table, x, W, vocab, scale);
  LGA_LAUNCH_RETURN();
}

extern "C" int lgs_embed_pos(const int* tokens, const int* pos, const void* table, const void* pos_table, int w_f32,
                             float scale, float* x, void* x_bf16, int T, int W, int vocab, int positions,
                             hipStream_t stream) {
  LGA_CHECK_ARG(tokens && pos && table && pos_table && x && T > 0 && W > 0 && vocab > 0 && positions > 0,
                "lgs_embed_pos: bad arguments");
  const dim3 grid = lgs::embed_grid(T, W);
  if (w_f32)
    lgs::embed_pos_kernel<true><<<grid, 256, 0, stream>>>(tokens, pos, table, pos_table, x, (uint16_t*)x_bf16, W, vocab,
                                                       positions, scale);
  else
    lgs::embed_pos_kernel<false><<<grid, 256, 0, stream>>>(tokens, pos, table, pos_table, x, (uint16_t*)x_bf16, W, vocab,
                                                        positions, scale);
  LGA_LAUNCH_RETURN();
}

extern "C" int lgs_layernorm(const float* y, const float* weight, const float* bias, float eps, float mult,
                             int accumulate, float* x, void* x_bf16, int rows, int n, hipStream_t stream) {
  LGA_CHECK_ARG(y && weight && x && rows > 0 && n > 0, "lgs_layernorm: bad arguments");
#define LGS_NORM(CPT, AHEAD) \
  lgs::layernorm_kernel<CPT, AHEAD><<<rows, 256, 0, stream>>>(y, weight, bias, eps, mult, accumulate, x, (uint16_t*)x_bf16, n)
  if (n <= 256) LGS_NORM(1, true);
  else if (n <= 1024) LGS_NORM(4, true);
  else if (n <= 2048) LGS_NORM(8, true);
  else if (n <= 8192) LGS_NORM(16, true);
  else LGS_NORM(16, false);
#undef LGS_NORM
  LGA_LAUNCH_RETURN();
}

extern "C" int lgs_softcap(float* z, long n, float cap, hipStream_t stream) {
  LGA_CHECK_ARG(z && n > 0 && cap > 0.0f, "lgs_softcap: bad arguments");
  lgs::softcap_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(z, (size_t)n, cap);
  LGA_LAUNCH_RETURN();
}

extern "C" int lgs_rmsnorm(const float* x, long ldx, const float* weight, float offset, float eps, float* y, long ldy,
                           int rows, int groups, int n, void* y_bf16, hipStream_t stream) {
  LGA_CHECK_ARG(x && y && rows > 0 && groups > 0 && groups <= 65535 && n > 0, "lgs_rmsnorm: bad arguments");
#define LGS_RMSNORM(CPT) \
  lgs::rmsnorm_kernel<CPT><<<dim3(rows, groups), 256, 0, stream>>>(x, ldx, weight, offset, eps, y, ldy, n, (uint16_t*)y_bf16)
  if (n <= 256) LGS_RMSNORM(1);
  else if (n <= 1024) LGS_RMSNORM(4);
  else if (n <= 2048) LGS_RMSNORM(8);
  else LGS_RMSNORM(16);
#undef LGS_RMSNORM
  LGA_LAUNCH_RETURN();
}

extern "C" int lgs_gather_rows(const float* x, const int* rows, float* y, int n_rows, int W, hipStream_t stream) {
  LGA_CHECK_ARG(x && rows && y && n_rows > 0 && W > 0, "lgs_gather_rows: bad arguments");
  lgs::gather_rows_kernel<<<n_rows, 256, 0, stream>>>(x, rows, y, W);
  LGA_LAUNCH_RETURN();
}
