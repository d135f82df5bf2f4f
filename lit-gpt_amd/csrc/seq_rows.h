// Products of up to eight fp32 rows with bf16 weights on the matrix cores, for kernels that finish the sums themselves.
#pragma once

#include "gemm_tiles.h"
#include "seq_common.h"

namespace lgs {

typedef __bf16 rows_bf16x8 __attribute__((ext_vector_type(8)));
typedef float rows_f32x4 __attribute__((ext_vector_type(4)));

// Up to eight rows of A on bf16 weights, on the matrix cores: the operands are the same (A rounded to bf16), and a weight
// costs no vector instruction however many rows there are. A workgroup owns 16 NR columns; its KW waves each take a
// range of K, 128 values at a time: the columns' 256 bytes of W and the MR rows' 512 of A come by LDS-DMA (whole lines,
// source-swizzled so that fragments are read without bank conflicts) into LDS of the wave's own, so that no barrier is theirs, and are
// fetched anew as soon as they are in registers. One block's buffers a wave where several workgroups share a compute unit: they hide its
// trips better than blocks ahead do (us with one / two blocks' buffers: 8 x 32000 x 2048 30.2 / 32.8, x 8192 x 2048 9.4 / 10.2, x 8192 x 4096
// 15.2 / 16.6, 3 x 6144 x 4096 12.6 / 13.5); two where a workgroup of four waves has one alone (8 x 4096 x 4096 11.3 / 9.3, 3 rows 10.0 / 8.7,
// 11264 long 23.2 / 18.1, 8 x 6144 x 4096 14.7 / 13.4, 8 x 4096 x 2048 7.2 / 6.6; three are no faster, eight waves' 128 KB slower: 8 x 2048 x
// 2048 5.9 / 6.6). The rows are read as vectors of the compiler's own: a read of HIP's float4 may alias the DMAs for it, and waits for all.
// Sums: two instructions (one below K 2048), then vector adds, then the ranges pairwise, so that the error against float64 is at most
// what the lanes' sums of lin_gemv_kernel leave: rms of 8 rows at K 128 / 512 / 1024 / 2048 / 4096 / 11008 4.8e-8 / 6.1e-8 / 6.7e-8 / 7.4e-8
// / 8.0e-8 / 9.5e-8 of the results, 4.8e-8 / 6.2e-8 / 6.8e-8 / 7.5e-8 / 8.4e-8 / 1.1e-7 there. (Two instructions at K 128 / 512 / 1024 5.0e-8 /
// 6.3e-8 / 6.9e-8, one at 4096 / 11008 8.3e-8 / 1.1e-7; one chain of instructions 1.5 to 3 times as much.)
// Bound by memory, with few columns by its latency. Loaded into registers as the instructions take them, every lane's 16 bytes lay
// in a line of their own, and a compute unit got some 17 bytes a ns of W and A together, from whichever cache. us there / here, weights
// from memory, the same bits: 8 x 2048 x 2048 11.9 / 5.9, x 4096 x 2048 10.1 / 6.6, x 6288 x 2048 14.2 / 9.0, x 32000 x 2048 44.5 / 30.2, x
// 4096 x 4096 14.4 / 9.3, x 12288 x 4096 35.2 / 23.4, 3 x 12288 x 4096 30.5 / 20.6, x 32000 x 4096 59 / 48.
template <int NR, int KW, int MR, int RB>
struct RowsTile {
  static constexpr int W_BYTES = NR * 4096, A_BYTES = MR * 512, SLOT = W_BYTES + A_BYTES, LDS = KW * RB * SLOT;
  static_assert(LDS <= 163840 && NR * 1024 <= SLOT, "LDS");
};

// Whether a sum takes one instruction
inline bool rows_one(int K) { return K < 2048; }

// weights(r): the K values of column r of the workgroup's 16 NR; x0: M rows, ldx apart. The ranges' sums are left in LDS, for rows_sum
// behind the barrier that ends this.
template <int NR, int KW, int MR, int RB, bool ONE, class Weights>
__device__ __forceinline__ void rows_products(unsigned char* lds_all, Weights&& weights, const float* x0, long ldx, int M, int K) {
  using T = RowsTile<NR, KW, MR, RB>;
  constexpr int W_BYTES = T::W_BYTES, SLOT = T::SLOT, PW = NR * 4, PA = MR / 2;
  const int tid = threadIdx.x, lane = tid & 63, l15 = lane & 15, q4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned char* lds = lds_all + wave * (RB * SLOT);
  const int nb = K / 128, b0 = wave * nb / KW, b1 = (wave + 1) * nb / KW;
  const unsigned char *w[PW], *a[PA];
#pragma unroll
  for (int i = 0; i < PW; ++i) {  // four rows of 256 bytes
    const int row = i * 4 + q4;
    w[i] = (const unsigned char*)weights(row) + 16 * (l15 ^ (row & 15));
  }
#pragma unroll
  for (int i = 0; i < PA; ++i) {  // two rows of 512
    const int row = i * 2 + (lane >> 5);
    a[i] = (const unsigned char*)(x0 + (size_t)min(row, M - 1) * ldx) + 16 * ((lane & 31) ^ row);
  }
  auto dma = [&](int b, int slot) {  // (past the range: its last block, never used)
    const size_t at = (size_t)min(b, b1 - 1) * 256;
#pragma unroll
    for (int i = 0; i < PW; ++i) lga::gemm_dma16(w[i] + at, lds + slot + i * 1024);
#pragma unroll
    for (int i = 0; i < PA; ++i) lga::gemm_dma16(a[i] + 2 * at, lds + slot + W_BYTES + i * 1024);
  };
  const rows_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  rows_f32x4 acc[4][NR];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NR; ++j) acc[i][j] = zero;
  if (b0 < b1) {  // (fewer blocks than waves: those without one fetch nothing)
#pragma unroll
    for (int r = 0; r < RB; ++r) dma(b0 + r, r * SLOT);
  }
  int slot = 0;
  const int arow = l15 & (MR - 1), w_at = l15 * 256, a_at = W_BYTES + arow * 512;
  for (int b = b0; b < b1; b += 2) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (b + s < b1) {
        lga::gemm_wait_vm<(RB - 1) * (PW + PA)>();
        rows_bf16x8 wr[4][NR];
        rows_f32x4 x[4][2];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
#pragma unroll
          for (int j = 0; j < NR; ++j) wr[m][j] = *(const rows_bf16x8*)(lds + slot + w_at + j * 4096 + 16 * ((m * 4 + q4) ^ l15));
#pragma unroll
          for (int e = 0; e < 2; ++e) x[m][e] = *(const rows_f32x4*)(lds + slot + a_at + 16 * ((m * 8 + q4 * 2 + e) ^ arow));
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (read before it is filled again)
        __builtin_amdgcn_sched_barrier(0);
        if (RB > 1 || b + s + RB < b1) dma(b + s + RB, slot);  // (several are counted by the wait: one more always)
        slot = slot + SLOT == RB * SLOT ? 0 : slot + SLOT;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          rows_f32x4 v[2][NR];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const int m = 2 * u + e;
            const uint4 x16 = make_uint4(pack2(x[m][0].x, x[m][0].y), pack2(x[m][0].z, x[m][0].w), pack2(x[m][1].x, x[m][1].y), pack2(x[m][1].z, x[m][1].w));
#pragma unroll
            for (int j = 0; j < NR; ++j)
              v[e][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wr[m][j], __builtin_bit_cast(rows_bf16x8, x16),
                                                                ONE || e == 0 ? zero : v[0][j], 0, 0, 0);
          }
#pragma unroll
          for (int e = ONE ? 0 : 1; e < 2; ++e)
#pragma unroll
            for (int j = 0; j < NR; ++j) acc[s * 2 + u][j] += v[e][j];
        }
      }
    }
  }
  lga::gemm_wait_vm<0>();  // no DMA may outlive its slot
  __syncthreads();
  rows_f32x4* part = (rows_f32x4*)lds_all;  // [KW][NR][64]
#pragma unroll
  for (int j = 0; j < NR; ++j) part[(wave * NR + j) * 64 + lane] = (acc[0][j] + acc[1][j]) + (acc[2][j] + acc[3][j]);
  __syncthreads();
}

// row l15's sums with columns 4 q4 .. + 3 of group j, in lane 16 q4 + l15
template <int NR, int KW>
__device__ __forceinline__ rows_f32x4 rows_sum(const unsigned char* lds_all, int j, int lane) {
  const rows_f32x4* part = (const rows_f32x4*)lds_all;  // [KW][NR][64]
  rows_f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < KW; k += 4) {
    const rows_f32x4* at = part + (k * NR + j) * 64 + lane;
    v += (at[0] + at[NR * 64]) + (at[2 * NR * 64] + at[3 * NR * 64]);
  }
  return v;
}

}  // namespace lgs
