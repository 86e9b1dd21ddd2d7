// y[M, N] = x[M, K] . w[N, K]^T in float32 throughout, on the float32 matrix instructions (v_mfma_f32_16x16x4_f32: float32
// operands, float32 products and sums; 256 operations a cycle and compute unit, the vector unit's fused multiply-adds
// half of that). The 32-bit path's product for any number of rows (reference layers/linear.py:26,45: F.linear).
//
// The order in which an output's K terms are added must not depend on how many rows the launch has, so that a token's
// result is the same bits however its request was cut: K is walked in blocks of 32, block i belongs to wave i mod 4 of
// the workgroup, and the four waves' sums meet as (0 + 1) + (2 + 3). The tile (TM rows x TN features, every wave the whole
// tile over its share of K) is then free to follow the shape. No two waves of a workgroup read the same operand, so
// operands go from memory to registers: a lane holds 4 consecutive k of one row (16 lanes x 4 lane groups: 16 k of 16
// rows, 64 bytes of each row a load, the other half of the line in the step behind it), which are the operands of
// four matrix instructions (both operands see the same permutation of k). A ring of DEPTH steps of loads is in flight.
// Workgroups that share weight rows run side by side on one XCD, at most 8 tiles of rows at a time, so that a weight
// comes from memory once and the rows stay in that XCD's L2.
// Measured (us; in brackets a kernel of 64 x 64 tiles through LDS with plain multiply-adds, the 32-bit product before): 300
// rows of 4096 x 1024 42 (194), 1024 x 2048 24 (380), 6144 x 1024 58 (200), 1024 x 3072 36 (560), 151936 x 1024 1,258 (2,400;
// 74 TFLOP/s, about half of the 157 that the matrix pipes could do at 2.4 GHz: a full chip of them does not keep that clock;
// 80 workgroups alone reach 82 % of it). Few and many rows: one row of 4096 x 1024 7.3 (125), of 4096 x 12288 34 (1,694), 64 rows
// of it 93 (2,008), 4,096 rows 4,990 (8,480; 83 TFLOP/s). Error against 64 bits over 1,024-3,072 terms 3-5e-7 of the result's
// norm, less than one chain of multiply-adds (four shorter chains).
#include "common.h"

// Keeps a step's loads where they are issued (else they sink to their use in the next round of the ring).
__device__ __forceinline__ void f32_pin() { asm volatile("" ::: "memory"); }

#define F32_ROW_GROUP 8

// VEC: rows of 16-byte aligned pieces, K in whole steps of 4 (else every value is loaded by itself; the same sums).
template <int TM, int TN, int DEPTH, bool VEC>
__global__ void __launch_bounds__(256)
gemm_f32_kernel(const float* __restrict__ x, int64_t ldx, const float* __restrict__ w, int64_t ldw, float* __restrict__ y,
                int64_t ldy, int M, int N, int K, int m_tiles, int n_tiles, int vec_out) {
  constexpr int MI = TM / 16, NI = TN / 16;
  __shared__ f32x4 merge[2][4][TM * 4];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int rows = min(F32_ROW_GROUP, m_tiles), per_xcd = (n_tiles + 7) >> 3;
  const int group = slot / (per_xcd * rows), rest = slot % (per_xcd * rows);
  const int mt = group * rows + rest % rows, nt = rest / rows * 8 + xcd;
  if (mt >= m_tiles || nt >= n_tiles) return;
  const int m0 = mt * TM, n0 = nt * TN;

  // rows beyond the matrix are read from its last row and never stored
  const float* xr[MI];
  const float* wr[NI];
#pragma unroll
  for (int i = 0; i < MI; ++i) xr[i] = x + (int64_t)min(m0 + 16 * i + r, M - 1) * ldx;
#pragma unroll
  for (int i = 0; i < NI; ++i) wr[i] = w + (int64_t)min(n0 + 16 * i + r, N - 1) * ldw;

  auto first_k = [&](int s) { return ((s >> 1) * 4 + wave) * 32 + (s & 1) * 16; };      // of step s of this wave
  auto piece = [&](const float* row, int k) {
    if (VEC) return *reinterpret_cast<const f32x4*>(row + (k < K ? k : 0));
    f32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = row[k + j < K ? k + j : 0];
    return v;
  };
  f32x4 fx[DEPTH][MI], fw[DEPTH][NI];
  auto fetch = [&](int s, f32x4 (&bx)[MI], f32x4 (&bw)[NI]) {
    const int k = first_k(s) + 4 * g;
#pragma unroll
    for (int i = 0; i < NI; ++i) bw[i] = piece(wr[i], k);
#pragma unroll
    for (int i = 0; i < MI; ++i) bx[i] = piece(xr[i], k);
    f32_pin();
  };
  f32x4 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int d = 0; d < DEPTH; ++d) fetch(d, fx[d], fw[d]);
  const int steps = 2 * ((K + 127) / 128);
  for (int s0 = 0; s0 < steps; s0 += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      const int s = s0 + d, k0 = first_k(s);
      if (k0 < K) {
        if (k0 + 16 > K) {                       // terms beyond K are zeros in both operands
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const bool in = k0 + 4 * g + j < K;
#pragma unroll
            for (int i = 0; i < MI; ++i) fx[d][i][j] = in ? fx[d][i][j] : 0.f;
#pragma unroll
            for (int i = 0; i < NI; ++i) fw[d][i][j] = in ? fw[d][i][j] : 0.f;
          }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int n = 0; n < NI; ++n)
              acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[d][n][j], fx[d][i][j], acc[i][n], 0, 0, 0);
      }
      fetch(s + DEPTH, fx[d], fw[d]);            // beyond the last step: row starts, never used
    }
  }

  // a lane holds features 4 g .. 4 g + 3 of row r: the waves' sums meet 16 features at a time through LDS
#pragma unroll
  for (int n = 0; n < NI; ++n) {
#pragma unroll
    for (int i = 0; i < MI; ++i) merge[n & 1][wave][(16 * i + r) * 4 + g] = acc[i][n];
    __syncthreads();                             // the buffer of the round before is free again two rounds on
    for (int e = tid; e < TM * 4; e += 256) {
      const f32x4 v = (merge[n & 1][0][e] + merge[n & 1][1][e]) + (merge[n & 1][2][e] + merge[n & 1][3][e]);
      const int m = m0 + e / 4, f = n0 + 16 * n + (e & 3) * 4;
      if (m < M) {
        float* at = y + (int64_t)m * ldy + f;
        if (vec_out && f + 3 < N) *reinterpret_cast<f32x4*>(at) = v;
        else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (f + j < N) at[j] = v[j];
        }
      }
    }
  }
}

extern "C" int me_gemm_f32(const float* x, int64_t ldx, const float* w, int64_t ldw, float* y, int64_t ldy, int M, int N, int K,
                           int tile_rows, int tile_features, hipStream_t stream) {
  if (M == 0 || N == 0) return 0;
  ME_CHECK(K >= 1 && ldx >= K && ldw >= K && ldy >= N, "gemm (float32): bad leading dimensions");
  ME_CHECK(K <= 2147483647 - 4096, "gemm (float32): rows of %d terms", K);
  const bool vec = K % 4 == 0 && ldx % 4 == 0 && ldw % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0;
  const int vec_out = ldy % 4 == 0 && (uintptr_t)y % 16 == 0;
#define F32_TILE(TM, TN, DEPTH)                                                                                            \
  if (tile_rows == TM && tile_features == TN) {                                                                            \
    const int64_t mt = (M + TM - 1) / TM, nt = (N + TN - 1) / TN, rows = mt < F32_ROW_GROUP ? mt : F32_ROW_GROUP;          \
    const int64_t blocks = (mt + rows - 1) / rows * rows * ((nt + 7) / 8) * 8;                                             \
    ME_CHECK(blocks <= 2147483647ll, "gemm (float32): too many tiles for one launch");                                     \
    if (vec) gemm_f32_kernel<TM, TN, DEPTH, true><<<(unsigned)blocks, 256, 0, stream>>>(x, ldx, w, ldw, y, ldy, M, N, K, (int)mt, (int)nt, vec_out); \
    else gemm_f32_kernel<TM, TN, DEPTH, false><<<(unsigned)blocks, 256, 0, stream>>>(x, ldx, w, ldw, y, ldy, M, N, K, (int)mt, (int)nt, vec_out);    \
    ME_LAUNCH_CHECK();                                                                                                     \
    return 0;                                                                                                              \
  }
  F32_TILE(16, 16, 8)
  F32_TILE(16, 32, 4)
  F32_TILE(32, 32, 4)
  F32_TILE(64, 32, 2)
  F32_TILE(64, 64, 2)
#undef F32_TILE
  ME_CHECK(false, "gemm (float32): no tile of %d rows x %d features", tile_rows, tile_features);
}
