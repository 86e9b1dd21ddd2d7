// y[M, N] = x[M, K] . w[N, K]^T of float32 operands to float32 precision on the bfloat16 matrix instructions
// (v_mfma_f32_16x16x32_bf16: products exact, sums float32). The 32-bit path's product for any number of rows (reference
// layers/linear.py:26,45: F.linear).
//
// An operand of 2^-110 or more is the exact sum of three bfloat16 numbers (`Thirds`; smaller ones: F32_SMALLEST), and of the nine products of two operands' thirds the six
// largest are formed, the smallest first; the other three are below 2^-24 of the product. A float32 matrix instruction does
// 256 operations a cycle and compute unit, six of these 683. Weights that came as bfloat16, as most checkpoints
// hold them, have one third only: a wave that sees no bit in the lower halves of its 32 k of weights leaves out the three products
// with their other thirds, which are zeros (the same bits, at twice the rate).
//
// The order in which an output's K terms are added must not depend on how many rows the launch has, so that a token's
// result is the same bits however its request was cut: K is walked in blocks of 32, block i belongs to wave i mod 4 of
// the workgroup, and the four waves' sums meet as (0 + 1) + (2 + 3). The tile (TM rows x TN features, every wave the whole
// tile over its share of K) is then free to follow the shape, every value is split by one wave of a workgroup only, and no wave
// waits for another before the end: each brings its own blocks into a ring in LDS of its own (global_load_lds_dwordx4), reads
// a block into registers, asks for the one behind the ring in its place and works. What bounds it: at many rows the instructions
// that split (3.5 a number of the rows, 1 of bfloat16 weights) and the LDS (a value in and out) about evenly, which is why two or
// three workgroups share a compute unit and the ring of the large tiles is one block; at few rows the chain of a block in a wave.
// The path through LDS is there for the loads: operands read straight into the matrix instruction's layout (neighbouring lanes in
// different rows) come at 14 bytes a cycle and compute unit, whole lines of 128 bytes at more than three times that.
// Workgroups that share weight rows run side by side on one XCD, at most 8 tiles of rows at a time, so that a weight
// comes from memory once and the rows stay in that XCD's L2.
// Measured (us, weights from bfloat16 / with all bits; in brackets the float32 matrix instructions on operands read straight from
// memory, the 32-bit product before): 300 rows of 4096 x 1024 22 / 27 (43), 1024 x 2048 16 / 20 (25), 6144 x 1024 26 / 34 (57), 1024
// x 3072 22 / 28 (37), 151936 x 1024 540 / 738 (1,263). Few rows: 16 of 4096 x 1024 7.1 / 7.4 (8.4), of 1024 x 3072 10.9 / 12.4
// (16.2), one row of 6144 x 1024 8.4 / 8.4 (9.7 / 9.2), of 4096 x 1024 6.5 / 6.7 (6.5), of 12288 x 4096 46 / 46 (56). Behind the product before, for
// one to four rows: few workgroups, a compute unit each, where a block's chain of conversions and products is what is waited for: one row of
// 1024 x 2048 7.4 / 8.2 (7.2), 1024 x 3072 10.2 / 11.3 (9.8), 512 x 4096 13.0 / 14.6 (11.4); four rows 7.4 / 8.2 (8.0), 10.3 / 11.4 (11.0), 13.0 / 14.7 (12.9). A form of
// its own for them would give a token other bits alone than among others; reading a block ahead of its use, deeper rings and a
// second wave to split the features were no faster. Error against 64
// bits over 1,024 / 2,048 / 3,072 / 12,288 terms 1.7 / 2.4 / 2.9 / 6.1e-7 of the result's norm with bfloat16 weights, 2.3 / 3.4 / 4.2 /
// 9.0e-7 with all bits (2.9 / 4.1 / 5.0 / 9.9e-7).
#include "common.h"


#define F32_ROW_GROUP 8
// What three bfloat16 parts cannot give, an infinity, a value that rounds up to one and one below 2^-110, whose last bits are below the
// smallest bfloat16 of 2^-133, shows in the sums: they are not finite, or small. Sums that are not finite, and those below this,
// are formed again (end of the kernel): from here up a value that lost what is below 2^-134 moves a sum by less than float32's own
// rounding as long as its terms' operands add up to less than 2^46. Sums of zero stay: operands below 2^-134 count as zeros where
// none of a sum's terms has larger ones.
#define F32_SMALLEST 0x1f800000u                   // 2^-64

// A lane's 8 values of one row as sums of three bfloat16 numbers each: the value rounded, what that leaves rounded, and the rest,
// which has no more than 8 bits: the three add up to the value exactly. The remainders come from the dot product of two
// bfloat16 pairs with a float32 sum, whose one product that is not zero is the value's own rounded part times -1.
struct Thirds { bf16x8 high, mid, low; };
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t f32_bits(float v) { return __float_as_uint(v); }
template <bool ALL>                                // false: the rounded values alone
__device__ __forceinline__ void f32_thirds(const f32x4 (&v)[2], Thirds& t) {
  union { bf16x2 u[4]; bf16x8 v; } high, mid, low;
  // -1 times the lower, the upper one of a pair; opaque, for as an inline constant of the instruction -1 would stand in both halves
  uint32_t lower = 0x0000bf80u, upper = 0xbf800000u;
  asm("" : "+s"(lower), "+s"(upper));
  const bf16x2 first = __builtin_bit_cast(bf16x2, lower), second = __builtin_bit_cast(bf16x2, upper);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float a = v[j >> 1][(j & 1) * 2], b = v[j >> 1][(j & 1) * 2 + 1];
    high.u[j] = bf16x2{(__bf16)a, (__bf16)b};
    if (ALL) {
      const float ra = __builtin_amdgcn_fdot2_f32_bf16(high.u[j], first, a, false), rb = __builtin_amdgcn_fdot2_f32_bf16(high.u[j], second, b, false);
      mid.u[j] = bf16x2{(__bf16)ra, (__bf16)rb};
      const float sa = __builtin_amdgcn_fdot2_f32_bf16(mid.u[j], first, ra, false), sb = __builtin_amdgcn_fdot2_f32_bf16(mid.u[j], second, rb, false);
      low.u[j] = bf16x2{(__bf16)sa, (__bf16)sb};
    }
  }
  t.high = high.v;
  if (ALL) { t.mid = mid.v; t.low = low.v; }
}

// 16 bytes per lane and load into LDS at lds_addr + 1024 j + 16 lane for load j of a group of two or four; its memory is base +
// voff + 1024 j (an instruction's offset counts on both sides). A group names its place in LDS once.
__device__ __forceinline__ void f32_dma_group(const void* b0, const void* b1, uint32_t v0, uint32_t v1, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %3\n\tglobal_load_lds_dwordx4 %2, %4 offset:1024"
               ::"s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(v0), "v"(v1), "s"(b0), "s"(b1) : "memory");
}
__device__ __forceinline__ void f32_dma_group(const void* b0, const void* b1, const void* b2, const void* b3, uint32_t v0, uint32_t v1,
                                              uint32_t v2, uint32_t v3, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %5\n\tglobal_load_lds_dwordx4 %2, %6 offset:1024\n\t"
               "global_load_lds_dwordx4 %3, %7 offset:2048\n\tglobal_load_lds_dwordx4 %4, %8 offset:3072"
               ::"s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(v0), "v"(v1), "v"(v2), "v"(v3), "s"(b0), "s"(b1), "s"(b2), "s"(b3) : "memory");
}
template <int N> __device__ __forceinline__ void f32_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ void f32_wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// RING: blocks of a wave that wait in LDS or are on their way there; 0: operands that are no whole 16-byte pieces, every value
// loaded by itself straight into registers (the same sums).
// Tiles of 32 x 64 and 64 x 32 are held to 256 registers, of which matrix instructions then use the ordinary ones: the sums are not copied
// to others and back around every block (300 rows, weights from bfloat16 / with all bits, 4096 x 1024 19.9 -> 18.8 / 25.3 -> 24.7 us, 1024 x 2048
// 14.8 -> 13.5 / 20.2 -> 20.3, 1024 x 3072 20.1 -> 18.4 / 28.2 -> 28.5). Smaller ones with all bits lose by it (512 x 4096 14.6 -> 15.1), larger ones
// have more sums than that.
template <int TM, int TN, int RING>
__global__ void __launch_bounds__(256, TM * TN == 2048 ? 2 : 1)
gemm_f32_kernel(const float* __restrict__ x, int64_t ldx, const float* __restrict__ w, int64_t ldw, float* __restrict__ y,
                int64_t ldy, int M, int N, int K, int m_tiles, int n_tiles, int vec_out) {
  constexpr int MI = TM / 16, NI = TN / 16;
  constexpr int ROWS = TM + TN, BLOCK = ROWS * 128, LOADS = ROWS / 8;       // a wave's block of 32 k: bytes, load instructions
  static_assert(LOADS % 2 == 0 && LOADS * RING < 64, "groups of loads, and what the counter of loads can tell apart");
  extern __shared__ __align__(16) unsigned char f32_lds[];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int rows = min(F32_ROW_GROUP, m_tiles), per_xcd = (n_tiles + 7) >> 3;
  const int group = slot / (per_xcd * rows), rest = slot % (per_xcd * rows);
  const int mt = group * rows + rest % rows, nt = rest / rows * 8 + xcd;
  if (mt >= m_tiles || nt >= n_tiles) return;
  const int m0 = mt * TM, n0 = nt * TN;
  const float* x0 = x + (int64_t)m0 * ldx;
  const float* w0 = w + (int64_t)n0 * ldw;

  const int blocks = ((K + 31) / 32 - wave + 3) / 4;     // of this wave: block s holds k from (4 s + wave) 32 on
  auto first_k = [&](int s) { return (s * 4 + wave) * 32; };
  f32x4 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto products = [&](auto wp, auto xp) {         // one third of the features with one third of the rows, added up
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int n = 0; n < NI; ++n) acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wp(n), xp(i), acc[i][n], 0, 0, 0);
  };
  auto work = [&](int k0, f32x4 (&fx)[MI][2], f32x4 (&fw)[NI][2]) {
    if (k0 + 32 > K) {                           // terms beyond K are zeros in both operands
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const bool in = k0 + 8 * g + j < K;
#pragma unroll
        for (int i = 0; i < MI; ++i) fx[i][j >> 2][j & 3] = in ? fx[i][j >> 2][j & 3] : 0.f;
#pragma unroll
        for (int i = 0; i < NI; ++i) fw[i][j >> 2][j & 3] = in ? fw[i][j >> 2][j & 3] : 0.f;
      }
    }
    Thirds tx[MI], tw[NI];
#pragma unroll
    for (int i = 0; i < MI; ++i) f32_thirds<true>(fx[i], tx[i]);
    uint32_t any = 0;
#pragma unroll
    for (int n = 0; n < NI; ++n)
#pragma unroll
      for (int j = 0; j < 8; ++j) any |= f32_bits(fw[n][j >> 2][j & 3]);
    if (__builtin_amdgcn_ballot_w64((any & 0xffffu) != 0) == 0) {
#pragma unroll
      for (int n = 0; n < NI; ++n) f32_thirds<false>(fw[n], tw[n]);
      products([&](int n) { return tw[n].high; }, [&](int i) { return tx[i].low; });
      products([&](int n) { return tw[n].high; }, [&](int i) { return tx[i].mid; });
      products([&](int n) { return tw[n].high; }, [&](int i) { return tx[i].high; });
    } else {
#pragma unroll
      for (int n = 0; n < NI; ++n) f32_thirds<true>(fw[n], tw[n]);
      products([&](int n) { return tw[n].high; }, [&](int i) { return tx[i].low; });
      products([&](int n) { return tw[n].mid; }, [&](int i) { return tx[i].mid; });
      products([&](int n) { return tw[n].low; }, [&](int i) { return tx[i].high; });
      products([&](int n) { return tw[n].high; }, [&](int i) { return tx[i].mid; });
      products([&](int n) { return tw[n].mid; }, [&](int i) { return tx[i].high; });
      products([&](int n) { return tw[n].high; }, [&](int i) { return tx[i].high; });
    }
  };

  if constexpr (RING == 0) {
    for (int s = 0; s < blocks; ++s) {
      const int k0 = first_k(s);
      f32x4 fx[MI][2], fw[NI][2];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int k = min(k0 + 8 * g + j, K - 1);
#pragma unroll
        for (int i = 0; i < MI; ++i) fx[i][j >> 2][j & 3] = x0[(int64_t)min(16 * i + r, M - 1 - m0) * ldx + k];
#pragma unroll
        for (int i = 0; i < NI; ++i) fw[i][j >> 2][j & 3] = w0[(int64_t)min(16 * i + r, N - 1 - n0) * ldw + k];
      }
      work(k0, fx, fw);
    }
  } else {
    // What a lane names in memory: an instruction brings 8 rows of 128 bytes. Piece p of 16 bytes of a row lies in place
    // p ^ (row mod 8) of its line in LDS, so that the 16 rows that are read at once lie in different banks. Rows beyond the
    // matrix are read from its last row and never stored.
    const int own = lane >> 3, p = (lane & 7) ^ own;
    uint32_t voff[LOADS];                        // from 4,096 bytes in front of the tile's first row, less the place in its group
#pragma unroll
    for (int q = 0; q < LOADS; ++q) {
      const int R = 8 * q + own;
      voff[q] = (q < TM / 8 ? (uint32_t)(min(R, M - 1 - m0) * ldx * 4) : (uint32_t)(min(R - TM, N - 1 - n0) * ldw * 4)) + 16 * p + 4096 - 1024 * (q & 3);
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)f32_lds + wave * BLOCK;
    auto stage = [&](int s, int at) {
      const int k0 = first_k(s);
      const char *xk = reinterpret_cast<const char*>(x0 + k0) - 4096, *wk = reinterpret_cast<const char*>(w0 + k0) - 4096;
      const uint32_t to = lds0 + at * 4 * BLOCK;
      auto from = [&](int q) { return q < TM / 8 ? xk : wk; };
      auto groups = [&](uint32_t back) {
#pragma unroll
        for (int q = 0; q + 3 < LOADS; q += 4)
          f32_dma_group(from(q), from(q + 1), from(q + 2), from(q + 3), voff[q] - back, voff[q + 1] - back, voff[q + 2] - back, voff[q + 3] - back, to + q * 1024);
        if constexpr (LOADS % 4 == 2) f32_dma_group(from(LOADS - 2), from(LOADS - 1), voff[LOADS - 2] - back, voff[LOADS - 1] - back, to + (LOADS - 2) * 1024);
      };
      if (k0 + 32 <= K) groups(0);
      else groups(k0 + 4 * p < K ? 0 : 16 * p);  // pieces beyond K: the block's first one, zeroed in `work`
    };
#pragma unroll
    for (int s = 0; s < RING; ++s)
      if (s < blocks) stage(s, s);
    for (int s = 0, at = 0; s < blocks; ++s) {
      if (s + RING <= blocks) f32_wait<LOADS * (RING - 1)>(); else f32_wait<0>();
      const unsigned char* block = f32_lds + wave * BLOCK + at * 4 * BLOCK + r * 128;
      f32x4 fx[MI][2], fw[NI][2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int place = ((2 * g + h) ^ (r & 7)) * 16;
#pragma unroll
        for (int i = 0; i < MI; ++i) fx[i][h] = *reinterpret_cast<const f32x4*>(block + i * 2048 + place);
#pragma unroll
        for (int i = 0; i < NI; ++i) fw[i][h] = *reinterpret_cast<const f32x4*>(block + TM * 128 + i * 2048 + place);
      }
      f32_wait_lds();                            // the block is in registers: its place is free
      if (s + RING < blocks) stage(s + RING, at);
      work(first_k(s), fx, fw);
      at = at + 1 == RING ? 0 : at + 1;
    }
    __syncthreads();                             // all blocks have been read: LDS takes the sums
  }

  // What the parts cannot give (F32_SMALLEST): a bit for each of a thread's outputs that is formed again below.
  static_assert(TM * 4 <= 256 && NI <= 8, "four outputs of every sixteen features to a thread");
  uint32_t again = 0;
  f32x4 (*merge)[4][TM * 4] = reinterpret_cast<f32x4 (*)[4][TM * 4]>(f32_lds);
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
        bool odd = false;                        // (as whole numbers the sizes of floats have their order)
#pragma unroll
        for (int j = 0; j < 4; ++j) odd |= (f32_bits(v[j]) & 0x7fffffffu) - F32_SMALLEST >= 0x7f800000u - F32_SMALLEST;
        if (__builtin_expect(odd, 0)) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (f + j < N && v[j] != 0.f && !(fabsf(v[j]) >= __uint_as_float(F32_SMALLEST) && fabsf(v[j]) < INFINITY)) again |= 1u << (4 * n + j);
        }
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

  // These once more, 16 x 16 outputs at a time, on the float32 matrix instructions: blocks and chains as above, all by the wave that has
  // the outputs, a lane's 4 consecutive k of a row straight from memory. The others keep their bits. (300 rows of 151936 x 1024, one of which is
  // not a number, 0.51 -> 2.4 ms.)
#pragma unroll 1
  for (int n = 0; n < NI; ++n) {
    const uint32_t mine = again >> (4 * n) & 15u;
    if (__ballot(mine != 0) == 0) continue;
    const float *xr = x0 + (int64_t)min(16 * wave + r, M - 1 - m0) * ldx, *wr = w0 + (int64_t)min(16 * n + r, N - 1 - n0) * ldw;
    f32x4 chain[4] = {};
#pragma unroll 1
    for (int k0 = 4 * g; k0 - 4 * g < K; k0 += k0 & 16 ? 112 : 16)
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int k = k0 + 32 * c + j, at = min(k, K - 1);
          chain[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(k < K ? wr[at] : 0.f, k < K ? xr[at] : 0.f, chain[c], 0, 0, 0);
        }
    // a lane holds features 4 g .. 4 g + 3 of row r, and stored those of 4 (lane % 4) on of row lane / 4
    const f32x4 v = (chain[0] + chain[1]) + (chain[2] + chain[3]);
    const int from = (lane & 3) * 16 + (lane >> 2);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float o = __shfl(v[j], from);
      if (mine >> j & 1) y[(int64_t)(m0 + tid / 4) * ldy + n0 + 16 * n + (tid & 3) * 4 + j] = o;
    }
  }
}

extern "C" int me_gemm_f32(const float* x, int64_t ldx, const float* w, int64_t ldw, float* y, int64_t ldy, int M, int N, int K,
                           int tile_rows, int tile_features, hipStream_t stream) {
  if (M == 0 || N == 0) return 0;
  ME_CHECK(K >= 1 && ldx >= K && ldw >= K && ldy >= N, "gemm (float32): bad leading dimensions");
  ME_CHECK(K <= 2147483647 - 4096, "gemm (float32): rows of %d terms", K);
  const int64_t far = ldx > ldw ? ldx : ldw;          // a tile's rows lie within 4 GB of its first one
  const bool vec = K % 4 == 0 && ldx % 4 == 0 && ldw % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0 && far < (1 << 22);
  const int vec_out = ldy % 4 == 0 && (uintptr_t)y % 16 == 0;
#define F32_TILE(TM, TN, RING)                                                                                                                        \
  if (tile_rows == TM && tile_features == TN) {                                                                                                       \
    const int64_t mt = (M + TM - 1) / TM, nt = (N + TN - 1) / TN, rows = mt < F32_ROW_GROUP ? mt : F32_ROW_GROUP;                                     \
    const int64_t blocks = (mt + rows - 1) / rows * rows * ((nt + 7) / 8) * 8;                                                                        \
    ME_CHECK(blocks <= 2147483647ll, "gemm (float32): too many tiles for one launch");                                                                \
    constexpr int sums = 2 * 4 * TM * 4 * (int)sizeof(f32x4), ring = RING * 4 * (TM + TN) * 128, lds = ring > sums ? ring : sums;                     \
    static bool allowed = lds <= 65536;                /* more than a kernel may have unasked */                                                      \
    if (!allowed) {                                                                                                                                   \
      const hipError_t e = hipFuncSetAttribute((const void*)gemm_f32_kernel<TM, TN, RING>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);          \
      ME_CHECK(e == hipSuccess, "gemm (float32): cannot get %d bytes of LDS: %s", lds, hipGetErrorString(e));                                         \
      allowed = true;                                                                                                                                 \
    }                                                                                                                                                 \
    if (vec) gemm_f32_kernel<TM, TN, RING><<<(unsigned)blocks, 256, lds, stream>>>(x, ldx, w, ldw, y, ldy, M, N, K, (int)mt, (int)nt, vec_out);       \
    else gemm_f32_kernel<TM, TN, 0><<<(unsigned)blocks, 256, sums, stream>>>(x, ldx, w, ldw, y, ldy, M, N, K, (int)mt, (int)nt, vec_out);             \
    ME_LAUNCH_CHECK();                                                                                                                                \
    return 0;                                                                                                                                         \
  }
  F32_TILE(16, 16, 4)
  F32_TILE(16, 32, 3)
  F32_TILE(32, 32, 2)
  F32_TILE(32, 64, 1)
  F32_TILE(64, 32, 1)
  F32_TILE(64, 64, 1)
  F32_TILE(64, 128, 1)
#undef F32_TILE
  ME_CHECK(false, "gemm (float32): no tile of %d rows x %d features", tile_rows, tile_features);
}
