// y[M, N] = x[M, K] . w[N, K]^T for prompts and other steps of many rows, bfloat16 operands, float32 sums (reference
// layers/linear.py:26,45: F.linear), optionally with the gating of a packed gate/up weight in the epilogue.
//
// A workgroup owns a tile of TM rows x TN features and walks K 64 at a time through two stages of LDS; the loads write LDS
// themselves (16 bytes a lane, 1 KB a wave's instruction = 8 rows of 128 bytes). The 16-byte piece c of row R lies at
// position c ^ (R >> 1 & 7), so that the 16 lanes of an operand read touch 16 different bank groups. The weight rows are
// the matrix instruction's A operand: a lane then holds 4 consecutive features of one row.
//
// A wave's share of a step is four quarters: half of its rows by half of its features, in the order (rows 0, features 0),
// (0, 1), (1, 1), (1, 0). A quarter brings in the operands it is the first to need (the features' first half a quarter
// early, so that the reads are spread evenly over the four), asks for one region of a later step (half of the tile's rows or
// features) as soon as the region it overwrites has been read by every wave, and waits only for what the next quarter reads:
// five of eight regions stay on their way at any time. With eight waves the two waves of a SIMD run half a quarter apart
// (the second four pass one barrier more at the start, the first four at the end): while one multiplies, the other reads.
// With four waves several workgroups share a compute unit and fill each other's waits.
//
// What bounds it: the matrix pipes at the clock that a full chip keeps for tiles of 256 x 256 (8,192 x 8,192 x 8,192: 1,554
// TFLOP/s, the library's kernel 1,307); the reads of LDS for the others, whose waves have fewer products for an operand read
// (256 x 128: 176 KB of LDS traffic a step at 128 bytes a cycle is 0.6 us, which is what a step takes; 128 x 128 96 KB, 0.33
// of 0.44 us). us, the library / this: 2,048 rows of 24576 x 4096 348 / 303 (with the gating 385 with a kernel
// behind it / 310), of 6144 x 4096 83 / 81, of 4096 x 4096 61 / 58, of 4096 x 12288 176 / 163, of 6144 x 1024 28.6 / 27.6 (with
// the gating 37.4 / 30.0), of 4096 x 1024 22.2 / 19.1; 512 rows of 4096 x 1024 10.9 / 9.0, of 6144 x 1024 with the gating 19.5 / 11.8.
// Sums that are rounded before the gating, with the library's exponential, cost a tile 1-3 us more than unrounded ones would
// (281 and 23.4): the bits stay those of the product and the gating kernel.
//
// Outputs in bfloat16 are written 16 bytes a lane, 64 contiguous bytes of a row by four lanes: within a wave's half of the
// features the weight rows are laid into LDS so that two matrix results of a lane are 8 consecutive features (8-byte stores
// in pieces of 32: 2,048 rows of 24576 x 4096 307 us). Tiles are dealt to the XCDs in contiguous runs of a grouped order
// (8 tiles of rows at a time), so that the tiles under way on one share operands in its L2.
#include "common.h"
#include <type_traits>

// gbase and lds_addr are the same in every lane; the first lane's values are taken so that they lie in scalar registers.
// The write to m0 needs one wait state before an instruction that reads it for an LDS address.
__device__ __forceinline__ void tile_dma16(const bf16_t* gbase, uint32_t voff, uint32_t lds_addr) {
  const uint64_t g = reinterpret_cast<uint64_t>(gbase);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(g >> 32)), lo = __builtin_amdgcn_readfirstlane((uint32_t)g);
  const uint64_t base = (uint64_t)hi << 32 | lo;
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voff), "s"(base) : "memory");
}
template <int N> __device__ __forceinline__ void tile_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ void tile_wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
// Nothing crosses it in either direction, matrix instructions included.
__device__ __forceinline__ void tile_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// The regions of a stage in the order in which they are asked for: features' first half, rows' first half, features' second,
// rows' second. Odd: rows; bit 1: the half.
enum { REGION_W0 = 0, REGION_X0 = 1, REGION_W1 = 2, REGION_X1 = 3 };
#define TILE_INT(v) std::integral_constant<int, v>{}

// Writes a wave's sums: its rows are m0 + 16 j of the lane, its features begin at n0 (ACT: its gated features).
template <int MI, int NI, bool ACT, typename TO>
__device__ __forceinline__ void tile_store(const f32x4 (&acc)[NI][MI], TO* __restrict__ out, int64_t ldy, int M, int N, int m0, int n0, int g,
                                           const GateForm& form, int rounded) {
  constexpr int NH = NI / 2;
  constexpr bool PAIRED = sizeof(TO) == 2;
  const int I = N / 2, F = ACT ? I : N;
#pragma unroll
  for (int j = 0; j < MI; ++j) {
    const int m = m0 + 16 * j;
    if (m >= M) continue;
    TO* row = out + (int64_t)m * ldy;
#pragma unroll
    for (int h = 0; h < (ACT ? 1 : 2); ++h) {
      const int f0 = ACT ? n0 : n0 + h * (8 * NI);
      auto value = [&](int i, int e, int f) {
        if constexpr (ACT) {
          float gate = acc[i][j][e], up = acc[NH + i][j][e];
          if (rounded) { gate = (float)(bf16_t)gate; up = (float)(bf16_t)up; }
          if (form.bias) { gate += form.bias[f]; up += form.bias[I + f]; }
          return rounded ? gate_value<false>(gate, up, form) : gate_value<true>(gate, up, form);
        } else {
          return acc[h * NH + i][j][e];
        }
      };
#pragma unroll
      for (int i = 0; i < NH; ++i) {
        if constexpr (!PAIRED) {
          const int f = f0 + 16 * i + 4 * g;
          if (f < F) *reinterpret_cast<f32x4*>(row + f) = acc[h * NH + i][j];
        } else if (i / 2 < NH / 2) {
          if (i & 1) continue;                                       // i and i + 1: 8 consecutive features (F is in eights)
          const int f = f0 + 16 * i + 8 * g;
          if (f < F) {
            bf16x8 r;
#pragma unroll
            for (int e = 0; e < 8; ++e) r[e] = (bf16_t)value(i + e / 4, e & 3, f + e);
            *reinterpret_cast<bf16x8*>(row + f) = r;
          }
        } else {
          const int f = f0 + 16 * i + 4 * g;
          if (f < F) {
            bf16x4 r;
#pragma unroll
            for (int e = 0; e < 4; ++e) r[e] = (bf16_t)value(i, e, f + e);
            *reinterpret_cast<bf16x4*>(row + f) = r;
          }
        }
      }
    }
  }
}

// WGM x WGN waves, each with MI tiles of 16 rows x NI tiles of 16 features (both even). ACT: w is a packed gate/up weight
// [2 I, K] (gate rows first, N = 2 I); the first half of a wave's features are gates, the second their ups, and what is
// written is their gated product [M, I] (reference layers/activation.py:5-7), formed from the unrounded sums as the other
// products with this epilogue form it, or with `rounded` from the sums rounded to bfloat16: the bits of the product and the
// gating kernel (csrc/elementwise.hip) behind it.
template <int WGM, int WGN, int MI, int NI, bool ACT, typename TO>
__global__ void __launch_bounds__(WGM* WGN * 64, 2)
gemm_tile_kernel(const bf16_t* __restrict__ x, int64_t ldx, const bf16_t* __restrict__ w, int64_t ldw, TO* __restrict__ y, int64_t ldy,
                 int M, int N, int steps_per_split, int all_steps, int m_tiles, int n_tiles, int group_m, GateForm form, int rounded) {
  extern __shared__ __align__(16) unsigned char tile_lds[];          // [2][STAGE]
  constexpr int NW = WGM * WGN, TM = WGM * MI * 16, TN = WGN * NI * 16, MH = MI / 2, NH = NI / 2;
  constexpr int STAGE = (TM + TN) * 128;
  constexpr bool PING = NW == 8, PAIRED = sizeof(TO) == 2;
  // a half of the rows (features) comes in XC (WC) pieces of 8 rows: each wave brings XD of them and, where they do not come
  // out even, half of the waves one more: the first half of the waves for the first half of the rows, the second for the second
  constexpr int XC = WGM * MI, WC = WGN * NI, XD = XC / NW, WD = WC / NW;
  constexpr bool XODD = XC % NW != 0, WODD = WC % NW != 0;
  static_assert(MI % 2 == 0 && NI % 2 == 0 && XC % (NW / 2) == 0 && WC % (NW / 2) == 0, "whole pieces for the waves");
  constexpr int XS = XD + XODD, WS = WD + WODD;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int late = wave / (NW / 2);                                  // the second half of the waves
  const int n = lane & 15, g = lane >> 4;
  const int tiles = m_tiles * n_tiles, per_xcd = (tiles + 7) >> 3;
  const int t = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (t >= tiles) return;
  const int group = t / (group_m * n_tiles), rest = t % (group_m * n_tiles);
  const int in_group = min(group_m, m_tiles - group * group_m);
  const int mt = group * group_m + rest % in_group, nt = rest / in_group;
  const int I = N / 2;                                               // ACT only
  const int m0 = mt * TM, n0 = nt * (ACT ? TN / 2 : TN);
  const int first = blockIdx.z * steps_per_split;
  const int steps = min(steps_per_split, all_steps - first);          // two or more (the launcher)

  // what a lane names in memory for each piece of its wave, and where the piece lies in a stage; rows beyond the matrix are
  // read from its last row and never stored
  uint32_t xoff[2][XS], woff[2][WS], xlds[2][XS], wlds[2][WS];
  const int r8 = lane >> 3, c8 = lane & 7;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int q = 0; q < XS; ++q) {
      const int piece = q < XD ? wave + NW * q : NW * XD + wave % (NW / 2);
      const int row0 = piece / MI * (16 * MI) + h * (8 * MI) + piece % MI * 8, R = row0 + r8;
      xoff[h][q] = (uint32_t)((int64_t)min(m0 + R, M - 1) * ldx * 2 + 16 * (c8 ^ ((R >> 1) & 7)));
      xlds[h][q] = row0 * 128;
    }
#pragma unroll
    for (int q = 0; q < WS; ++q) {
      const int piece = q < WD ? wave + NW * q : NW * WD + wave % (NW / 2);
      const int owner = piece / NI, r0 = piece % NI * 8, row0 = owner * (16 * NI) + h * (8 * NI) + r0, R = row0 + r8;
      int f = r0 + r8;                                               // the feature that row f of the half holds:
      if (PAIRED && (f >> 5) < NH / 2) f = (f & ~31) + 8 * ((f & 15) >> 2) + 4 * ((f >> 4) & 1) + (f & 3);
      const int64_t row = ACT ? (int64_t)h * I + min(n0 + owner * (8 * NI) + f, I - 1) : min(n0 + owner * (16 * NI) + h * (8 * NI) + f, N - 1);
      woff[h][q] = (uint32_t)(row * ldw * 2 + 16 * (c8 ^ ((R >> 1) & 7)));
      wlds[h][q] = (TM + row0) * 128;
    }
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)tile_lds;
  const bf16_t* xk = x + (int64_t)first * 64;
  const bf16_t* wk = w + (int64_t)first * 64;
  auto ask = [&](int k, auto region) {
    constexpr int R = decltype(region)::value, h = R >> 1;
    if constexpr (R & 1) {
#pragma unroll
      for (int q = 0; q < XS; ++q)
        if (q < XD || late == h) tile_dma16(xk + (int64_t)k * 64, xoff[h][q], lds0 + (k & 1) * STAGE + xlds[h][q]);
    } else {
#pragma unroll
      for (int q = 0; q < WS; ++q)
        if (q < WD || late == h) tile_dma16(wk + (int64_t)k * 64, woff[h][q], lds0 + (k & 1) * STAGE + wlds[h][q]);
    }
  };
  // waits until no more is on its way than the last `count` regions asked for, the oldest of them `oldest`
  auto wait = [&](auto oldest, auto count) {
    constexpr auto pieces = [](int second) {
      int sum = 0;
      for (int i = 0; i < decltype(count)::value; ++i) {
        const int R = (decltype(oldest)::value + i) & 3, h = R >> 1;
        sum += (R & 1) ? XD + (XODD && second == h) : WD + (WODD && second == h);
      }
      return sum;
    };
    if constexpr (pieces(0) == pieces(1)) tile_wait<pieces(0)>();
    else if (late) tile_wait<pieces(1)>();
    else tile_wait<pieces(0)>();
  };

  const int wm = wave / WGN, wn = wave % WGN, swizzle = (n >> 1) & 7;
  uint32_t rd_x[2], rd_w[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    rd_x[s] = (wm * (16 * MI) + n) * 128 + (((4 * s + g) ^ swizzle) * 16);
    rd_w[s] = (TM + wn * (16 * NI) + n) * 128 + (((4 * s + g) ^ swizzle) * 16);
  }
  f32x4 acc[NI][MI];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 fx[MH][2], fw[2][NH][2], ahead[NH][2];
  auto read_x = [&](int k, int h) {
    const unsigned char* buf = tile_lds + (k & 1) * STAGE;
#pragma unroll
    for (int j = 0; j < MH; ++j)
#pragma unroll
      for (int s = 0; s < 2; ++s) fx[j][s] = *reinterpret_cast<const bf16x8*>(buf + rd_x[s] + (h * MH + j) * 2048);
  };
  auto read_w = [&](int k, int h, bf16x8 (&into)[NH][2]) {
    const unsigned char* buf = tile_lds + (k & 1) * STAGE;
#pragma unroll
    for (int i = 0; i < NH; ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s) into[i][s] = *reinterpret_cast<const bf16x8*>(buf + rd_w[s] + (h * NH + i) * 2048);
  };
  auto multiply = [&](int hx, int hw) {
    if (PING) tile_barrier();
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < NH; ++i)
#pragma unroll
        for (int j = 0; j < MH; ++j)
          acc[hw * NH + i][hx * MH + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[hw][i][s], fx[j][s], acc[hw * NH + i][hx * MH + j], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
    tile_barrier();
  };
  // Why no wait is missing. A region is read in one quarter q by both halves of the waves; the half that runs late reads it
  // half a quarter after, and has it in registers before the barrier behind its products, which the other half passes at the
  // end of its reads of quarter q + 1. The request that overwrites the region is made in quarter q + 2. The features' first half, read
  // in quarter 3 (and in front of the first step) for the quarter behind, is waited for at the beginning of that quarter: a late wave
  // has it before the barrier in front of its products, which an early wave passes in front of its quarter 1, where the request is made.
  // It has had a quarter's products to arrive by then. (Four waves are never apart: there the products of quarter 0 wait in time.)
  // What quarter q reads has been waited for by the wave that asked for it in quarter q - 1 before a barrier that every reader has
  // passed.
  auto step = [&](int k, auto kind) {                                 // kind 0: two steps or more follow, 1: one, 2: none
    constexpr int KIND = decltype(kind)::value;
    if (PING) tile_wait_lds();
    read_x(k, 0);
    if constexpr (KIND < 2) { ask(k + 1, TILE_INT(REGION_X1)); wait(TILE_INT(REGION_X1), TILE_INT(5)); } else wait(TILE_INT(REGION_X1), TILE_INT(1));
    multiply(0, 0);
    read_w(k, 1, fw[1]);
    if constexpr (KIND == 0) { ask(k + 2, TILE_INT(REGION_W0)); wait(TILE_INT(REGION_W0), TILE_INT(5)); }
    else if constexpr (KIND == 1) wait(TILE_INT(REGION_W0), TILE_INT(4));
    else tile_wait<0>();
    multiply(0, 1);
    read_x(k, 1);
    if constexpr (KIND == 0) { ask(k + 2, TILE_INT(REGION_X0)); wait(TILE_INT(REGION_X0), TILE_INT(5)); }
    else if constexpr (KIND == 1) wait(TILE_INT(REGION_X0), TILE_INT(3));
    multiply(1, 1);
    if constexpr (KIND < 2) read_w(k + 1, 0, ahead);
    if constexpr (KIND == 0) { ask(k + 2, TILE_INT(REGION_W1)); wait(TILE_INT(REGION_W1), TILE_INT(5)); }
    else if constexpr (KIND == 1) wait(TILE_INT(REGION_W1), TILE_INT(2));
    multiply(1, 0);
    if constexpr (KIND < 2) {
#pragma unroll
      for (int i = 0; i < NH; ++i)
#pragma unroll
        for (int s = 0; s < 2; ++s) fw[0][i][s] = ahead[i][s];
    }
  };
  ask(0, TILE_INT(REGION_W0)); ask(0, TILE_INT(REGION_X0)); ask(0, TILE_INT(REGION_W1)); ask(0, TILE_INT(REGION_X1));
  ask(1, TILE_INT(REGION_W0)); ask(1, TILE_INT(REGION_X0)); ask(1, TILE_INT(REGION_W1));
  wait(TILE_INT(REGION_W1), TILE_INT(5));
  tile_barrier();
  read_w(0, 0, fw[0]);
  if (PING && late) tile_barrier();
  int k = 0;
  for (; k < steps - 2; ++k) step(k, TILE_INT(0));
  step(k, TILE_INT(1));
  step(k + 1, TILE_INT(2));
  if (PING && !late) tile_barrier();

  tile_store<MI, NI, ACT>(acc, y + (int64_t)blockIdx.z * M * ldy, ldy, M, N, m0 + wm * (16 * MI) + n, n0 + wn * (ACT ? 8 * NI : 16 * NI), g, form, rounded);
}

// The same by four waves for launches of one workgroup to a compute unit, which no other fills the waits of: whole steps of 64 of K in
// a ring of RING_STAGES, a barrier a step. A wave reads the next step's operands and asks for the step behind the ring between its
// products, so that neither stands in a row of its own: 16 products of 128 x 64 beside 12 reads and 6 requests take about what the requests take
// (24 KB a step at the 64 bytes a cycle that reach a compute unit; 2,048 rows of 1024 x 2048 with 4 / 5 / 6 stages 12.9 / 11.9 / 12.5 us). In quarters, with four barriers
// a step and the reads in front of the products, a step took 0.29-0.48 us whatever the tile; now 0.17 for 64 x 64, 0.31 for 64 x 128, 0.49 for 128 x
// 128. us of a launch in a chain, the library / quarters / this: 2,048 rows of 1024 x 2048 16.4 / 14.0 / 11.9, of 1024 x 3072 19.3 / 19.5 / 16.8,
// 700 rows 10.2 / 10.7 / 8.4 and 13.9 / 15.1 / 11.5, 800 rows of 4096 x 4096 39.9 / 38.9 / 32.9; the same bits (K in one order).
#define RING_STAGES 5
template <int WGM, int WGN, int MI, int NI, bool ACT, typename TO>
__global__ void __launch_bounds__(WGM* WGN * 64, 1)
gemm_ring_kernel(const bf16_t* __restrict__ x, int64_t ldx, const bf16_t* __restrict__ w, int64_t ldw, TO* __restrict__ y, int64_t ldy,
                 int M, int N, int steps_per_split, int all_steps, int m_tiles, int n_tiles, int group_m, GateForm form, int rounded) {
  extern __shared__ __align__(16) unsigned char tile_lds[];          // [ST][STAGE]
  constexpr int NW = WGM * WGN, TM = WGM * MI * 16, TN = WGN * NI * 16, NH = NI / 2, ST = RING_STAGES;
  constexpr int STAGE = (TM + TN) * 128;
  constexpr bool PAIRED = sizeof(TO) == 2;
  constexpr int XS = TM / 8 / NW, WS = TN / 8 / NW, PIECES = XS + WS;   // a wave's pieces of 8 rows of a stage: rows, then features
  static_assert(TM / 8 % NW == 0 && TN / 8 % NW == 0 && PIECES * (ST - 2) < 64, "whole pieces, and what the counter of loads can tell apart");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int tiles = m_tiles * n_tiles, per_xcd = (tiles + 7) >> 3;
  const int t = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per_xcd || t >= tiles) return;
  const int group = t / (group_m * n_tiles), rest = t % (group_m * n_tiles);
  const int in_group = min(group_m, m_tiles - group * group_m);
  const int mt = group * group_m + rest % in_group, nt = rest / in_group;
  const int I = N / 2;                                               // ACT only
  const int m0 = mt * TM, n0 = nt * (ACT ? TN / 2 : TN);
  const int first = blockIdx.z * steps_per_split;
  const int steps = min(steps_per_split, all_steps - first);          // one or more

  uint32_t off[PIECES];                                               // what a lane names in memory for each piece
  const int r8 = lane >> 3, c8 = lane & 7;
#pragma unroll
  for (int q = 0; q < XS; ++q) {
    const int R = 8 * (wave + NW * q) + r8;
    off[q] = (uint32_t)((int64_t)min(m0 + R, M - 1) * ldx * 2 + 16 * (c8 ^ ((R >> 1) & 7)));
  }
#pragma unroll
  for (int q = 0; q < WS; ++q) {
    const int R = 8 * (wave + NW * q) + r8, owner = R / (16 * NI), h = R % (16 * NI) / (8 * NI);
    int f = R % (8 * NI);                                             // laid out as in `gemm_tile_kernel`
    if (PAIRED && (f >> 5) < NH / 2) f = (f & ~31) + 8 * ((f & 15) >> 2) + 4 * ((f >> 4) & 1) + (f & 3);
    const int64_t row = ACT ? (int64_t)h * I + min(n0 + owner * (8 * NI) + f, I - 1) : min(n0 + owner * (16 * NI) + h * (8 * NI) + f, N - 1);
    off[XS + q] = (uint32_t)(row * ldw * 2 + 16 * (c8 ^ ((R >> 1) & 7)));
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)tile_lds + 1024 * wave;
  const bf16_t* xa = x + (int64_t)first * 64;                         // of the step that is asked for next
  const bf16_t* wa = w + (int64_t)first * 64;
  auto ask_piece = [&](uint32_t slot, int q) {
    if (q < XS) tile_dma16(xa, off[q], lds0 + slot + NW * q * 1024);
    else tile_dma16(wa, off[q], lds0 + slot + TM * 128 + NW * (q - XS) * 1024);
  };
  const int wm = wave / WGN, wn = wave % WGN, swizzle = (n >> 1) & 7;
  uint32_t rd_x[2], rd_w[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    rd_x[s] = (wm * (16 * MI) + n) * 128 + (((4 * s + g) ^ swizzle) * 16);
    rd_w[s] = (TM + wn * (16 * NI) + n) * 128 + (((4 * s + g) ^ swizzle) * 16);
  }
  struct Operands { bf16x8 x[MI][2], w[NI][2]; } one, two;
  constexpr int READS = 2 * (NI + MI), PRODUCTS = 2 * NI * MI;
  auto read_one = [&](uint32_t slot, Operands& o, int r) {            // in the order of use
    const int s = r / (NI + MI), q = r % (NI + MI);
    if (q < NI) o.w[q][s] = *reinterpret_cast<const bf16x8*>(tile_lds + slot + rd_w[s] + q * 2048);
    else o.x[q - NI][s] = *reinterpret_cast<const bf16x8*>(tile_lds + slot + rd_x[s] + (q - NI) * 2048);
  };
  f32x4 acc[NI][MI];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto next_slot = [&](uint32_t s) { return s == (ST - 1) * STAGE ? 0u : s + STAGE; };

  const int early = min(ST - 1, steps);
#pragma unroll
  for (int s = 0; s < ST - 1; ++s)
    if (s < early) {
#pragma unroll
      for (int q = 0; q < PIECES; ++q) ask_piece(s * STAGE, q);
      xa += 64; wa += 64;
    }
  // waits until no more than the last `count` steps asked for are on their way
  auto wait = [&](int count) {
    if (count <= 0) tile_wait<0>();
    else if (count == 1) tile_wait<PIECES>();
    else if (count == 2) tile_wait<2 * PIECES>();
    else tile_wait<3 * PIECES>();
  };
  static_assert(ST - 2 == 3, "`wait` knows up to three steps");
  wait(early - 1);
  tile_barrier();
#pragma unroll
  for (int r = 0; r < READS; ++r) read_one(0, one, r);
  // The first operands are there before the loop, where the compiler then counts the reads of LDS alone and waits for as many as it needs.
  __builtin_amdgcn_s_waitcnt(0xC07F);                                 // lgkmcnt(0)
  uint32_t slot = 0, free_slot = (ST - 1) * STAGE;                    // where step k is; where step k + ST - 1 goes, which held step k - 1
  int k = 0;
  // Why no wait is missing: step k + 1 has been waited for by every wave that asked for part of it before the barrier of step k, behind
  // which it is read. A wave passes that barrier with its products of step k - 1 behind it, so with its reads of that step done: the
  // requests of step k overwrite what nobody reads any more.
  auto step = [&](const Operands& cur, Operands& nxt, auto asks, auto more) {
    uint32_t s1 = 0;
    if constexpr (decltype(more)::value) { tile_barrier(); s1 = next_slot(slot); }
#pragma unroll
    for (int c = 0; c < PRODUCTS; ++c) {
      const int s = c / (NI * MI), i = c / MI % NI, j = c % MI;
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cur.w[i][s], cur.x[j][s], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (decltype(more)::value) {
#pragma unroll
        for (int r = c * READS / PRODUCTS; r < (c + 1) * READS / PRODUCTS; ++r) read_one(s1, nxt, r);
      }
      if constexpr (decltype(asks)::value) {
#pragma unroll
        for (int q = c * PIECES / PRODUCTS; q < (c + 1) * PIECES / PRODUCTS; ++q) ask_piece(free_slot, q);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (decltype(asks)::value) { xa += 64; wa += 64; }
    if constexpr (decltype(more)::value) { free_slot = slot; slot = s1; }
    ++k;
  };
  const std::true_type yes;
  const std::false_type no;
  auto steady = [&](const Operands& cur, Operands& nxt) { tile_wait<PIECES * (ST - 3)>(); step(cur, nxt, yes, yes); };
  auto ending = [&](const Operands& cur, Operands& nxt) {             // near the end: what is left decides
    if (k + 1 < steps) {
      wait(min(ST - 3, steps - 2 - k));
      if (k + ST - 1 < steps) step(cur, nxt, yes, yes); else step(cur, nxt, no, yes);
    } else {
      step(cur, nxt, no, no);
    }
  };
  while (k + ST < steps) { steady(one, two); steady(two, one); }
  while (k < steps) {
    ending(one, two);
    if (k < steps) ending(two, one);
  }
  tile_store<MI, NI, ACT>(acc, y + (int64_t)blockIdx.z * M * ldy, ldy, M, N, m0 + wm * (16 * MI) + n, n0 + wn * (ACT ? 8 * NI : 16 * NI), g, form, rounded);
}

// Whether a launch of so many tiles (times slices of K), each of `per_split` steps, goes through the ring: tiles of four waves where there is at
// most a workgroup to a compute unit. Below 16 steps the quarters are level or ahead (8 steps a slice, 128 rows of 1024 x 2048 in tiles of 128 x
// 64 6.3 / 6.7 us). Tiles of 128 x 128, whose ring fills a compute unit's LDS, gain from 32 steps on and up to 248 workgroups (16 steps 12.3 /
// 16.5 with 256 of them, 32 steps 20.2 / 23.2, with 208 19.5 / 18.5).
extern "C" int me_gemm_tile_rings(int tile_rows, int tile_features, int64_t tiles, int per_split) {
  const bool large = tile_rows == 128 && tile_features == 128;
  return tile_rows * tile_features <= 128 * 128 && tile_rows <= 128 && tile_features <= 128 && tiles <= (large ? 248 : 256) && per_split >= (large ? 32 : 16);
}

// y: [M, N] of out_dtype (ksplit 1), or float32 partial sums [ksplit, M, N] with ldy = N; act: w is a packed gate/up weight
// [N = 2 I, K] and y is the gated product [M, I] (bfloat16, ksplit 1) in the form that limit, alpha and bias give (`GateForm`);
// 1: of the unrounded sums, 2: of the sums rounded to bfloat16.
// tile_rows x tile_features: one of the tiles below (the result's sums do not depend on it).
extern "C" int me_gemm_tile_bf16(const void* x, int64_t ldx, const void* w, int64_t ldw, void* y, int64_t ldy, int out_dtype, int ksplit,
                                 int M, int N, int K, int act, float limit, float alpha, const float* bias, int tile_rows, int tile_features,
                                 hipStream_t stream) {
  if (M == 0 || N == 0) return 0;
  ME_CHECK(M > 0 && N > 0 && (out_dtype == ME_BF16 || out_dtype == ME_F32), "tile gemm: %d x %d, output dtype %d", M, N, out_dtype);
  ME_CHECK(act >= 0 && act <= 2, "tile gemm: no gating %d", act);
  ME_CHECK(act || (limit == 0.f && bias == nullptr), "tile gemm: limits and biases belong to the gating epilogue");
  ME_CHECK(K >= 128 && K % 64 == 0, "tile gemm: K=%d must be two steps of 64 or more", K);
  ME_CHECK(N % (act ? 16 : 8) == 0 && ldy % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0, "tile gemm: N=%d and the row strides must keep 16-byte pieces whole", N);
  ME_CHECK(ldx >= K && ldw >= K && ldy >= (act ? N / 2 : N), "tile gemm: a row stride is shorter than its row");
  ME_CHECK((uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0 && (uintptr_t)y % 16 == 0, "tile gemm: operands must be 16-byte aligned");
  ME_CHECK((int64_t)M * ldx * 2 < (1ll << 32) && (int64_t)N * ldw * 2 < (1ll << 32), "tile gemm: an operand beyond 4 GB");
  ME_CHECK(ksplit >= 1 && (ksplit == 1 || out_dtype == ME_F32), "tile gemm: %d slices: partial sums are float32", ksplit);
  ME_CHECK(!act || (ksplit == 1 && out_dtype == ME_BF16), "tile gemm: the gating wants one bfloat16 result");
  const int steps = K / 64, per_split = (steps + ksplit - 1) / ksplit;
  ME_CHECK((int64_t)(ksplit - 1) * per_split <= steps - 2, "tile gemm: %d slices leave one of %d steps with fewer than two", ksplit, steps);
  const GateForm form{limit, alpha, bias};
#define TILE_LAUNCH(KERNEL, WGM, WGN, MI, NI, ACT, TO)                                                                               \
  do {                                                                                                                               \
    auto kernel = KERNEL<WGM, WGN, MI, NI, ACT, TO>;                                                                                 \
    if (lds > 65536) {                                         /* more than a kernel may have unasked */                             \
      static bool allowed = false;                                                                                                   \
      if (!allowed) {                                                                                                                \
        const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);         \
        ME_CHECK(e == hipSuccess, "tile gemm: cannot get %zu bytes of LDS: %s", lds, hipGetErrorString(e));                          \
        allowed = true;                                                                                                              \
      }                                                                                                                              \
    }                                                                                                                                \
    kernel<<<grid, WGM * WGN * 64, lds, stream>>>((const bf16_t*)x, ldx, (const bf16_t*)w, ldw, (TO*)y, ldy, M, N, per_split, steps, \
                                                  (int)m_tiles, (int)n_tiles, (int)(m_tiles < 8 ? m_tiles : 8), form, act == 2);               \
  } while (0)
#define TILE_KIND(KERNEL, WGM, WGN, MI, NI)                                                                           \
  do {                                                                                                                \
    if (act) TILE_LAUNCH(KERNEL, WGM, WGN, MI, NI, true, bf16_t);                                                     \
    else if (out_dtype == ME_F32) TILE_LAUNCH(KERNEL, WGM, WGN, MI, NI, false, float);                                \
    else TILE_LAUNCH(KERNEL, WGM, WGN, MI, NI, false, bf16_t);                                                        \
  } while (0)
// RING: whether the tile has a form that goes through the ring.
#define TILE(WGM, WGN, MI, NI, RING)                                                                                  \
  if (tile_rows == WGM * MI * 16 && tile_features == WGN * NI * 16) {                                                 \
    const int64_t m_tiles = ((int64_t)M + tile_rows - 1) / tile_rows;                                                 \
    const int64_t n_tiles = act ? ((int64_t)N / 2 + tile_features / 2 - 1) / (tile_features / 2) : ((int64_t)N + tile_features - 1) / tile_features; \
    const int64_t blocks = (m_tiles * n_tiles + 7) / 8 * 8;                                                           \
    ME_CHECK(blocks < (1ll << 31) && 8 * n_tiles < (1ll << 31) && ksplit <= 65535, "tile gemm: too many tiles");      \
    const dim3 grid((unsigned)blocks, 1, (unsigned)ksplit);                                                           \
    if constexpr (RING)                                                                                               \
      if (me_gemm_tile_rings(tile_rows, tile_features, m_tiles * n_tiles * ksplit, per_split)) {                      \
        const size_t lds = (size_t)(tile_rows + tile_features) * 128 * RING_STAGES;                                   \
        TILE_KIND(gemm_ring_kernel, WGM, WGN, MI, NI);                                                                \
        ME_LAUNCH_CHECK();                                                                                            \
        return 0;                                                                                                     \
      }                                                                                                               \
    const size_t lds = (size_t)(tile_rows + tile_features) * 256;                                                     \
    TILE_KIND(gemm_tile_kernel, WGM, WGN, MI, NI);                                                                    \
    ME_LAUNCH_CHECK();                                                                                                \
    return 0;                                                                                                         \
  }
  TILE(2, 4, 8, 4, false)     // 256 x 256
  TILE(4, 2, 4, 6, false)     // 256 x 192
  TILE(2, 4, 6, 4, false)     // 192 x 256
  TILE(2, 4, 4, 4, false)     // 128 x 256
  TILE(4, 2, 4, 4, false)     // 256 x 128
  TILE(4, 2, 2, 6, false)     // 128 x 192
  TILE(2, 2, 4, 4, true)     // 128 x 128
  TILE(2, 2, 2, 4, true)     // 64 x 128
  TILE(2, 2, 4, 2, true)     // 128 x 64
  TILE(2, 2, 2, 2, true)     // 64 x 64
#undef TILE
#undef TILE_KIND
#undef TILE_LAUNCH
  ME_CHECK(false, "tile gemm: no tile of %d rows x %d features", tile_rows, tile_features);
}
