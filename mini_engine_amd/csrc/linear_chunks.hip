// The recurrence S_t = a_t S_(t-1) + b_t k_t v_t^T, y_t = S_t^T q_t (+ skip v_t) with one decay per head and token (recurrent.hip) sixteen
// tokens at a time, for long requests in bfloat16: with S the state in front of a chunk and c_i = a_1 ... a_i,
//   y_i = c_i S^T q_i + sum_{j <= i} (q_i . k_j) F_ij v_j + skip v_i,      F_ij = (a_{j+1} ... a_i) b_j
//   S <- c_16 S + sum_j k_j ((a_{j+1} ... a_16) b_j v_j)^T
// as products on the float32 matrix instructions. The decays are numbers per token here, so q, k and q . k are the same for all heads of
// a group. A first kernel lays out q, k and their products per chunk and group, decays and v per chunk and head; a second walks a
// request's chunks. Every product of decays is formed as such (an exponential of a sum, or a power of a
// fixed decay), none by a division. us, four tokens at a time in spans side by side (recurrent.hip) / so, both kernels: 8 requests of up to
// 350 tokens, 16 heads of 128 x 128, fixed decays, 161 / 51, 32 heads of 128 x 64 over shared keys with step sizes 146 / 46; one of 2,048
// tokens 168 / 98, 153 / 91; 16 of 700 685 / 320, 591 / 224. Error against 64 bits (700 tokens, relative to the norm of y): fixed decays of
// 0.97 to 0.9999 1.1e-6 / 1.7e-7, step sizes 1.3e-7 / 1.0e-7.
#include "chunks.h"
#include <type_traits>

struct LinArgs {
  const void* q; const void* k; const void* v; const void* dt;
  int64_t q_stride, k_stride, v_stride, dt_stride;
  const float* decay;                                        // [H], or null: step sizes
  const float* dt_bias; const float* rate; const float* skip;
  float* state; int64_t state_stride;
  const int32_t* slots; const int32_t* cu;
  float* y;
  int H, G, N, P, silu, num_seqs, col_blocks;
  int64_t from, upto;                                        // the places that scratch holds now (me_linear_chunks)
};

// Floats of a chunk: of a group q [tokens, rows], k [rows, tokens] and their products; of a head F, c, (a_{j+1} ... a_16) b_j, c_16 (with
// what fills 16 numbers) and v.
__host__ __device__ constexpr int linear_group_floats(int rows) { return 32 * rows + 256; }
__host__ __device__ constexpr int64_t linear_head_floats(int col_blocks) { return 304 + (int64_t)256 * col_blocks; }

__device__ __forceinline__ float lin_silu(float v) { return v * (1.0f / (1.0f + expf(-v))); }

// One workgroup per place and group (the first G of the grid's second side) or head. What bounds it: a trip to memory for its rows and
// the store of what it makes of them.
template <typename TX, int NR>
__global__ void __launch_bounds__(256)
linear_chunk_kernel(LinArgs a, float* __restrict__ group_chunks, float* __restrict__ head_chunks) {
  constexpr int C = DC_TOKENS, ROW = NR + 4;                 // (rows of LDS four numbers apart in banks)
  __shared__ __align__(16) float sq[C][ROW], sk[C][ROW];
  __shared__ float sl[C], sb[C];
  const int tid = threadIdx.x, lane = tid & 63;
  const int64_t slot = blockIdx.x, place = a.from + slot;
  const int b = chunk_request(a.cu, a.num_seqs, place, lane);
  if (b < 0) return;
  const int begin = a.cu[b], at = (int)(place - chunk_place(a.cu, b)) * C, n_tok = min(C, a.cu[b + 1] - begin - at);
  if (n_tok <= 0) return;
  const int64_t first = (int64_t)begin + at;
  const int i = tid >> 4, j = tid & 15;

  if ((int)blockIdx.y < a.G) {
    const int g = blockIdx.y;
    const TX* qp = (const TX*)a.q + (int64_t)g * a.N; const TX* kp = (const TX*)a.k + (int64_t)g * a.N;
    TX q[NR / 16], k[NR / 16];
#pragma unroll
    for (int e = 0; e < NR / 16; ++e) {                      // NR threads to a token
      const int token = (tid + 256 * e) / NR, n = min((tid + 256 * e) % NR, a.N - 1);
      const int64_t row = first + min(token, n_tok - 1);
      q[e] = qp[row * a.q_stride + n];
      k[e] = kp[row * a.k_stride + n];
    }
#pragma unroll
    for (int e = 0; e < NR / 16; ++e) {
      const int token = (tid + 256 * e) / NR, n = (tid + 256 * e) % NR;
      const bool in = token < n_tok && n < a.N;
      float qv = to_f32<TX>(q[e]), kv = to_f32<TX>(k[e]);
      if (a.silu) { qv = lin_silu(qv); kv = lin_silu(kv); }
      sq[token][n] = in ? qv : 0.f;
      sk[token][n] = in ? kv : 0.f;
    }
    __syncthreads();
    f32x4 dot = {0.f, 0.f, 0.f, 0.f};                        // q_i . k_j in four sums
#pragma unroll 8
    for (int n = 0; n < NR; n += 4) {
      const f32x4 qi = *reinterpret_cast<const f32x4*>(&sq[i][n]), kj = *reinterpret_cast<const f32x4*>(&sk[j][n]);
#pragma unroll
      for (int e = 0; e < 4; ++e) dot[e] = fmaf(qi[e], kj[e], dot[e]);
    }
    float* out = group_chunks + (slot * a.G + g) * (int64_t)linear_group_floats(NR);
    out[32 * NR + (j >> 2) * 64 + i * 4 + (j & 3)] = (dot[0] + dot[1]) + (dot[2] + dot[3]);
    for (int e = tid; e < C * NR / 4; e += 256) {
      const int tile = e >> 6, four = e >> 4 & 3, low = e & 15;
      *reinterpret_cast<f32x4*>(out + e * 4) = *reinterpret_cast<const f32x4*>(&sq[low][16 * tile + 4 * four]);
      f32x4 w;
#pragma unroll
      for (int t = 0; t < 4; ++t) w[t] = sk[4 * four + t][16 * tile + low];
      *reinterpret_cast<f32x4*>(out + C * NR + e * 4) = w;
    }
    return;
  }

  const int h = blockIdx.y - a.G;
  float* out = head_chunks + (slot * a.H + h) * linear_head_floats(a.col_blocks);
  // token j's -log of the decay and its factor b
  if (tid < C) {
    float l = 0.f, f = j < n_tok ? 1.f : 0.f;
    if (a.dt && j < n_tok) {
      const float z = to_f32<TX>(((const TX*)a.dt)[(first + j) * a.dt_stride + h]) + a.dt_bias[h];
      f = z > 20.f ? z : log1pf(expf(z));
      l = a.rate[h] * f;
    }
    sl[j] = l;
    sb[j] = f;
  }
  for (int e = tid; e < 64 * a.col_blocks; e += 256) {       // [16 columns][4 tokens][column]; columns beyond the last are copies of it
    const int column = min(e >> 6 << 4 | (e & 15), a.P - 1);
    f32x4 v;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int token = (e >> 4 & 3) * 4 + t;
      float x = to_f32<TX>(((const TX*)a.v)[(first + min(token, n_tok - 1)) * a.v_stride + (int64_t)h * a.P + column]);
      if (a.silu) x = lin_silu(x);
      v[t] = token < n_tok ? x : 0.f;
    }
    *reinterpret_cast<f32x4*>(out + 304 + e * 4) = v;
  }
  __syncthreads();
  // the product of the decays behind token `from` (-1: all of the chunk's) up to token `to`; tokens that are not there have none
  auto over = [&](int from, int to) {
    if (a.decay) {
      double p = 1.0;                                        // a power rounded once
      const double d = a.decay[h];
      for (int m = from; m < min(to, n_tok - 1); ++m) p *= d;
      return (float)p;
    }
    float sum = 0.f;
    for (int m = from + 1; m <= to; ++m) sum += sl[m];
    return expf(-sum);
  };
  out[(j >> 2) * 64 + i * 4 + (j & 3)] = j <= i ? over(j, i) * sb[j] : 0.f;
  if (i == 0) out[256 + j] = over(-1, j);
  if (i == 1) out[272 + j] = over(j, C - 1) * sb[j];
  if (i == 2) out[288 + j] = over(-1, C - 1);
}

// One workgroup per request, head and 16 columns; its waves share the state's rows, RT tiles of 16 each. A lane holds rows 4 g .. 4 g + 3
// (g: its lane group) of a column of each tile, which is what a matrix instruction leaves in it and what the next one wants as its
// operand, so neither the state nor what is added to it ever moves between lanes; products are formed in instructions of four k each. Only
// outputs need the sum over all rows: they come after four chunks, a quarter a wave (in every chunk, one wave's output made all
// wait: 64 rows 0.57 -> 0.35 us a chunk). Operands are asked for two chunks ahead (four: no faster, and short requests half as slow
// again for their registers). What bounds it: 16 matrix instructions of 32 cycles a chunk and wave with 128 rows where the chip is full, else
// the chain through them, 0.65 us a chunk.
template <typename TX, int NR, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, 2)       // up to 256 registers, of which matrix instructions then use the ordinary ones: no copies
linear_chunk_walk_kernel(LinArgs a, const float* __restrict__ group_chunks, const float* __restrict__ head_chunks, int groups) {
  constexpr int C = DC_TOKENS, RT = NR / (16 * WAVES);
  __shared__ f32x4 part_y[2][4][WAVES][64];
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the column blocks of one request and head, which read the same operands, run on one XCD
  const int slot = blockIdx.x >> 3, group = slot / a.col_blocks * 8 + (blockIdx.x & 7), cb = slot % a.col_blocks;
  if (group >= groups) return;
  const int b = group / a.H, h = group % a.H;
  // of the request the chunks whose places scratch holds; the state waits in its row between two walks
  const int all_begin = __builtin_amdgcn_readfirstlane(a.cu[b]), all_tok = __builtin_amdgcn_readfirstlane(a.cu[b + 1]) - all_begin;
  const int all_place = __builtin_amdgcn_readfirstlane((int)chunk_place(a.cu, b));
  const int first = max((int)a.from - all_place, 0), count = min((all_tok + C - 1) / C, (int)a.upto - all_place) - first;
  if (all_tok <= 0 || count <= 0) return;
  const int begin = all_begin + C * first, n_tok = min(all_tok - C * first, C * count);
  const int p = cb * 16 + col, pc = min(p, a.P - 1);
  const bool live = p < a.P;
  float* srow = a.state + (int64_t)a.slots[b] * a.state_stride + (int64_t)h * a.N * a.P;
  const int row0 = wave * RT * 16 + 4 * g;
  f32x4 S[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int n = row0 + 16 * t + e;
      S[t][e] = n < a.N ? srow[(int64_t)n * a.P + pc] : 0.f;
    }
  const float skip = a.skip ? a.skip[h] : 0.f;
  const int64_t place = all_place + first - (int)a.from;
  const int64_t group_pace = (int64_t)a.G * linear_group_floats(NR), head_pace = a.H * linear_head_floats(a.col_blocks);
  const float* of_group = group_chunks + place * group_pace + (int64_t)(h / (a.H / a.G)) * linear_group_floats(NR);
  const float* of_head = head_chunks + place * head_pace + h * linear_head_floats(a.col_blocks);
  float* out = a.y + (int64_t)begin * (a.H * a.P) + (int64_t)h * a.P + pc;

  const uint32_t lane16 = lane * 16, tokens16 = g * 16;
  auto at = [](const float* from, uint32_t bytes) { return *reinterpret_cast<const f32x4*>(reinterpret_cast<const char*>(from) + bytes); };
  struct Chunk { f32x4 q[RT], w[RT], dots, F, c, e, end, v; };
  auto fetch = [&](int i, Chunk& o) {
    const float* from = of_group + min(i, count - 1) * group_pace;
    const float* head = of_head + min(i, count - 1) * head_pace;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      o.q[t] = at(from + (wave * RT + t) * 256, lane16);
      o.w[t] = at(from + C * NR + (wave * RT + t) * 256, lane16);
    }
    o.dots = at(from + 32 * NR, lane16);
    o.F = at(head, lane16);
    o.c = at(head + 256, tokens16);
    o.e = at(head + 272, tokens16);
    o.end = at(head + 288, 0);
    o.v = at(head + 304 + cb * 256, lane16);
    asm volatile("" ::: "memory");
  };
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  // Code of each wave's own, and for whole chunks no branch around a load or a store: the wait for a chunk's operands then counts
  // what was asked for behind them; behind a branch it would be for everything. (A lane behind the last column has that column's
  // numbers and stores them again.)
  Chunk o[2];
  fetch(0, o[0]);
  fetch(1, o[1]);
  int i0 = 0;
  auto four = [&](auto which, auto all) {
    constexpr int ME = decltype(which)::value;
    constexpr bool WHOLE = decltype(all)::value;
    f32x4(*sums)[WAVES][64] = part_y[i0 >> 2 & 1];
    f32x4 A[4 / WAVES], c[4 / WAVES], v[4 / WAVES];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      if (WHOLE || i0 + d < count) {
        Chunk& k = o[d & 1];
        f32x4 r[RT];
#pragma unroll
        for (int t = 0; t < RT; ++t) r[t] = zero;
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int t = 0; t < RT; ++t) r[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k.q[t][e], S[t][e], r[t], 0, 0, 0);
        const f32x4 u = k.v * k.e;
#pragma unroll
        for (int t = 0; t < RT; ++t) S[t] *= k.end[0];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int t = 0; t < RT; ++t) S[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k.w[t][e], u[e], S[t], 0, 0, 0);
#pragma unroll
        for (int t = 1; t < RT; ++t) r[0] += r[t];
        sums[d][wave][lane] = r[0];
        if (d % WAVES == ME) {
#pragma unroll
          for (int e = 0; e < 4; ++e) A[d / WAVES][e] = 4 * g + e <= col ? k.dots[e] * k.F[e] : 0.f;
          c[d / WAVES] = k.c;
          v[d / WAVES] = k.v;
        }
        fetch(i0 + d + 2, k);
      }
    }
    __syncthreads();                                         // (nobody is two rounds ahead, so the sums read below are still there)
#pragma unroll
    for (int d = ME; d < 4; d += WAVES) {
      if (WHOLE || i0 + d < count) {
        f32x4 y = sums[d][0][lane] + sums[d][1][lane];
        if constexpr (WAVES == 4) y += sums[d][2][lane] + sums[d][3][lane];
        y = chunk_lower(A[d / WAVES], v[d / WAVES], y * c[d / WAVES], g);
        float* to = out + (int64_t)(C * (i0 + d)) * (a.H * a.P);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (WHOLE || C * (i0 + d) + 4 * g + e < n_tok) to[(4 * g + e) * (a.H * a.P)] = a.skip ? fmaf(skip, v[d / WAVES][e], y[e]) : y[e];
      }
    }
    i0 += 4;
  };
  auto walk = [&](auto which) {
    while (i0 + 4 <= n_tok / C) four(which, std::true_type{});
    if (i0 < count) four(which, std::false_type{});
  };
  static_assert(WAVES == 2 || WAVES == 4, "each wave's walk is code of its own");
  if (wave == 0) walk(std::integral_constant<int, 0>{});
  else if (wave == 1) walk(std::integral_constant<int, 1>{});
  else if (wave == 2) walk(std::integral_constant<int, 2 % WAVES>{});
  else walk(std::integral_constant<int, 3 % WAVES>{});
  if (live) {
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int n = row0 + 16 * t + e;
        if (n < a.N) srow[(int64_t)n * a.P + p] = S[t][e];
      }
  }
}

// chunks: scratch of `room` floats; a place takes G linear_group_floats + H linear_head_floats of them, for N rounded up to 32, 64 or 128.
// There are T / 16 + num_seqs places; those that scratch does not hold at once are laid out and walked one part behind the other, with
// the same bits.
extern "C" int me_linear_chunks(const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v, int64_t v_stride,
                                const void* dt, int64_t dt_stride, const float* decay, const float* dt_bias, const float* rate, const float* skip,
                                float* state, int64_t state_stride, const int32_t* slots, const int32_t* cu, float* y, int num_seqs, int H,
                                int G, int N, int P, int silu, int64_t T, float* chunks, int64_t room, hipStream_t stream) {
  if (num_seqs == 0 || T == 0) return 0;
  ME_CHECK(H >= 1 && G >= 1 && H % G == 0 && N >= 1 && N <= 128 && P >= 1 && P <= (1 << 28), "linear_chunks: %d heads over %d groups, state %d x %d "
           "(up to 128 rows)", H, G, N, P);
  ME_CHECK((dt != nullptr) != (decay != nullptr) && (dt == nullptr || (dt_bias && rate)), "linear_chunks: fixed decays, or step sizes with bias and rates");
  const int64_t places = T / DC_TOKENS + num_seqs, groups = (int64_t)num_seqs * H;
  const int col_blocks = (P + 15) / 16, NR = N <= 32 ? 32 : N <= 64 ? 64 : 128;
  const int64_t group_floats = (int64_t)G * linear_group_floats(NR), head_floats = H * linear_head_floats(col_blocks);
  const int64_t held = room / (group_floats + head_floats), part = held < places ? held : places;
  ME_CHECK(places <= 2147483647ll && (int64_t)H + G <= 65535 && (groups + 7) / 8 * 8 * col_blocks <= 2147483647ll, "linear_chunks: too many tokens, heads or columns");
  ME_CHECK(chunks != nullptr && (uintptr_t)chunks % 16 == 0 && part >= 1, "linear_chunks: scratch too small");
  LinArgs a;
  a.q = q; a.k = k; a.v = v; a.dt = dt; a.q_stride = q_stride; a.k_stride = k_stride; a.v_stride = v_stride; a.dt_stride = dt_stride;
  a.decay = decay; a.dt_bias = dt_bias; a.rate = rate; a.skip = skip; a.state = state; a.state_stride = state_stride; a.slots = slots; a.cu = cu;
  a.y = y; a.H = H; a.G = G; a.N = N; a.P = P; a.silu = silu; a.num_seqs = num_seqs; a.col_blocks = col_blocks;
  const unsigned wgrid = (unsigned)((groups + 7) / 8 * 8 * col_blocks);
#define LC(NR)                                                                                                                        \
  do {                                                                                                                                \
    constexpr int WAVES = NR >= 64 ? 4 : 2;                                                                                           \
    linear_chunk_kernel<bf16_t, NR><<<dim3((unsigned)(a.upto - a.from), H + G), 256, 0, stream>>>(a, chunks, heads);                  \
    linear_chunk_walk_kernel<bf16_t, NR, WAVES><<<wgrid, 64 * WAVES, 0, stream>>>(a, chunks, heads, (int)groups);                     \
  } while (0)
  float* heads = chunks + part * group_floats;
  for (a.from = 0; a.from < places; a.from = a.upto) {
    a.upto = a.from + part < places ? a.from + part : places;
    if (NR == 32) LC(32); else if (NR == 64) LC(64); else LC(128);
    ME_LAUNCH_CHECK();
  }
#undef LC
  return 0;
}
