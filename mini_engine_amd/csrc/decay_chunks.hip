// The recurrence with a decay per state row (hybrid.hip) sixteen tokens at a time, for long requests in bfloat16: what a chunk of
// tokens does to the state is written as products, and they run on the float32 matrix instructions. With S the state in front
// of a chunk, d_i a token's decays, c_i = d_1 ... d_i (row by row) and b_i its write strength:
//   y_i = S^T (c_i q_i) + sum_{j <= i} A_ij u_j,      A_ij = sum_n q_i k_j (d_{j+1} ... d_i)
//   u_i = v_i, or under the delta rules b_i (v_i - S^T (c_i k_i) - sum_{j < i} B_ij u_j),   B_ij = sum_n k_i k_j (d_{j+1} ... d_i),
//         i.e. U = T (V - K~ S) with T = (1 + diag(b) B)^-1 diag(b)
//   S <- c_16 S + sum_j (d_{j+1} ... d_16 k_j) u_j^T
// (bonus rule: y reads the state in front of the token, so c_{i-1}, j < i, one decay less, and A_ii = sum_n q_i bonus k_i). Every
// product of decays is formed as such, none by a division, so none is larger than 1 and one that is zero does no harm.
// A first kernel forms, for every chunk and head at once, what does not depend on the state (decay_chunk_kernel); a second
// walks a request's chunks (decay_chunk_walk_kernel). us, token by token / so, both kernels of each: 2,048 tokens beside 1,075, delta
// rule, 4 heads of 128 x 128 269 / 146, bonus rule, 16 heads of 64 x 64 151 / 79; 16 prompts of 512 tokens over the former 267 / 102,
// 13 over the latter 160 / 85; 9 prompts of 2,048, one decay per head, 8 heads of 128 x 128 702 / 496; four of 512, gated rule, 4
// heads of 128 x 256 105 / 45. Error against 64 bits (1,500 tokens, relative to the norm of y): delta 3.2e-7 / 2.0e-7, gated 1.7 / 1.4,
// one decay per head 2.2 / 1.9, bonus 1.18 / 1.17: a decay over many tokens is rounded once here, not once a token.
#include "decay.h"
#include <type_traits>

// Floats that a chunk of one head takes: c q [tokens, rows], what it writes (K^) [rows, tokens], c_16, A; delta rules: c k, T; and v.
__host__ __device__ constexpr int chunk_fixed(int rows, bool delta) { return (delta ? 49 : 33) * rows + (delta ? 512 : 256); }
__host__ __device__ constexpr int64_t chunk_floats(int rows, bool delta, int col_blocks) { return chunk_fixed(rows, delta) + (int64_t)256 * col_blocks; }

// One workgroup per (place, head). All of it is laid out as the walk's lanes take it as operands: 16 bytes a lane, a wave's 1 KB in
// one piece. What bounds it: instructions, about half of them those that form A and B (a thread has one token j and every sixteenth
// group of four rows, and goes through the tokens behind j), the rest the decays' exponentials; a lone chunk takes 14 us. (3,123 tokens, delta
// rule, 4 heads of 128 rows 31 us, bonus rule, 16 heads of 64 rows 28; with all of a phase's loads brought forward by the compiler into
// 390 registers, or spilled, 95 and 30.)
template <typename TX, int NR, int RULE>
__global__ void __launch_bounds__(256, 4)
decay_chunk_kernel(DrArgs a, int num_seqs, int col_blocks, float* __restrict__ chunks) {
  constexpr bool DELTA = RULE == 1 || RULE == 3;
  constexpr int PER = (NR + 63) / 64, C = DC_TOKENS;
  __shared__ __align__(16) float sq[C][NR], sk[C][NR], sd[C][NR], sl[C][NR];      // sl: -log of the decays
  __shared__ __align__(16) float sA[C][C], sB[C][C], sT[C][C], sx[C];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t place = blockIdx.x;
  const int h = blockIdx.y, g = h / (a.H / a.G);
  const int b = chunk_request(a.cu, num_seqs, place, lane);
  if (b < 0) return;
  const int begin = a.cu[b], at = (int)(place - chunk_place(a.cu, b)) * C, n_tok = min(C, a.cu[b + 1] - begin - at);
  if (n_tok <= 0) return;
  const int64_t first = (int64_t)begin + at;

  {
    const TX* qp = (const TX*)a.q; const TX* kp = (const TX*)a.k; const TX* rp = (const TX*)a.raw; const TX* bp = (const TX*)a.beta;
    float base[PER], bonus[PER];
    float q[C / 4][PER], k[C / 4][PER], d[C / 4][PER], beta[C / 4];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int n = lane + 64 * i;
      const bool in = n < a.N && n < NR;
      base[i] = RULE == 3 ? a.base[h] : (in ? a.base[h * a.N + n] : 0.f);
      bonus[i] = (RULE == 0 && in) ? a.bonus[h * a.N + n] : 0.f;
    }
#pragma unroll
    for (int t = 0; t < C / 4; ++t) {                        // tokens wave, wave + 4, ...; those behind the last are read from it
      const int64_t row = first + min(wave + 4 * t, n_tok - 1);
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int n = lane + 64 * i;
        const bool in = n < a.N && n < NR;
        q[t][i] = in ? to_f32<TX>(qp[row * a.q_stride + g * a.N + n]) : 0.f;
        k[t][i] = in ? to_f32<TX>(kp[row * a.k_stride + g * a.N + n]) : 0.f;
        if (RULE == 3) d[t][i] = to_f32<TX>(rp[row * a.raw_stride + h]);
        else d[t][i] = in ? to_f32<TX>(rp[row * a.raw_stride + h * a.N + n]) : 0.f;
      }
      beta[t] = DELTA ? to_f32<TX>(bp[row * a.beta_stride + h]) : 0.f;
    }
    const float rate = RULE != 0 ? a.rate[h] : 0.f;
#pragma unroll
    for (int t = 0; t < C / 4; ++t) {
      const int token = wave + 4 * t;
      const bool on = token < n_tok;                         // a token that is not there: keys, queries and strength 0, decays 1
      __builtin_amdgcn_sched_barrier(0);                     // one token after the other: four at once take 250 registers
      float qs = a.q_scale, ks = 1.0f;
      if (a.unit) {
        float q2 = 0.f, k2 = 0.f;
#pragma unroll
        for (int i = 0; i < PER; ++i) { q2 += q[t][i] * q[t][i]; k2 += k[t][i] * k[t][i]; }
        qs = a.q_scale / sqrtf(wave_sum(q2) + a.unit_eps);
        ks = 1.0f / sqrtf(wave_sum(k2) + a.unit_eps);
      }
      float own = 0.f;                                       // bonus rule: sum_n q_n bonus_n k_n
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int n = lane + 64 * i;
        const float qv = q[t][i] * qs, kv = k[t][i] * ks, z = d[t][RULE == 3 ? 0 : i] + base[i];
        const float log = !on || n >= a.N ? 0.f : RULE == 0 ? expf(z) : rate * hy_softplus(RULE == 2 ? -z : z);
        own += qv * bonus[i] * kv;
        if (n < NR) {
          sq[token][n] = on ? qv : 0.f;
          sk[token][n] = on ? kv : 0.f;
          sd[token][n] = expf(-log);
          sl[token][n] = log;
        }
      }
      const float x = DELTA ? hy_sigmoid(beta[t]) : RULE == 0 ? wave_sum(own) : 0.f;
      if (lane == 0) sx[token] = on ? x : 0.f;
    }
  }
  __syncthreads();

  {
    const int j = tid >> 4, s = tid & 15;
    f32x4 r[PER], kj[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int n = 64 * u + 4 * s;
      r[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      kj[u] = NR % 64 == 0 || n < NR ? *reinterpret_cast<const f32x4*>(&sk[j][n]) : r[u];
    }
#pragma unroll 2                                             // (unrolled, all of its loads would come first)
    for (int i = 0; i < C; ++i) {
      float A = 0.f, B = 0.f;
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int n = NR % 64 == 0 ? 64 * u + 4 * s : min(4 * s, NR - 4);
        const f32x4 di = *reinterpret_cast<const f32x4*>(&sd[i][n]), qi = *reinterpret_cast<const f32x4*>(&sq[i][n]);
        f32x4 ki = {0.f, 0.f, 0.f, 0.f};
        if (DELTA) ki = *reinterpret_cast<const f32x4*>(&sk[i][n]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float next = i == j ? kj[u][e] : r[u][e] * di[e];
          A = fmaf(qi[e], RULE == 0 ? r[u][e] : next, A);    // bonus rule: the state in front of token i
          if (DELTA) B = fmaf(ki[e], next, B);
          r[u][e] = next;
        }
      }
      A = group_sum<16>(A);
      if (DELTA) B = group_sum<16>(B);
      if (s == 0) {
        sA[i][j] = i > j || (RULE != 0 && i == j) ? A : (RULE == 0 && i == j ? sx[i] : 0.f);
        if (DELTA) sB[j][i] = i > j ? B : 0.f;               // by columns
      }
    }
  }
  __syncthreads();

  if (DELTA && wave == 0) {
    // T by forward substitution: a lane has rows 4 g .. 4 g + 3 of a column of what is left of the right side
    const int j = lane & 15, g4 = lane >> 4;
    f32x4 left;
#pragma unroll
    for (int e = 0; e < 4; ++e) left[e] = 4 * g4 + e == j ? 1.f : 0.f;
#pragma unroll 1
    for (int m4 = 0; m4 < 4; ++m4) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = 4 * m4 + e;
        const float t = m < j ? 0.f : sx[m] * __shfl(left[e], m4 * 16 + j, ME_WAVE);
        const f32x4 Bm = *reinterpret_cast<const f32x4*>(&sB[m][4 * g4]);
#pragma unroll
        for (int r = 0; r < 4; ++r) left[r] = fmaf(-Bm[r], t, left[r]);
        if (g4 == m4) sT[m][j] = t;
      }
    }
  }
  float* out = chunks + (place * a.H + h) * chunk_floats(NR, DELTA, col_blocks);
  float* out_k = out + C * NR;
  float* out_c = out + 2 * C * NR;
  float* out_a = out_c + NR;
  // Row n, four tokens: the decays up to a token and behind it, as one exponential of a sum each (rounded once; a product of sixteen
  // decays would be as often as it has factors). Under the delta rules the first wave has T to do.
  for (int item = tid - (DELTA ? 64 : 0); item < 4 * NR; item += DELTA ? 192 : 256) {
    if (DELTA && wave == 0) break;
    const int n = item % NR, t4 = item / NR * 4;
    float before = 0.f, behind = 0.f, log[4], w[4];
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const float l = sl[i][n];
      if (i < t4) before += l;
      if (i > t4 + 3) behind += l;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) log[i] = sl[t4 + i][n];
#pragma unroll
    for (int i = 3; i >= 0; --i) {
      w[i] = sk[t4 + i][n] * expf(-behind);
      behind += log[i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (RULE == 0) sq[t4 + i][n] *= expf(-before);
      before += log[i];
      if (RULE != 0) {
        const float c = expf(-before);
        sq[t4 + i][n] *= c;
        if (DELTA) sk[t4 + i][n] *= c;
      }
    }
    if (t4 == C - 4) out_c[n] = expf(-before);
    *reinterpret_cast<f32x4*>(out_k + n / 16 * 256 + t4 * 16 + n % 16 * 4) = f32x4{w[0], w[1], w[2], w[3]};
  }
  __syncthreads();
  for (int e = tid; e < C * NR / 4; e += 256) {              // [16 rows][4 rows][token]
    const int tile = e >> 6, four = e >> 4 & 3, token = e & 15;
    *reinterpret_cast<f32x4*>(out + e * 4) = *reinterpret_cast<const f32x4*>(&sq[token][16 * tile + 4 * four]);
    if (DELTA) *reinterpret_cast<f32x4*>(out_a + 256 + e * 4) = *reinterpret_cast<const f32x4*>(&sk[token][16 * tile + 4 * four]);
  }
  float* out_v = out + chunk_fixed(NR, DELTA);               // [16 columns][4 tokens][column]; columns beyond the last are copies of it
  for (int e = tid; e < 64 * col_blocks; e += 256) {
    const int column = min(e >> 6 << 4 | (e & 15), a.P - 1);
    f32x4 v;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int token = (e >> 4 & 3) * 4 + t;
      const float at_token = to_f32<TX>(((const TX*)a.v)[(first + min(token, n_tok - 1)) * a.v_stride + (int64_t)h * a.P + column]);
      v[t] = token < n_tok ? at_token : 0.f;
    }
    *reinterpret_cast<f32x4*>(out_v + e * 4) = v;
  }
  if (tid < 64) {
    *reinterpret_cast<f32x4*>(out_a + tid * 4) = *reinterpret_cast<const f32x4*>(&sA[tid & 15][tid >> 4 << 2]);
    if (DELTA) *reinterpret_cast<f32x4*>(out_a + 256 + C * NR + tid * 4) = *reinterpret_cast<const f32x4*>(&sT[tid & 15][tid >> 4 << 2]);
  }
}

// One workgroup per request, head and 16 columns; its waves share the state's rows, RT tiles of 16 each. A lane holds rows 4 g .. 4 g + 3
// (g: its lane group) of a column of each tile, which is what a matrix instruction leaves in it and what the next one wants as its
// operand, so neither the state nor U ever moves between lanes. Products are formed in four instructions of four k each. Under the
// delta rules U needs the sum over all rows, so a chunk is two halves with a barrier between them; otherwise only y does. Outputs
// come after four chunks, a quarter a wave: in every chunk, one wave's output made all wait (bonus rule, 64 rows, 0.57 -> 0.35 us a chunk). Operands
// are asked for two chunks ahead (four: no faster, and short requests half as slow again for their registers).
// What bounds it: the chain of a chunk through one wave, which has its SIMD to itself: under the delta rules with 128 rows 28 matrix
// instructions of 32 cycles, about 110 others, the sums' way through LDS and a barrier, 0.85 us, where a token of the walk
// by tokens takes 0.12.
template <typename TX, int NR, int RULE, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, 2)       // up to 256 registers, of which matrix instructions then use the ordinary ones: no copies
decay_chunk_walk_kernel(DrArgs a, const float* __restrict__ chunks, int groups, int col_blocks) {
  constexpr bool DELTA = RULE == 1 || RULE == 3;
  constexpr int C = DC_TOKENS, RT = NR / (16 * WAVES), FIXED = chunk_fixed(NR, DELTA);
  __shared__ f32x4 part_y[DELTA ? 1 : 2][4][WAVES][64], part_u[2][DELTA ? WAVES : 1][64];
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the column blocks of one request and head, which read the same operands, run on one XCD
  const int slot = blockIdx.x >> 3, group = slot / col_blocks * 8 + (blockIdx.x & 7), cb = slot % col_blocks;
  if (group >= groups) return;
  const int b = group / a.H, h = group % a.H;
  const int begin = __builtin_amdgcn_readfirstlane(a.cu[b]), n_tok = __builtin_amdgcn_readfirstlane(a.cu[b + 1]) - begin;
  if (n_tok <= 0) return;
  const int count = (n_tok + C - 1) / C;
  const int p = cb * 16 + col, pc = min(p, a.P - 1);
  const bool live = p < a.P;
  float* srow = a.state + (int64_t)a.slots[b] * a.state_stride + (int64_t)h * a.N * a.P;
  const int row0 = wave * RT * 16 + 4 * g;                   // of tile 0's first row in this lane
  f32x4 S[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int n = row0 + 16 * t + e;
      S[t][e] = n < a.N ? srow[(int64_t)n * a.P + pc] : 0.f;
    }
  const int64_t floats = chunk_floats(NR, DELTA, col_blocks);
  const float* mine = chunks + ((int64_t)__builtin_amdgcn_readfirstlane((int)chunk_place(a.cu, b)) * a.H + h) * floats;
  float* out = a.y + (int64_t)begin * (a.H * a.P) + (int64_t)h * a.P + pc;

  // where a lane's operands lie in a chunk, in bytes: the rest of an address is the same for all lanes
  const uint32_t lane16 = lane * 16, rows16 = g * 16;
  auto at = [](const float* from, uint32_t bytes) { return *reinterpret_cast<const f32x4*>(reinterpret_cast<const char*>(from) + bytes); };
  struct Chunk { f32x4 q[RT], k[DELTA ? RT : 1], w[RT], c[RT], A, T, v; };
  const int64_t pace = a.H * floats;
  auto fetch = [&](int i, Chunk& o) {
    const float* from = mine + min(i, count - 1) * pace;
    const float* own = from + wave * RT * 256;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      if (DELTA) o.k[t] = at(own + 33 * NR + 256 + t * 256, lane16);
      o.q[t] = at(own + t * 256, lane16);
      o.w[t] = at(own + C * NR + t * 256, lane16);
      o.c[t] = at(from + 2 * C * NR + (wave * RT + t) * 16, rows16);
    }
    o.A = at(from + 33 * NR, lane16);
    if (DELTA) o.T = at(from + 49 * NR + 256, lane16);
    o.v = at(from + FIXED + cb * 256, lane16);
    asm volatile("" ::: "memory");
  };
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  // this wave's rows of M^T S, [tokens, columns]
  auto read_state = [&](const f32x4* M) {
    f32x4 r[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) r[t] = zero;
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int t = 0; t < RT; ++t) r[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(M[t][e], S[t][e], r[t], 0, 0, 0);
#pragma unroll
    for (int t = 1; t < RT; ++t) r[0] += r[t];
    return r[0];
  };
  auto sum_of = [&](const f32x4 (*part)[64]) {
    if constexpr (WAVES == 4) return (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
    else return part[0][lane] + part[1][lane];
  };
  // Four chunks one after the other, then their outputs, 4 / WAVES of them a wave's: with code of each wave's own, and for whole chunks
  // no branch around a load or a store: the wait for a chunk's operands then counts what was asked for behind them; behind a
  // branch it would be for everything. (A lane behind the last column has that column's numbers and stores them again.)
  Chunk o[2];
  fetch(0, o[0]);
  fetch(1, o[1]);
  int i0 = 0;
  auto four = [&](auto which, auto all) {
    constexpr int ME = decltype(which)::value;
    constexpr bool WHOLE = decltype(all)::value;
    f32x4(*sums)[WAVES][64] = part_y[DELTA ? 0 : i0 >> 2 & 1];     // (delta rules: nobody writes before all have passed a barrier behind the last outputs)
    f32x4 A[4 / WAVES], U[4 / WAVES];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      if (WHOLE || i0 + d < count) {
        Chunk& c = o[d & 1];
        f32x4 u = c.v, read;
        if (DELTA) {
          part_u[d & 1][wave][lane] = read_state(c.k);
          __syncthreads();                                   // the other buffer's sums have been read by all when this is passed again
          u -= sum_of(part_u[d & 1]);
          read = read_state(c.q);
          u = chunk_lower(c.T, u, zero, g);
        } else {
          read = read_state(c.q);
        }
        sums[d][wave][lane] = read;
#pragma unroll
        for (int t = 0; t < RT; ++t) S[t] *= c.c[t];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int t = 0; t < RT; ++t) S[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(c.w[t][e], u[e], S[t], 0, 0, 0);
        if (d % WAVES == ME) {
          A[d / WAVES] = c.A;
          U[d / WAVES] = u;
        }
        fetch(i0 + d + 2, c);
      }
    }
    __syncthreads();
#pragma unroll
    for (int d = ME; d < 4; d += WAVES) {
      if (WHOLE || i0 + d < count) {
        const f32x4 y = chunk_lower(A[d / WAVES], U[d / WAVES], sum_of(sums[d]), g);
        float* to = out + (int64_t)(C * (i0 + d)) * (a.H * a.P);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (WHOLE || C * (i0 + d) + 4 * g + e < n_tok) to[(4 * g + e) * (a.H * a.P)] = y[e];
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

// chunks: scratch of (T / 16 + num_seqs) H chunk_floats floats, for N rounded up to 32, 64 or 128; `room`: how many it has.
extern "C" int me_decay_rows_chunks(const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v, int64_t v_stride,
                                    const void* raw, int64_t raw_stride, const void* beta, int64_t beta_stride,
                                    const float* base, const float* rate, const float* bonus, float* state, int64_t state_stride,
                                    const int32_t* slots, const int32_t* cu, float* y, int num_seqs, int H, int G, int N, int P,
                                    int rule, int unit, float unit_eps, float q_scale, int64_t T, float* chunks, int64_t room, hipStream_t stream) {
  if (num_seqs == 0 || T == 0) return 0;
  ME_CHECK(H >= 1 && G >= 1 && H % G == 0 && N >= 1 && N <= 128 && P >= 1 && P <= (1 << 28), "decay_rows_chunks: %d heads over %d groups, state %d x %d "
           "(up to 128 rows)", H, G, N, P);
  ME_CHECK(rule >= 0 && rule <= 3, "decay_rows_chunks: unknown rule %d", rule);
  ME_CHECK(rule == 0 ? bonus != nullptr : (rate != nullptr && (rule == 2 || beta != nullptr)), "decay_rows_chunks: the rule's constants are missing");
  const int64_t places = T / DC_TOKENS + num_seqs, groups = (int64_t)num_seqs * H;
  const int col_blocks = (P + 15) / 16;
  const bool delta = rule == 1 || rule == 3;
  const int NR = N <= 32 ? 32 : N <= 64 ? 64 : 128;
  ME_CHECK(places <= 2147483647ll && H <= 65535 && (groups + 7) / 8 * 8 * col_blocks <= 2147483647ll, "decay_rows_chunks: too many tokens, heads or columns");
  ME_CHECK(chunks != nullptr && (uintptr_t)chunks % 16 == 0 && room >= places * H * chunk_floats(NR, delta, col_blocks), "decay_rows_chunks: scratch too small");
  DrArgs a;
  a.q = q; a.k = k; a.v = v; a.raw = raw; a.beta = beta;
  a.q_stride = q_stride; a.k_stride = k_stride; a.v_stride = v_stride; a.raw_stride = raw_stride; a.beta_stride = beta_stride;
  a.base = base; a.rate = rate; a.bonus = bonus; a.state = state; a.state_stride = state_stride; a.slots = slots; a.cu = cu; a.y = y;
  a.H = H; a.G = G; a.N = N; a.P = P; a.unit = unit; a.unit_eps = unit_eps; a.q_scale = q_scale;
  const dim3 pgrid((unsigned)places, H);
  const unsigned wgrid = (unsigned)((groups + 7) / 8 * 8 * col_blocks);
#define DC(NR, R)                                                                                                                    \
  do {                                                                                                                               \
    constexpr int WAVES = NR >= 64 ? 4 : 2;                                                                                          \
    decay_chunk_kernel<bf16_t, NR, R><<<pgrid, 256, 0, stream>>>(a, num_seqs, col_blocks, chunks);                                   \
    decay_chunk_walk_kernel<bf16_t, NR, R, WAVES><<<wgrid, 64 * WAVES, 0, stream>>>(a, chunks, (int)groups, col_blocks);             \
  } while (0)
#define DC_RULES(NR) do { if (rule == 0) DC(NR, 0); else if (rule == 1) DC(NR, 1); else if (rule == 2) DC(NR, 2); else DC(NR, 3); } while (0)
  if (NR == 32) DC_RULES(32); else if (NR == 64) DC_RULES(64); else DC_RULES(128);
#undef DC_RULES
#undef DC
  ME_LAUNCH_CHECK();
  return 0;
}
