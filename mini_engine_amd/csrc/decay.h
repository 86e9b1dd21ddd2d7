// What the kernels of the recurrences share: those with a decay per state row (hybrid.hip walks token by token, decay_chunks.hip sixteen
// tokens at a time; the update rules stand in hybrid.hip), and by chunks those with one per head (linear_chunks.hip).
#pragma once
#include "common.h"

__device__ __forceinline__ float hy_sigmoid(float v) { return 1.0f / (1.0f + expf(-v)); }
__device__ __forceinline__ float hy_softplus(float v) { return v > 20.f ? v : log1pf(expf(v)); }

struct DrArgs {
  const void* q; const void* k; const void* v; const void* raw; const void* beta;
  int64_t q_stride, k_stride, v_stride, raw_stride, beta_stride;
  const float* base; const float* rate; const float* bonus;
  float* state; int64_t state_stride;
  const int32_t* slots; const int32_t* cu;
  float* y;
  int H, G, N, P;
  int unit; float unit_eps, q_scale;
};

// Sum over the RG neighbouring lanes that share a state column (RG 1, 4 or 16, aligned groups), left in all of them: lane
// exchanges inside a row of 16 lanes (quad permutations, then rotations of the row), no trip through LDS.
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int RG>
__device__ __forceinline__ float group_sum(float v) {
  if (RG >= 2) v += dpp_f<0xB1>(v);      // quad_perm [1, 0, 3, 2]
  if (RG >= 4) v += dpp_f<0x4E>(v);      // quad_perm [2, 3, 0, 1]
  if (RG >= 8) v += dpp_f<0x124>(v);     // row_ror 4
  if (RG >= 16) v += dpp_f<0x128>(v);    // row_ror 8
  return v;
}

// What a token's q, k, raw decay and write strength become before the recurrence reads them, for one wave that holds
// rows lane, lane + 64, ... of one head: q and k at unit length and scaled, the decay, and the token's own number
// (sigmoid(beta), or sum_n q_n bonus_n k_n under the bonus rule), which every lane gets.
// (RULE 3: every lane holds the head's one raw decay and its base in d[0], base[0] and gets the decay there.)
template <int PER, int RULE>
__device__ __forceinline__ float shape_token(const DrArgs& a, int lane, int nr_rows, float (&q)[PER], float (&k)[PER], float (&d)[PER],
                                             const float (&base)[PER], const float (&bonus)[PER], float rate, float beta) {
  float qs = a.q_scale, ks = 1.0f;
  if (a.unit) {
    float q2 = 0.f, k2 = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) { q2 += q[i] * q[i]; k2 += k[i] * k[i]; }
    qs = a.q_scale / sqrtf(wave_sum(q2) + a.unit_eps);
    ks = 1.0f / sqrtf(wave_sum(k2) + a.unit_eps);
  }
  float own = 0.f;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int n = lane + 64 * i;
    q[i] *= qs;
    k[i] *= ks;
    if (RULE == 3) continue;
    float dv;
    if (RULE == 0) dv = expf(-expf(d[i] + base[i]));
    else if (RULE == 2) dv = expf(-rate * hy_softplus(-(d[i] + base[i])));
    else dv = expf(-rate * hy_softplus(d[i] + base[i]));
    d[i] = (n < a.N && n < nr_rows) ? dv : 1.0f;
    own += q[i] * bonus[i] * k[i];
  }
  if (RULE == 3) d[0] = expf(-rate * hy_softplus(d[0] + base[0]));
  if (RULE == 2) return 0.f;
  return (RULE == 1 || RULE == 3) ? hy_sigmoid(beta) : wave_sum(own);
}

// ------------------------------------------------------------------ sixteen tokens at a time
#define DC_TOKENS 16

// Chunk i of request b has place cu[b] / 16 + b + i (whole division): the places of two requests never meet, there are at most T / 16 +
// B, and neither the host nor a scan over the requests is needed to give them out.
__device__ __forceinline__ int64_t chunk_place(const int32_t* cu, int b) { return cu[b] / DC_TOKENS + b; }

// The request that place belongs to: the last one whose first place is not behind it (-1: none).
__device__ __forceinline__ int chunk_request(const int32_t* cu, int num_seqs, int64_t place, int lane) {
  int b = -1;
  for (int b0 = 0; b0 < num_seqs; b0 += 64) {
    const bool in = b0 + lane < num_seqs && chunk_place(cu, min(b0 + lane, num_seqs - 1)) <= place;
    const int count = __popcll(__ballot(in));
    b += count;
    if (count < 64) break;
  }
  return __builtin_amdgcn_readfirstlane(b);
}

// acc + M X for 16 x 16 matrices, M zero above its diagonal. Of M a lane has numbers 4 g .. 4 g + 3 of row lane % 16 (g: its lane group),
// of X and acc rows 4 g .. 4 g + 3 of column lane % 16.
__device__ __forceinline__ f32x4 chunk_lower(const f32x4& M, const f32x4& X, f32x4 acc, int g) {
  // a zero times what is not a number would reach the rows in front of it: then row by row, later rows of X taken out
  float odd = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) odd = fmaf(X[e], 0.f, odd);
  if (__builtin_expect(__ballot(odd != 0.f) != 0, 0)) {
    f32x4 r = acc;
#pragma unroll 1
    for (int i = 0; i < DC_TOKENS; ++i) {
      f32x4 one = acc;
#pragma unroll
      for (int e = 0; e < 4; ++e) one = __builtin_amdgcn_mfma_f32_16x16x4f32(M[e], 4 * g + e <= i ? X[e] : 0.f, one, 0, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = 4 * g + e == i ? one[e] : r[e];
    }
    return r;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(M[e], X[e], acc, 0, 0, 0);
  return acc;
}
