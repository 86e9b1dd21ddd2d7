// Sixteen tokens of a recurrence at a time: where a request's chunks lie, and the product of two 16 x 16 matrices of which one has
// nothing above its diagonal (linear_chunks.hip).
#pragma once
#include "common.h"

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
