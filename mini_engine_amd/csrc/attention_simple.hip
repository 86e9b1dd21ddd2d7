// Paged causal attention, the exact and slow form: one workgroup per (query token, head),
// scalar float32 arithmetic throughout. It takes any head size, page size and head grouping; the float32 path's
// usual sizes run on the float32 matrix instructions instead (attn_f32 below).
//
// Formulas as in the reference's pure-torch paged path (layers/attention.py:21-40): key j of
// the request is kept iff j <= position of the query (and j < context length); scores are
// scale * q.k; softmax over kept keys; output = sum p_j v_j. A window w additionally keeps
// only j > position - w (not in the reference). Three further options: `keep_first` n keeps the keys j < n visible
// behind a window; `softcap` c > 0 bends every score to c * tanh(score / c) before the softmax; `sinks` (one float per
// query head) adds exp(sink) to the softmax's denominator, a term without key or value. `slopes` (one float per query
// head) takes slope * (position - j) off the score of key j, behind the cap.
//
// Keys are processed in chunks whose boundaries are multiples of the chunk size counted from
// position 0 of the request, so the order of every sum for a given token is the same however
// the request was cut into steps or batched.
#include "common.h"

#define AS_THREADS 256
#define AS_CHANNELS 4

template <typename T>
__global__ void __launch_bounds__(AS_THREADS)
attn_simple_kernel(const T* __restrict__ q, int64_t q_stride, T* __restrict__ out, int64_t out_stride,
                   const T* __restrict__ k_cache, const T* __restrict__ v_cache,
                   const int32_t* __restrict__ block_tables, int bt_stride,
                   const int32_t* __restrict__ seq_of_token, const int32_t* __restrict__ positions,
                   const int32_t* __restrict__ context_lens, int Hq, int Hkv, int D, int page, float scale,
                   int window, int keep_first, float softcap, const float* __restrict__ sinks,
                   const float* __restrict__ slopes) {
  extern __shared__ float lds[];
  float* qs = lds;                 // D
  float* sc = lds + D;             // AS_THREADS scores / probabilities
  __shared__ float red[16];

  const int64_t t = blockIdx.x;
  const int h = blockIdx.y;
  const int kvh = h / (Hq / Hkv);
  const int b = seq_of_token[t];
  const int pos = positions[t];
  const int32_t* bt = block_tables + (int64_t)b * bt_stride;
  const int tid = threadIdx.x;

  for (int d = tid; d < D; d += AS_THREADS) qs[d] = to_f32<T>(q[t * q_stride + (int64_t)h * D + d]);
  __syncthreads();

  // keys [lo, hi): up to the query's own position, never past the request's context (a padding
  // row has context 0 and sees nothing)
  const int hi = min(pos + 1, context_lens[b]);
  // window > 0: the last `window` keys; window < 0: a block mask, only the keys of the query's own block of -window positions
  const int lo = window > 0 ? max(0, pos - window + 1) : (window < 0 ? pos - pos % (-window) : 0);
  // behind a window the first keep_first keys stay visible: the chunks walk [0, kept) and then [lo, hi)
  const int kept = (window > 0 && keep_first > 0) ? min(min(keep_first, lo), hi) : 0;
  float m = -INFINITY, l = 0.f;
  // a thread owns the output channels tid, tid + AS_THREADS, ...
  float acc[AS_CHANNELS];
#pragma unroll
  for (int dd = 0; dd < AS_CHANNELS; ++dd) acc[dd] = 0.f;
  const float slope = slopes != nullptr ? slopes[h] : 0.f;

  const int first_c0 = (lo / AS_THREADS) * AS_THREADS;
  for (int c0 = kept > 0 ? 0 : first_c0; c0 < hi; c0 += AS_THREADS) {
    if (c0 >= kept && c0 < first_c0) { c0 = first_c0 - AS_THREADS; continue; }   // nothing visible between the kept keys and the window
    const int j = c0 + tid;
    float s = -INFINITY;
    bool keep = (j >= lo || j < kept) && j < hi;
    if (keep) {
      const int64_t pg = bt[j / page];
      keep = pg >= 0;                        // a page that is not held is never dereferenced
      if (keep) {
        const int off = j % page;
        const T* kr = k_cache + ((pg * Hkv + kvh) * (int64_t)page + off) * D;
        float dot = 0.f;
        for (int d = 0; d < D; ++d) dot += qs[d] * to_f32<T>(kr[d]);
        s = dot * scale;
        if (softcap > 0.f) s = softcap * tanhf(s / softcap);
        s -= slope * (float)(pos - j);
      }
    }
    // chunk max
    float cm = wave_max(s);
    __syncthreads();
    if ((tid & 63) == 0) red[tid >> 6] = cm;
    __syncthreads();
    cm = red[0];
    for (int w = 1; w < AS_THREADS / 64; ++w) cm = fmaxf(cm, red[w]);
    const float m_new = fmaxf(m, cm);
    const float p = (keep && m_new > -INFINITY) ? expf(s - m_new) : 0.f;
    sc[tid] = p;
    float ps = wave_sum(p);
    __syncthreads();
    if ((tid & 63) == 0) red[8 + (tid >> 6)] = ps;
    __syncthreads();
    ps = 0.f;
    for (int w = 0; w < AS_THREADS / 64; ++w) ps += red[8 + w];
    const float alpha = (m == -INFINITY) ? 0.f : expf(m - m_new);   // m finite implies m_new finite
    l = l * alpha + ps;
    m = m_new;
    const int jb = kept > 0 ? c0 : max(c0, lo), je = min(c0 + AS_THREADS, hi);
#pragma unroll
    for (int dd = 0; dd < AS_CHANNELS; ++dd) {
      const int d = tid + dd * AS_THREADS;
      if (d < D) {
        float a = 0.f;
        for (int jj = jb; jj < je; ++jj) {
          if (jj < lo && jj >= kept) continue;   // its probability is 0 and its page may have been given back
          const int64_t pg = bt[jj / page];
          if (pg < 0) continue;                // its probability is 0
          const int off = jj % page;
          a += sc[jj - c0] * to_f32<T>(v_cache[((pg * Hkv + kvh) * (int64_t)D + d) * page + off]);
        }
        acc[dd] = acc[dd] * alpha + a;
      }
    }
    __syncthreads();
  }
  if (sinks != nullptr) {
    // the sink joins the denominator under the same running maximum; alone (no visible key) it leaves an output of zero
    const float sk = sinks[h];
    const float m_new = fmaxf(m, sk);
    const float alpha = (m == -INFINITY) ? 0.f : expf(m - m_new);
    l = l * alpha + expf(sk - m_new);
#pragma unroll
    for (int dd = 0; dd < AS_CHANNELS; ++dd) acc[dd] *= alpha;
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
  for (int dd = 0; dd < AS_CHANNELS; ++dd)
    if (tid + dd * AS_THREADS < D) out[t * out_stride + (int64_t)h * D + tid + dd * AS_THREADS] = from_f32<T>(acc[dd] * inv);
}

// ------------------------------------------------------------------ the same on the float32 matrix instructions
// Head sizes up to 128 in steps of 16, pages in steps of 4 keys: products on v_mfma_f32_16x16x4_f32 (float32 operands,
// products and sums), up to 16 tokens of one request and one head to a workgroup. attn_simple reads every key row and value row
// once per token from a thread of its own; here they are read once per 16 tokens in pieces of 16 bytes, and what bounds a
// workgroup is its chain of blocks (64 matrix instructions of 32 cycles for 16 keys at head size 128). A prompt of 300 tokens,
// 16 heads of 128: 279 -> 25 us; with a workgroup for each request of a tile and no more (for each of its rows, most found nothing to do and held
// 34 KB of LDS meanwhile), the longest tiles first, and what each wave counts worked out once a row, 23.3 -> 18.3, of 1,000 tokens 106 -> 72. A decoding row fills one of 16 columns, but reads its keys in pieces of 16 bytes with four waves
// where attn_simple has a lane walk a key's row: one row over 60 / 512 / 4,096 keys 22 / 138 / 1,128 -> 8 / 21 / 136 us, 64 rows
// over 300 / 2,048 keys 122 / 893 -> 55 / 300, a prompt of 16 tokens 10.0 -> 10.3. Larger heads would need more registers than a wave has and stay with attn_simple, as do
// odd head sizes and pages.
//
// S^T = K Q^T with the keys as the 16-row operand: a lane then holds the scores of keys 4 g .. 4 g + 3 (g: its lane
// group) for token lane % 16, which is the operand that O^T += V^T P^T wants, with the lanes' keys as its k. Keys go in
// blocks of 16 counted from position 0, block i to wave i mod 4; every wave keeps a running maximum, sum and result of its
// own, and the four meet at the end in one order. A block in which a token sees nothing leaves its numbers as they
// are, so a token's bits do not depend on the others of its tile, i.e. on how the request was cut.
// Values of keys that a token does not see meet a probability of zero; where such a value is not a finite number it is
// taken out of the product and joined by hand for the tokens that do see it.
#define F32_WAVES 4
template <int NS, bool MANY>        // NS: head size / 16; MANY: a tile may hold more runs of rows than workgroups are sent to it (a loop, which costs a single row 3 %)
__global__ void __launch_bounds__(64 * F32_WAVES, 2)       // two waves to a SIMD asked for: without it head size 96 took 276 registers and scratch, now 151
attn_f32_kernel(const float* __restrict__ q, int64_t q_stride, float* __restrict__ out, int64_t out_stride,
                const float* __restrict__ k_cache, const float* __restrict__ v_cache, const int32_t* __restrict__ block_tables,
                int bt_stride, const int32_t* __restrict__ seq_of_token, const int32_t* __restrict__ positions,
                const int32_t* __restrict__ context_lens, int num_tokens, int Hq, int Hkv, int page, float scale, int window,
                int keep_first, float softcap, const float* __restrict__ sinks, const float* __restrict__ slopes, int runs) {
  constexpr int D = 16 * NS;
  __shared__ float merge_acc[F32_WAVES][16][D + 4];
  __shared__ float merge_m[F32_WAVES][16], merge_l[F32_WAVES][16], merge_a[F32_WAVES][16], merge_inv[16];
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // The heads of a key head, a tile and a run of its rows share keys: one such unit after the other goes to each XCD (consecutive
  // workgroups go to the XCDs in turn; with all heads side by side those of a key head were on as many XCDs, 64 decoding rows over 2,048
  // keys, 32 and 8 heads of 128, 580 us, now 430). The first tile, which holds the decoding rows, is asked for first, then the last tiles (a
  // prompt's longest): what a compute unit takes beside one of them is short (5 decoding rows beside 200 tokens, 4 and 2 heads of 64, 13.5 -> 11.1 us).
  const uint32_t tiles = (uint32_t)(num_tokens + 15) >> 4, unit = (blockIdx.z * 65535 + blockIdx.y) * 8 + (blockIdx.x & 7);
  const uint32_t place = unit / (uint32_t)Hkv, first_run = place / tiles, rank = place - first_run * tiles;
  if (first_run >= (uint32_t)runs) return;
  const int kvh = unit - place * Hkv, h = kvh * (Hq / Hkv) + (blockIdx.x >> 3);
  const int tile = (rank == 0 ? 0 : tiles - rank) * 16;
  // the tile's runs of rows of one request, by the row at which each begins; this workgroup takes every `runs`-th of them
  const int at_row = tile + col, here = min(at_row, num_tokens - 1);
  const int whose = seq_of_token[here], before = seq_of_token[max(here - 1, 0)], where = positions[here];
  const uint32_t begins = (uint32_t)__ballot(at_row < num_tokens && (col == 0 || whose != before)) & 0xffffu;
  const int in_tile = min(16, num_tokens - tile);
  const int nth = (begins >> col & 1) ? __popc(begins & ((1u << col) - 1u)) : -1;          // the run that begins at this lane's row
  int run = first_run;
  if (run >= __popc(begins)) return;
  do {
  const int z = __builtin_ctzll(__ballot(nth == run)), r0 = tile + z;
  const int rows = (begins >> (z + 1) ? z + 1 + __builtin_ctz(begins >> (z + 1)) : in_tile) - z;
  const int b = __builtin_amdgcn_readlane(whose, z);
  const bool mine = col < rows;
  const int row = mine ? r0 + col : r0;
  const int32_t* bt = block_tables + (int64_t)b * bt_stride;

  // what this lane's token sees, [lo, hi) and [0, kept) as in attn_simple, and the reach of the tile's tokens together
  const int pos = __shfl(where, mine ? z + col : z, ME_WAVE);
  const int hi = min(pos + 1, context_lens[b]);
  const int lo = window > 0 ? max(0, pos - window + 1) : (window < 0 ? pos - pos % (-window) : 0);
  const int kept = (window > 0 && keep_first > 0) ? min(min(keep_first, lo), hi) : 0;
  int hi_most = hi, hi_least = hi, lo_least = lo, lo_most = lo, kept_most = kept;
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) {
    hi_most = max(hi_most, __shfl_xor(hi_most, off, ME_WAVE)); hi_least = min(hi_least, __shfl_xor(hi_least, off, ME_WAVE));
    lo_most = max(lo_most, __shfl_xor(lo_most, off, ME_WAVE)); lo_least = min(lo_least, __shfl_xor(lo_least, off, ME_WAVE));
    kept_most = max(kept_most, __shfl_xor(kept_most, off, ME_WAVE));
  }
  hi_most = __builtin_amdgcn_readfirstlane(hi_most); hi_least = __builtin_amdgcn_readfirstlane(hi_least);
  lo_most = __builtin_amdgcn_readfirstlane(lo_most); lo_least = __builtin_amdgcn_readfirstlane(lo_least);
  kept_most = __builtin_amdgcn_readfirstlane(kept_most);

  f32x4 fq[NS], fk[NS], fv[NS], acc[NS];
  const float* qr = q + (int64_t)row * q_stride + (int64_t)h * D + 4 * g;
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    const float* at = qr + 16 * i;
    fq[i] = f32x4{at[0], at[1], at[2], at[3]};
    acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float m = -INFINITY, l = 0.f;
  const float slope = slopes != nullptr ? slopes[h] : 0.f;

  // this wave's next block of 16 keys at or behind kb (a multiple of 16 that is this wave's) in which some token sees a key
  auto next_block = [&](int kb) {
    if (kb >= kept_most && kb + 16 <= lo_least) kb += ((lo_least - 16 - kb) / (16 * F32_WAVES) + 1) * (16 * F32_WAVES);
    return kb;
  };
  auto page_of = [&](int j) { return bt[min(j, hi_most - 1) / page]; };      // hi_most > 0 wherever this is asked
  auto fetch_keys = [&](int kb, int pg) {
    const int j = kb + col;
    const float* kr = k_cache + ((int64_t)(pg < 0 ? 0 : pg) * Hkv + kvh) * page * D + (pg < 0 ? 0 : (min(j, hi_most - 1) % page) * D) + 4 * g;
#pragma unroll
    for (int i = 0; i < NS; ++i) fk[i] = *reinterpret_cast<const f32x4*>(kr + 16 * i);
  };
  int kb = next_block(16 * wave);            // (block i of 16 keys belongs to wave i mod F32_WAVES)
  int pk = 0, pv = 0;
  if (kb < hi_most) {
    pk = page_of(kb + col); pv = page_of(kb + 4 * g);
    fetch_keys(kb, pk);
  }
  while (kb < hi_most) {
    const int kn = next_block(kb + 16 * F32_WAVES);
    // four keys of a page lie side by side in every dimension's row of values; a group of four that begins behind the last
    // key any token sees is read from the last such group of the table's reach instead and zeroed below
    const int j0 = kb + 4 * g;
    const float* vr = v_cache + ((int64_t)(pv < 0 ? 0 : pv) * Hkv + kvh) * page * D + (j0 < hi_most ? j0 % page : 0);
#pragma unroll
    for (int i = 0; i < NS; ++i) fv[i] = *reinterpret_cast<const f32x4*>(vr + (16 * i + col) * page);
    int pk_next = 0, pv_next = 0;
    if (kn < hi_most) { pk_next = page_of(kn + col); pv_next = page_of(kn + 4 * g); }
    f32x4 s0 = f32x4{0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
    for (int i = 0; i < NS; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (i & 1) s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(fk[i][j], fq[i][j], s1, 0, 0, 0);
        else s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(fk[i][j], fq[i][j], s0, 0, 0, 0);
      }
    if (kn < hi_most) fetch_keys(kn, pk_next);
    f32x4 p;
    bool sees[4];
    float top = m;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int key = j0 + j;
      sees[j] = (key >= lo || key < kept) && key < hi && pv >= 0;
      float s = (s0[j] + s1[j]) * scale;
      if (softcap > 0.f) s = softcap * tanhf(s / softcap);
      s -= slope * (float)(pos - key);
      p[j] = sees[j] ? s : -INFINITY;
      top = fmaxf(top, p[j]);
    }
    top = fmaxf(top, __shfl_xor(top, 16, ME_WAVE));
    top = fmaxf(top, __shfl_xor(top, 32, ME_WAVE));
    const float alpha = m == -INFINITY ? 0.f : expf(m - top);        // m finite implies top finite
#pragma unroll
    for (int j = 0; j < 4; ++j) p[j] = (sees[j] && top > -INFINITY) ? expf(p[j] - top) : 0.f;
    l = l * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
    m = top;
    const bool inside = kb >= lo_least && kb + 16 <= hi_most && __ballot(pv < 0) == 0;
    if (!inside) {                               // keys that no token sees: whatever lies there is not a value
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool in = (j0 + j >= lo_least || j0 + j < kept_most) && j0 + j < hi_most && pv >= 0;
#pragma unroll
        for (int i = 0; i < NS; ++i) fv[i][j] = in ? fv[i][j] : 0.f;
      }
    }
#pragma unroll
    for (int i = 0; i < NS; ++i) acc[i] *= alpha;
    if (!inside || kb < lo_most || kb + 16 > hi_least) {             // some token does not see some key
      float odd = 0.f;                           // becomes a NaN at the first value that is not finite
#pragma unroll
      for (int i = 0; i < NS; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) odd = fmaf(fv[i][j], 0.f, odd);
      if (__ballot(odd != odd) != 0) {
#pragma unroll 1                                 // (a rare way: unrolled, it costs head sizes up to 48 a wave or two per SIMD)
        for (int from = 0; from < 4; ++from)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float pj = __shfl(p[j], from * 16 + col, ME_WAVE);
            const int seen = __shfl((int)sees[j], from * 16 + col, ME_WAVE);
#pragma unroll
            for (int i = 0; i < NS; ++i)
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const float v = __shfl(fv[i][j], from * 16 + 4 * g + e, ME_WAVE);
                if (seen && !(fabsf(v) < INFINITY)) acc[i][e] += pj * v;
              }
          }
#pragma unroll
        for (int i = 0; i < NS; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) fv[i][j] = fabsf(fv[i][j]) < INFINITY ? fv[i][j] : 0.f;
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < NS; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(fv[i][j], p[j], acc[i], 0, 0, 0);
    kb = kn; pk = pk_next; pv = pv_next;
  }
  l += __shfl_xor(l, 16, ME_WAVE);
  l += __shfl_xor(l, 32, ME_WAVE);
  // a lane holds dimensions 16 i + 4 g .. + 3 of token col
  if (g == 0) { merge_m[wave][col] = m; merge_l[wave][col] = l; }
#pragma unroll
  for (int i = 0; i < NS; ++i) *reinterpret_cast<f32x4*>(&merge_acc[wave][col][16 * i + 4 * g]) = acc[i];
  __syncthreads();
  // what each wave's numbers count in a row
  auto weigh = [&](int c, float (&count)[F32_WAVES]) {
    float top = sinks != nullptr ? sinks[h] : -INFINITY;
#pragma unroll
    for (int w = 0; w < F32_WAVES; ++w) top = fmaxf(top, merge_m[w][c]);
    float sum = sinks != nullptr ? expf(sinks[h] - top) : 0.f;
#pragma unroll
    for (int w = 0; w < F32_WAVES; ++w) {
      count[w] = merge_m[w][c] == -INFINITY ? 0.f : expf(merge_m[w][c] - top);
      sum += count[w] * merge_l[w][c];
    }
    return sum > 0.f ? 1.f / sum : 0.f;
  };
  auto put = [&](int c, int d, const float (&count)[F32_WAVES], float inv) {
    float o = 0.f;
#pragma unroll
    for (int w = 0; w < F32_WAVES; ++w) o += count[w] * merge_acc[w][c][d];
    out[(int64_t)(r0 + c) * out_stride + (int64_t)h * D + d] = o * inv;
  };
  float count[F32_WAVES];
  if (rows == 1) {                               // (a thread for every number: no second trip through LDS; 60 keys 6.3 -> 6.2 us)
    const float inv = weigh(0, count);
    if (tid < D) put(0, tid, count, inv);
  } else {                                       // once a row
    if (tid < 16) {
      merge_inv[tid] = weigh(tid, count);
#pragma unroll
      for (int w = 0; w < F32_WAVES; ++w) merge_a[w][tid] = count[w];
    }
    __syncthreads();
    for (int e = tid; e < rows * D; e += 64 * F32_WAVES) {
      const int c = e / D;
#pragma unroll
      for (int w = 0; w < F32_WAVES; ++w) count[w] = merge_a[w][c];
      put(c, e % D, count, merge_inv[c]);
    }
  }
  if (!MANY) return;
  run += runs;
  if (run < __popc(begins)) __syncthreads();       // the numbers in LDS have been read
  } while (run < __popc(begins));
}

extern "C" int me_attn_simple(const void* q, int64_t q_stride, void* out, int64_t out_stride, int dtype,
                              const void* k_cache, const void* v_cache, const int32_t* block_tables,
                              int bt_stride, const int32_t* seq_of_token, const int32_t* positions,
                              const int32_t* context_lens, int64_t num_tokens, int Hq, int Hkv, int D, int page, float scale, int window,
                              int keep_first, float softcap, const float* sinks, const float* slopes, int num_seqs, hipStream_t stream) {
  if (num_tokens == 0) return 0;
  ME_CHECK(Hq >= 1 && Hkv >= 1 && Hq % Hkv == 0, "attention: %d query heads are not a multiple of %d key heads", Hq, Hkv);
  ME_CHECK(D >= 1 && D <= AS_CHANNELS * AS_THREADS, "attention (float32 path): head_dim %d outside 1..%d", D, AS_CHANNELS * AS_THREADS);
  ME_CHECK(page >= 1, "attention: bad page size");
  ME_CHECK(keep_first >= 0 && softcap >= 0.f, "attention: keep_first and softcap must not be negative");
  dim3 grid(num_tokens, Hq), block(AS_THREADS);
  size_t lds = (size_t)(D + AS_THREADS) * sizeof(float);
  const int runs = num_seqs < 1 ? 1 : num_seqs < 16 ? num_seqs : 16;
  const int64_t units = (num_tokens + 15) / 16 * runs * Hkv;           // see `attn_f32_kernel`
  if (dtype == ME_F32 && D % 16 == 0 && D <= 128 && page % 4 == 0 && num_tokens <= 2147483647ll - 16 && units < (1ll << 31) &&
      Hq / Hkv < (1 << 20) &&       (uintptr_t)k_cache % 16 == 0 && (uintptr_t)v_cache % 16 == 0) {
    const int64_t eights = (units + 7) / 8;
    const dim3 tiles((unsigned)(Hq / Hkv * 8), (unsigned)(eights < 65535 ? eights : 65535), (unsigned)((eights + 65534) / 65535)), block(64 * F32_WAVES);
    const bool many = runs > 1 && runs < 16;
#define AS_ARGS <<<tiles, block, 0, stream>>>((const float*)q, q_stride, (float*)out, out_stride, (const float*)k_cache, (const float*)v_cache, \
        block_tables, bt_stride, seq_of_token, positions, context_lens, (int)num_tokens, Hq, Hkv, page, scale, window, keep_first, softcap, sinks, slopes, runs)
#define AS_F32(NS) case NS: if (many) attn_f32_kernel<NS, true> AS_ARGS; else attn_f32_kernel<NS, false> AS_ARGS; break
    switch (D / 16) { AS_F32(1); AS_F32(2); AS_F32(3); AS_F32(4); AS_F32(5); AS_F32(6); AS_F32(7); AS_F32(8); }
#undef AS_F32
#undef AS_ARGS
  } else if (dtype == ME_F32)
    attn_simple_kernel<float><<<grid, block, lds, stream>>>(
        (const float*)q, q_stride, (float*)out, out_stride, (const float*)k_cache, (const float*)v_cache,
        block_tables, bt_stride, seq_of_token, positions, context_lens, Hq, Hkv, D, page, scale, window, keep_first, softcap, sinks, slopes);
  else if (dtype == ME_BF16)
    attn_simple_kernel<bf16_t><<<grid, block, lds, stream>>>(
        (const bf16_t*)q, q_stride, (bf16_t*)out, out_stride, (const bf16_t*)k_cache, (const bf16_t*)v_cache,
        block_tables, bt_stride, seq_of_token, positions, context_lens, Hq, Hkv, D, page, scale, window, keep_first, softcap, sinks, slopes);
  else
    ME_CHECK(false, "attention: bad dtype code %d", dtype);
  ME_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------------ further terms of a softmax that another kernel has formed
// The matrix-core kernels attend over one contiguous range of keys. What a mask or a softmax has beyond that joins here:
// the keys at positions below keep_first that a window has left behind, and a sink per head. out holds the other
// kernel's normalised result and lse the natural logarithm of its denominator (-inf: it saw no key). With
// (m2, l2, acc2) the kept keys' maximum, sum and weighted values, sk the sink and M the largest of lse, m2, sk:
//   out <- (out e^(lse - M) + acc2 e^(m2 - M)) / (e^(lse - M) + l2 e^(m2 - M) + e^(sk - M)).
// One wave per (token, head); for the scores four neighbouring lanes share a key, sixteen keys at a time; for the values a
// lane takes the channels lane, lane + 64, ...
#define AT_MAX_D 512
template <typename T>
__global__ void __launch_bounds__(64)
attn_tail_kernel(const T* __restrict__ q, int64_t q_stride, T* __restrict__ out, int64_t out_stride, const float* __restrict__ lse,
                 const T* __restrict__ k_cache, const T* __restrict__ v_cache, const int32_t* __restrict__ block_tables, int bt_stride,
                 const int32_t* __restrict__ seq_of_token, const int32_t* __restrict__ positions,
                 const int32_t* __restrict__ context_lens, int Hq, int Hkv, int D, int page, float scale, int window,
                 int keep_first, float softcap, const float* __restrict__ sinks, const float* __restrict__ slopes) {
  __shared__ float qs[AT_MAX_D];
  __shared__ float sc[64];
  const int64_t t = blockIdx.x;
  const int h = blockIdx.y, lane = threadIdx.x;
  const int kvh = h / (Hq / Hkv);
  const int b = seq_of_token[t];
  const int pos = positions[t];
  const int32_t* bt = block_tables + (int64_t)b * bt_stride;
  const int hi = min(pos + 1, context_lens[b]);
  const int lo = window > 0 ? max(0, pos - window + 1) : 0;
  const int kept = (window > 0 && keep_first > 0) ? min(min(keep_first, lo), hi) : 0;
  const float slope = slopes != nullptr ? slopes[h] : 0.f;
  float m2 = -INFINITY, l2 = 0.f;
  float acc[AT_MAX_D / 64];
#pragma unroll
  for (int i = 0; i < AT_MAX_D / 64; ++i) acc[i] = 0.f;
  if (kept > 0) {
    for (int d = lane; d < D; d += 64) qs[d] = to_f32<T>(q[t * q_stride + (int64_t)h * D + d]);
    __syncthreads();
    // sixteen keys at a time: four neighbouring lanes share a key, each with every fourth of the head's dimensions
    const int part = lane & 3;
    for (int c0 = 0; c0 < kept; c0 += 16) {
      const int j = c0 + (lane >> 2);
      float s = -INFINITY;
      int64_t pg = -1;
      if (j < kept) pg = bt[j / page];
      float dot = 0.f;
      if (pg >= 0) {
        const T* kr = k_cache + ((pg * Hkv + kvh) * (int64_t)page + j % page) * D;
        for (int d = part; d < D; d += 4) dot += qs[d] * to_f32<T>(kr[d]);      // neighbours read neighbouring words
      }
      dot += __shfl_xor(dot, 1, ME_WAVE);
      dot += __shfl_xor(dot, 2, ME_WAVE);
      if (pg >= 0) {
        s = dot * scale;
        if (softcap > 0.f) s = softcap * tanhf(s / softcap);
        s -= slope * (float)(pos - j);
      }
      const float m_new = fmaxf(m2, wave_max(s));
      const float p = (s > -INFINITY) ? expf(s - m_new) : 0.f;
      const float alpha = (m2 == -INFINITY) ? 0.f : expf(m2 - m_new);
      l2 = l2 * alpha + wave_sum(part == 0 ? p : 0.f);
      m2 = m_new;
      __syncthreads();
      if (part == 0) sc[lane >> 2] = p;
      __syncthreads();
      const int je = min(16, kept - c0);
#pragma unroll
      for (int i = 0; i < AT_MAX_D / 64; ++i) {
        const int d = lane + 64 * i;
        if (d < D) {
          float a = 0.f;
          for (int jj = 0; jj < je; ++jj) {
            const int64_t vp = bt[(c0 + jj) / page];
            if (vp < 0) continue;
            a += sc[jj] * to_f32<T>(v_cache[((vp * Hkv + kvh) * (int64_t)D + d) * page + (c0 + jj) % page]);
          }
          acc[i] = acc[i] * alpha + a;
        }
      }
    }
  }
  const float l1 = lse[t * Hq + h];
  const float sk = sinks != nullptr ? sinks[h] : -INFINITY;
  const float M = fmaxf(fmaxf(l1, m2), sk);
  float w1 = 0.f, w2 = 0.f, ws = 0.f;
  if (M > -INFINITY) {
    w1 = l1 > -INFINITY ? expf(l1 - M) : 0.f;
    w2 = m2 > -INFINITY ? expf(m2 - M) : 0.f;
    ws = sk > -INFINITY ? expf(sk - M) : 0.f;
  }
  const float denom = w1 + w2 * l2 + ws;
  const float inv = denom > 0.f ? 1.f / denom : 0.f;
#pragma unroll
  for (int i = 0; i < AT_MAX_D / 64; ++i) {
    const int d = lane + 64 * i;
    if (d < D) {
      T* at = out + t * out_stride + (int64_t)h * D + d;
      *at = from_f32<T>((to_f32<T>(*at) * w1 + acc[i] * w2) * inv);
    }
  }
}

// The same for bfloat16 heads of 64 or 128 channels over pages in steps of 16 keys, where sixteen keys lie on one page and a
// channel's values of them are 32 adjacent bytes. The general kernel is a chain of loads of two bytes, each value behind a look
// into the block table; here a lane asks for a key's row and its channels' values in 16-byte pieces, all at once, and the four
// lanes of a key pick their every fourth dimension out of the same pieces. Every sum keeps its order, so the results are the
// same bits. A token without kept keys whose head has no sink is left as it is: its weights are exactly 1 over 1.
// (3,123 tokens, 16 heads of 128, 16 kept keys: 95.6 -> 24.1 us, of which the rows in and out take some 5)
template <int D>
__global__ void __launch_bounds__(64)
attn_tail_pages_kernel(const bf16_t* __restrict__ q, int64_t q_stride, bf16_t* __restrict__ out, int64_t out_stride,
                       const float* __restrict__ lse, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
                       const int32_t* __restrict__ block_tables, int bt_stride, const int32_t* __restrict__ seq_of_token,
                       const int32_t* __restrict__ positions, const int32_t* __restrict__ context_lens, int Hq, int Hkv, int page,
                       float scale, int window, int keep_first, float softcap, const float* __restrict__ sinks,
                       const float* __restrict__ slopes) {
  constexpr int NI = D / 64;
  __shared__ float qs[D];
  __shared__ float sc[16];
  const int64_t t = blockIdx.x;
  const int h = blockIdx.y, lane = threadIdx.x;
  const int kvh = h / (Hq / Hkv);
  const int b = seq_of_token[t];
  const int pos = positions[t];
  const float l1 = lse[t * Hq + h];
  const float sk = sinks != nullptr ? sinks[h] : -INFINITY;
  const float slope = slopes != nullptr ? slopes[h] : 0.f;
  const int32_t* bt = block_tables + (int64_t)b * bt_stride;
  const int hi = min(pos + 1, context_lens[b]);
  const int lo = window > 0 ? max(0, pos - window + 1) : 0;
  const int kept = (window > 0 && keep_first > 0) ? min(min(keep_first, lo), hi) : 0;
  if (kept <= 0 && sinks == nullptr && fabsf(l1) < INFINITY) return;
  bf16_t* row = out + t * out_stride + (int64_t)h * D;
  bf16_t held[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) held[i] = row[lane + 64 * i];
  float m2 = -INFINITY, l2 = 0.f;
  float acc[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) acc[i] = 0.f;
  if (kept > 0) {
    bf16_t qv[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) qv[i] = q[t * q_stride + (int64_t)h * D + lane + 64 * i];
    const int part = lane & 3;
    bool laid = false;
    for (int c0 = 0; c0 < kept; c0 += 16) {
      const int64_t pg = bt[c0 / page];
      if (pg < 0) continue;                       // a page that is not there: sixteen keys fewer
      const int off = c0 % page, je = min(16, kept - c0), j = c0 + (lane >> 2);
      const uint64_t* kr = (const uint64_t*)(k_cache + ((pg * Hkv + kvh) * (int64_t)page + off + (lane >> 2)) * D);
      ulong2 kw[D / 8];
      bf16x8 vw[NI][2];
#pragma unroll
      for (int i = 0; i < D / 8; ++i) kw[i] = ((const ulong2*)kr)[i];
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const bf16x8* vr = (const bf16x8*)(v_cache + ((pg * Hkv + kvh) * (int64_t)D + lane + 64 * i) * page + off);
        vw[i][0] = vr[0];
        vw[i][1] = vr[1];
      }
      if (!laid) {                                // behind the requests for keys and values: q is waited for with them
#pragma unroll
        for (int i = 0; i < NI; ++i) qs[lane + 64 * i] = to_f32<bf16_t>(qv[i]);
        laid = true;
      }
      __syncthreads();
      float dot = 0.f;
#pragma unroll
      for (int i = 0; i < D / 4; ++i) {           // dimension 4 i + part
        const uint64_t four = i & 1 ? kw[i >> 1].y : kw[i >> 1].x;
        dot += qs[4 * i + part] * __uint_as_float((uint32_t)(four >> (16 * part)) << 16);
      }
      dot += __shfl_xor(dot, 1, ME_WAVE);
      dot += __shfl_xor(dot, 2, ME_WAVE);
      float s = -INFINITY;
      if (j < kept) {
        s = dot * scale;
        if (softcap > 0.f) s = softcap * tanhf(s / softcap);
        s -= slope * (float)(pos - j);
      }
      const float m_new = fmaxf(m2, wave_max(s));
      const float p = (s > -INFINITY) ? expf(s - m_new) : 0.f;
      const float alpha = (m2 == -INFINITY) ? 0.f : expf(m2 - m_new);
      l2 = l2 * alpha + wave_sum(part == 0 ? p : 0.f);
      m2 = m_new;
      if (part == 0) sc[lane >> 2] = p;
      __syncthreads();
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        float a = 0.f;
#pragma unroll
        for (int jj = 0; jj < 16; ++jj)
          if (jj < je) a += sc[jj] * to_f32<bf16_t>(vw[i][jj >> 3][jj & 7]);
        acc[i] = acc[i] * alpha + a;
      }
    }
  }
  const float M = fmaxf(fmaxf(l1, m2), sk);
  float w1 = 0.f, w2 = 0.f, ws = 0.f;
  if (M > -INFINITY) {
    w1 = l1 > -INFINITY ? expf(l1 - M) : 0.f;
    w2 = m2 > -INFINITY ? expf(m2 - M) : 0.f;
    ws = sk > -INFINITY ? expf(sk - M) : 0.f;
  }
  const float denom = w1 + w2 * l2 + ws;
  const float inv = denom > 0.f ? 1.f / denom : 0.f;
#pragma unroll
  for (int i = 0; i < NI; ++i) row[lane + 64 * i] = from_f32<bf16_t>((to_f32<bf16_t>(held[i]) * w1 + acc[i] * w2) * inv);
}

extern "C" int me_attn_tail(const void* q, int64_t q_stride, void* out, int64_t out_stride, const float* lse, int dtype,
                            const void* k_cache, const void* v_cache, const int32_t* block_tables, int bt_stride,
                            const int32_t* seq_of_token, const int32_t* positions, const int32_t* context_lens,
                            int64_t num_tokens, int Hq, int Hkv, int D, int page, float scale, int window, int keep_first,
                            float softcap, const float* sinks, const float* slopes, hipStream_t stream) {
  if (num_tokens == 0) return 0;
  ME_CHECK(Hq >= 1 && Hkv >= 1 && Hq % Hkv == 0 && Hq <= 65535, "attention tail: %d query heads over %d key heads", Hq, Hkv);
  ME_CHECK(D >= 1 && D <= AT_MAX_D && page >= 1 && keep_first >= 0 && softcap >= 0.f, "attention tail: head size 1..%d", AT_MAX_D);
  ME_CHECK(lse != nullptr && num_tokens <= 2147483647ll, "attention tail: the other kernel's denominators are missing");
  dim3 grid((unsigned)num_tokens, Hq), block(64);
  if (dtype == ME_F32)
    attn_tail_kernel<float><<<grid, block, 0, stream>>>((const float*)q, q_stride, (float*)out, out_stride, lse, (const float*)k_cache,
        (const float*)v_cache, block_tables, bt_stride, seq_of_token, positions, context_lens, Hq, Hkv, D, page, scale, window,
        keep_first, softcap, sinks, slopes);
  else if ((D == 64 || D == 128) && page % 16 == 0 && (uintptr_t)k_cache % 16 == 0 && (uintptr_t)v_cache % 16 == 0) {
#define TAIL(DD) attn_tail_pages_kernel<DD><<<grid, block, 0, stream>>>((const bf16_t*)q, q_stride, (bf16_t*)out, out_stride, lse, \
        (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_tables, bt_stride, seq_of_token, positions, context_lens, Hq, Hkv, page, \
        scale, window, keep_first, softcap, sinks, slopes)
    if (D == 64) TAIL(64);
    else TAIL(128);
#undef TAIL
  } else
    attn_tail_kernel<bf16_t><<<grid, block, 0, stream>>>((const bf16_t*)q, q_stride, (bf16_t*)out, out_stride, lse, (const bf16_t*)k_cache,
        (const bf16_t*)v_cache, block_tables, bt_stride, seq_of_token, positions, context_lens, Hq, Hkv, D, page, scale, window,
        keep_first, softcap, sinks, slopes);
  ME_LAUNCH_CHECK();
  return 0;
}
