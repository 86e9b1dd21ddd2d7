// Kernels of mixers that run two token mixers side by side, one of them a recurrence whose state rows decay each at
// a rate of their own: the mix of a token's input with the previous token's, the recurrence itself under two update
// rules, the weighted sum of the two mixers' outputs, and the small elementwise steps around them (a bias on a
// projection's rows, an elementwise sigmoid gate). Everything that the recurrence reads
// besides the projections is formed here in float32: decays and their exponentials, softplus, write strengths, unit
// lengths.
#include "common.h"
#include <type_traits>

__device__ __forceinline__ float hy_sigmoid(float v) { return 1.0f / (1.0f + expf(-v)); }
__device__ __forceinline__ float hy_softplus(float v) { return v > 20.f ? v : log1pf(expf(v)); }

// Four adjacent values at an address of four elements' alignment, and the test for it.
template <typename T> struct Four;
template <> struct Four<float> { typedef f32x4 type; };
template <> struct Four<bf16_t> { typedef bf16x4 type; };
template <typename T>
__device__ __forceinline__ typename Four<T>::type four_of(const T* p) { return *(const typename Four<T>::type*)p; }
static bool by_fours(const void* p, int dtype, int64_t stride) {
  return (uintptr_t)p % (dtype == ME_F32 ? 16 : 8) == 0 && stride % 4 == 0;
}
// Whether T rows of n go to the kernels that take a row by fours with a column of workgroups each, and their threads: from 128
// numbers on (16,384 rows of 64: bias 4.5 us with a thread per number and 6.0 by fours, of 128 6.4 and 6.3, of 256 10.1 and
// 6.9), and while the grid's first side stays below 2^32 threads.
static int threads_by_fours(int n) { return n / 4 >= 256 ? 256 : 64; }
static bool rows_by_fours(int64_t T, int n) { return n % 4 == 0 && n >= 128 && n <= 4000000 && T * threads_by_fours(n) < (1ll << 32); }

// ------------------------------------------------------------------ rows + bias
// out[t, c] = (sum_p x[p, t, c]) + bias[c] for c < nb, without a bias beyond; x: `parts` stacked slices.
template <typename TX, typename TY>
__global__ void add_bias_kernel(const TX* __restrict__ x, int parts, int64_t part_stride, int64_t x_stride,
                                const float* __restrict__ bias, int nb, TY* __restrict__ out, int64_t T, int n) {
  const int64_t total = T * n;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = i / n;
    const int c = (int)(i - t * n);
    float v = 0.f;
    for (int p = 0; p < parts; ++p) v += to_f32<TX>(x[p * part_stride + t * x_stride + c]);
    if (c < nb) v += bias[c];
    out[i] = from_f32<TY>(v);
  }
}

// The same by fours, a row to a column of workgroups: no division by the row's length, and a 16-byte load where the general
// kernel has four. (3,123 rows of 4,096 float32 sums to bfloat16, 77 MB: 31.4 -> 13.7 us)
template <typename TX, typename TY>
__global__ void add_bias_fours_kernel(const TX* __restrict__ x, int parts, int64_t part_stride, int64_t x_stride,
                                      const float* __restrict__ bias, int nb, TY* __restrict__ out, int n) {
  const int64_t t = blockIdx.x;
  const int c = (blockIdx.y * blockDim.x + threadIdx.x) * 4;
  if (c >= n) return;
  f32x4 b = {0.f, 0.f, 0.f, 0.f}, v = {0.f, 0.f, 0.f, 0.f};
  if (c < nb) b = four_of<float>(bias + c);
  for (int p = 0; p < parts; ++p) {
    const auto one = four_of<TX>(x + p * part_stride + t * x_stride + c);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += to_f32<TX>(one[i]);
  }
  typename Four<TY>::type o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = from_f32<TY>(c < nb ? v[i] + b[i] : v[i]);
  *(typename Four<TY>::type*)(out + t * n + c) = o;
}

extern "C" int me_add_bias(const void* x, int x_dtype, int parts, int64_t part_stride, int64_t x_stride, const float* bias, int nb,
                           void* out, int out_dtype, int64_t T, int n, hipStream_t stream) {
  if (T == 0 || n == 0) return 0;
  ME_CHECK(parts >= 1 && nb >= 0 && nb <= n, "add_bias: bad slice count or bias length");
  const int64_t total = T * n;
  const dim3 grid((unsigned)((total + 255) / 256 < 65535 ? (total + 255) / 256 : 65535)), block(256);
  const int threads = threads_by_fours(n);
  const bool fours = rows_by_fours(T, n) && nb % 4 == 0 && (nb == 0 || by_fours(bias, ME_F32, 0)) && by_fours(x, x_dtype, x_stride) &&
                     (parts == 1 || part_stride % 4 == 0) && by_fours(out, out_dtype, 0);
  const dim3 rows((unsigned)T, (n / 4 + threads - 1) / threads);
#define AB(TX, TY) do { \
    if (fours) add_bias_fours_kernel<TX, TY><<<rows, threads, 0, stream>>>((const TX*)x, parts, part_stride, x_stride, bias, nb, (TY*)out, n); \
    else add_bias_kernel<TX, TY><<<grid, block, 0, stream>>>((const TX*)x, parts, part_stride, x_stride, bias, nb, (TY*)out, T, n); } while (0)
  if (x_dtype == ME_F32 && out_dtype == ME_F32) AB(float, float);
  else if (x_dtype == ME_F32) AB(float, bf16_t);
  else if (out_dtype == ME_F32) AB(bf16_t, float);
  else AB(bf16_t, bf16_t);
#undef AB
  ME_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------------ o *= sigmoid(g), element by element
template <typename TX>
__global__ void sigmoid_gate_kernel(TX* __restrict__ o, int64_t o_stride, const TX* __restrict__ g, int64_t g_stride, int64_t T, int n) {
  const int64_t total = T * n;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = i / n;
    const int c = (int)(i - t * n);
    TX* at = o + t * o_stride + c;
    *at = from_f32<TX>(to_f32<TX>(*at) * hy_sigmoid(to_f32<TX>(g[t * g_stride + c])));
  }
}

// The same by fours, a row to a column of workgroups. (3,123 rows of 2,048 in bfloat16, 38 MB: 16.3 -> 8.9 us)
template <typename TX>
__global__ void sigmoid_gate_fours_kernel(TX* __restrict__ o, int64_t o_stride, const TX* __restrict__ g, int64_t g_stride, int n) {
  const int64_t t = blockIdx.x;
  const int c = (blockIdx.y * blockDim.x + threadIdx.x) * 4;
  if (c >= n) return;
  auto v = four_of<TX>(o + t * o_stride + c);
  const auto gate = four_of<TX>(g + t * g_stride + c);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = from_f32<TX>(to_f32<TX>(v[i]) * hy_sigmoid(to_f32<TX>(gate[i])));
  *(typename Four<TX>::type*)(o + t * o_stride + c) = v;
}

extern "C" int me_sigmoid_gate(void* o, int64_t o_stride, const void* g, int64_t g_stride, int dtype, int64_t T, int n, hipStream_t stream) {
  if (T == 0 || n == 0) return 0;
  const int64_t total = T * n;
  const dim3 grid((unsigned)((total + 255) / 256 < 65535 ? (total + 255) / 256 : 65535)), block(256);
  if (rows_by_fours(T, n) && by_fours(o, dtype, o_stride) && by_fours(g, dtype, g_stride)) {
    const int threads = threads_by_fours(n);
    const dim3 rows((unsigned)T, (n / 4 + threads - 1) / threads);
    if (dtype == ME_F32) sigmoid_gate_fours_kernel<float><<<rows, threads, 0, stream>>>((float*)o, o_stride, (const float*)g, g_stride, n);
    else sigmoid_gate_fours_kernel<bf16_t><<<rows, threads, 0, stream>>>((bf16_t*)o, o_stride, (const bf16_t*)g, g_stride, n);
  } else if (dtype == ME_F32) sigmoid_gate_kernel<float><<<grid, block, 0, stream>>>((float*)o, o_stride, (const float*)g, g_stride, T, n);
  else sigmoid_gate_kernel<bf16_t><<<grid, block, 0, stream>>>((bf16_t*)o, o_stride, (const bf16_t*)g, g_stride, T, n);
  ME_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------------ weighted sum of sublayer outputs
// out[t, c] = sum_i scale_i * gate_i[t] * ((sum_p term_i[p, t, c]) + bias_i[c]), float32. Terms are rows in the compute dtype or
// stacked float32 partial sums. gate_i[t] = sigmoid(g_i[t * gate_stride_i]) for a term that has gate rows g_i (in the compute
// dtype or float32), else 1. With w: the norm on the sum as well, stream' = stream + w * out / rms(out), one
// workgroup per row (the sum is held in LDS between the two passes), the new stream also rounded to TY.
#define WS_MAX_TERMS 4
struct WsArgs {
  const void* term[WS_MAX_TERMS]; int dtype[WS_MAX_TERMS]; int parts[WS_MAX_TERMS]; int64_t part_stride[WS_MAX_TERMS];
  float scale[WS_MAX_TERMS]; const float* bias[WS_MAX_TERMS];
  const void* gate[WS_MAX_TERMS]; int gate_dtype[WS_MAX_TERMS]; int64_t gate_stride[WS_MAX_TERMS];
  int count, n;
};

__device__ __forceinline__ float ws_value(const WsArgs& a, int64_t t, int c) {
  float total = 0.f;
  for (int i = 0; i < a.count; ++i) {
    float v = 0.f;
    if (a.dtype[i] == ME_F32) {
      const float* x = (const float*)a.term[i];
      for (int p = 0; p < a.parts[i]; ++p) v += x[p * a.part_stride[i] + t * a.n + c];
    } else {
      v = to_f32<bf16_t>(((const bf16_t*)a.term[i])[t * a.n + c]);
    }
    if (a.bias[i] != nullptr) v += a.bias[i][c];
    if (a.gate[i] != nullptr) {
      const float g = a.gate_dtype[i] == ME_F32 ? ((const float*)a.gate[i])[t * a.gate_stride[i]]
                                                : to_f32<bf16_t>(((const bf16_t*)a.gate[i])[t * a.gate_stride[i]]);
      v *= 1.0f / (1.0f + expf(-g));
    }
    total += a.scale[i] * v;
  }
  return total;
}

__global__ void weighted_sum_kernel(WsArgs a, float* __restrict__ out, int64_t T) {
  const int64_t total = T * a.n;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = i / a.n;
    out[i] = ws_value(a, t, (int)(i - t * a.n));
  }
}

template <typename TY>
__global__ void weighted_sum_norm_kernel(WsArgs a, const float* __restrict__ w, float eps, const float* __restrict__ stream_in,
                                         float* __restrict__ stream_out, TY* __restrict__ rounded) {
  __shared__ float scratch[16];
  extern __shared__ float row[];
  const int64_t t = blockIdx.x;
  float ss = 0.f;
  for (int c = threadIdx.x; c < a.n; c += blockDim.x) {
    const float v = ws_value(a, t, c);
    row[c] = v;
    ss += v * v;
  }
  ss = block_sum(ss, scratch);
  const float inv = 1.0f / sqrtf(ss / (float)a.n + eps);
  for (int c = threadIdx.x; c < a.n; c += blockDim.x) {
    const float v = stream_in[t * a.n + c] + w[c] * (row[c] * inv);
    stream_out[t * a.n + c] = v;
    if (rounded != nullptr) rounded[t * a.n + c] = from_f32<TY>(v);
  }
}

// Rows of 1,024 to 4,096: a thread holds its values (the same ones, so the row's sum keeps its order) in registers and asks for a
// term's, the stream's and the weights' all at once; the general kernel goes to memory for one value at a time.
// (3,123 rows of 1,024, two terms: 20.8 -> 13.1 us; which launches it takes: rows_in_registers)
template <typename TY, int NV>
__global__ void __launch_bounds__(256)
weighted_sum_norm_regs_kernel(WsArgs a, const float* __restrict__ w, float eps, const float* __restrict__ stream_in,
                              float* __restrict__ stream_out, TY* __restrict__ rounded) {
  __shared__ float scratch[16];
  const int64_t t = blockIdx.x;
  const int n = a.n, tid = threadIdx.x;
  float held[NV], wv[NV], total[NV], v[NV], bias[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) total[k] = 0.f;
  for (int i = 0; i < a.count; ++i) {
    float g = 0.f;
    if (a.gate[i] != nullptr)
      g = a.gate_dtype[i] == ME_F32 ? ((const float*)a.gate[i])[t * a.gate_stride[i]]
                                    : to_f32<bf16_t>(((const bf16_t*)a.gate[i])[t * a.gate_stride[i]]);
    if (a.bias[i] != nullptr) {
#pragma unroll
      for (int k = 0; k < NV; ++k) bias[k] = a.bias[i][min(tid + 256 * k, n - 1)];
    }
    if (a.dtype[i] == ME_F32) {
#pragma unroll
      for (int k = 0; k < NV; ++k) v[k] = 0.f;
      for (int p = 0; p < a.parts[i]; ++p) {
        const float* x = (const float*)a.term[i] + p * a.part_stride[i] + t * n;
#pragma unroll
        for (int k = 0; k < NV; ++k) v[k] += x[min(tid + 256 * k, n - 1)];
      }
    } else {
      const bf16_t* x = (const bf16_t*)a.term[i] + t * n;
#pragma unroll
      for (int k = 0; k < NV; ++k) v[k] = to_f32<bf16_t>(x[min(tid + 256 * k, n - 1)]);
    }
    if (i == 0) {
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        held[k] = stream_in[t * n + min(tid + 256 * k, n - 1)];
        wv[k] = w[min(tid + 256 * k, n - 1)];
      }
    }
    const float share = a.gate[i] != nullptr ? 1.0f / (1.0f + expf(-g)) : 0.f;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      if (a.bias[i] != nullptr) v[k] += bias[k];
      if (a.gate[i] != nullptr) v[k] *= share;
      total[k] += a.scale[i] * v[k];
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < NV; ++k)
    if (tid + 256 * k < n) ss += total[k] * total[k];
  ss = block_sum(ss, scratch);
  const float inv = 1.0f / sqrtf(ss / (float)n + eps);
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int c = tid + 256 * k;
    if (c < n) {
      const float o = held[k] + wv[k] * (total[k] * inv);
      stream_out[t * n + c] = o;
      if (rounded != nullptr) rounded[t * n + c] = from_f32<TY>(o);
    }
  }
}

// Up to how many rows the form in registers takes a launch whose float32 terms have `sums` partial sums together. Its 65, 128
// and 238 registers leave a compute unit 7, 4 and 2 workgroups where the general kernel has 8: as long as the launch is a round or
// two of them that costs nothing, and reads of bfloat16 rows, one trip a term, are ahead at any number; but every partial sum is
// a trip of its own that few waves wait out. us, general kernel / registers: rows of 2,560, one float32 term and one of bfloat16 at
// 1,024 rows 21 / 18, at 2,048 26 / 33, with three partial sums at 512 rows 20 / 13, at 1,024 28 / 31, at 8,192 169 / 346; of
// 2,048, one term at 16,384 rows 196 / 148, nine partial sums at 1,024 rows 35 / 29, at 2,048 39 / 54; of 1,024, three at 8,192 rows
// 51 / 42, nine at 2,048 22 / 28.
static int64_t rows_in_registers(int n, int64_t sums, int64_t any) {
  if (sums == 0) return any;
  if (n <= 1024) return sums <= 4 ? any : 1024;
  if (n <= 2048) return sums == 1 ? any : 1024;
  return sums == 1 ? 1024 : 512;
}

extern "C" int me_weighted_sum(int count, const void** terms, const int* dtypes, const int* parts, const int64_t* part_strides,
                               const float* scales, const float** biases, float* out, const float* w, float eps,
                               const float* stream_in, float* stream_out, void* rounded, int rounded_dtype, int64_t T, int n,
                               const void** gates, const int* gate_dtypes, const int64_t* gate_strides, hipStream_t stream) {
  if (T == 0 || n == 0) return 0;
  ME_CHECK(count >= 1 && count <= WS_MAX_TERMS, "weighted_sum: 1..%d terms", WS_MAX_TERMS);
  WsArgs a;
  a.count = count; a.n = n;
  int64_t sums = 0;
  for (int i = 0; i < count; ++i) {
    ME_CHECK(parts[i] >= 1 && (dtypes[i] == ME_F32 || parts[i] == 1), "weighted_sum: partial sums are float32");
    if (dtypes[i] == ME_F32) sums += parts[i];
    a.term[i] = terms[i]; a.dtype[i] = dtypes[i]; a.parts[i] = parts[i]; a.part_stride[i] = part_strides[i];
    a.scale[i] = scales[i]; a.bias[i] = biases[i];
    a.gate[i] = gates ? gates[i] : nullptr; a.gate_dtype[i] = gates ? gate_dtypes[i] : ME_F32; a.gate_stride[i] = gates ? gate_strides[i] : 0;
  }
  if (w == nullptr) {
    const int64_t total = T * n;
    const dim3 grid((unsigned)((total + 255) / 256 < 65535 ? (total + 255) / 256 : 65535)), block(256);
    weighted_sum_kernel<<<grid, block, 0, stream>>>(a, out, T);
  } else {
    ME_CHECK(n <= 15360 && stream_in != nullptr && stream_out != nullptr, "weighted_sum: rows of up to 15360 with a stream");
    const dim3 grid((unsigned)T), block(n >= 1024 ? 256 : (n > 256 ? 128 : 64));
    const size_t lds = (size_t)n * sizeof(float);
#define WS(TY) do { \
    if (n <= 1024) weighted_sum_norm_regs_kernel<TY, 4><<<grid, block, 0, stream>>>(a, w, eps, stream_in, stream_out, (TY*)rounded); \
    else if (n <= 2048) weighted_sum_norm_regs_kernel<TY, 8><<<grid, block, 0, stream>>>(a, w, eps, stream_in, stream_out, (TY*)rounded); \
    else weighted_sum_norm_regs_kernel<TY, 16><<<grid, block, 0, stream>>>(a, w, eps, stream_in, stream_out, (TY*)rounded); } while (0)
    if (n >= 1024 && n <= 4096 && T <= rows_in_registers(n, sums, T)) {
      if (rounded == nullptr || rounded_dtype == ME_F32) WS(float);
      else WS(bf16_t);
    } else if (rounded == nullptr || rounded_dtype == ME_F32)
#undef WS
      weighted_sum_norm_kernel<float><<<grid, block, lds, stream>>>(a, w, eps, stream_in, stream_out, (float*)rounded);
    else
      weighted_sum_norm_kernel<bf16_t><<<grid, block, lds, stream>>>(a, w, eps, stream_in, stream_out, (bf16_t*)rounded);
  }
  ME_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------------ a token's input mixed with the previous token's
// out[s, t, c] = x[t, c] + (before[t, c] - x[t, c]) * mu[s, c], s < S. before: the row of the request's previous token;
// for the first token of the request's tokens in this step it comes from the request's state row (zeros at position 0,
// which the step function has written there), which then takes the step's last row. The thread of a request's first
// token reads the state before it writes it, so a step needs no second launch.
template <typename TX>
__global__ void token_shift_kernel(const TX* __restrict__ x, int64_t x_stride, const float* __restrict__ mu, int S,
                                   float* __restrict__ state, int64_t state_stride, const int32_t* __restrict__ slots,
                                   const int32_t* __restrict__ cu, const int32_t* __restrict__ seq_of_token,
                                   TX* __restrict__ out, int64_t T, int n) {
  const int64_t t = blockIdx.x;
  const int b = seq_of_token[t];
  const int64_t first = cu[b], last = (int64_t)cu[b + 1] - 1;
  for (int c = blockIdx.y * blockDim.x + threadIdx.x; c < n; c += gridDim.y * blockDim.x) {
    const float now = to_f32<TX>(x[t * x_stride + c]);
    float before;
    if (t == first) {
      float* held = state + (int64_t)slots[b] * state_stride + c;
      before = *held;
      *held = to_f32<TX>(x[last * x_stride + c]);
    } else {
      before = to_f32<TX>(x[(t - 1) * x_stride + c]);
    }
    const float d = before - now;
    for (int s = 0; s < S; ++s) out[((int64_t)s * T + t) * n + c] = from_f32<TX>(now + d * mu[(int64_t)s * n + c]);
  }
}

// The same by fours: the two rows once, then a mix's four weights and four results at a time.
// (3,123 tokens of 1,024 in bfloat16, five mixes: 19.7 -> 11.4 us)
template <typename TX>
__global__ void token_shift_fours_kernel(const TX* __restrict__ x, int64_t x_stride, const float* __restrict__ mu, int S,
                                         float* __restrict__ state, int64_t state_stride, const int32_t* __restrict__ slots,
                                         const int32_t* __restrict__ cu, const int32_t* __restrict__ seq_of_token,
                                         TX* __restrict__ out, int64_t T, int n) {
  const int64_t t = blockIdx.x;
  const int c = (blockIdx.y * blockDim.x + threadIdx.x) * 4;
  if (c >= n) return;
  const auto own = four_of<TX>(x + t * x_stride + c);
  const auto left = four_of<TX>(x + (t > 0 ? t - 1 : 0) * x_stride + c);
  const int b = seq_of_token[t];
  float now[4], d[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    now[i] = to_f32<TX>(own[i]);
    d[i] = to_f32<TX>(left[i]) - now[i];
  }
  if (t == cu[b]) {
    float* held = state + (int64_t)slots[b] * state_stride + c;
    const TX* last = x + ((int64_t)cu[b + 1] - 1) * x_stride + c;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      d[i] = held[i] - now[i];
      held[i] = to_f32<TX>(last[i]);
    }
  }
#pragma unroll 4
  for (int s = 0; s < S; ++s) {
    const f32x4 m = four_of<float>(mu + (int64_t)s * n + c);
    typename Four<TX>::type o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = from_f32<TX>(now[i] + d[i] * m[i]);
    *(typename Four<TX>::type*)(out + ((int64_t)s * T + t) * n + c) = o;
  }
}

extern "C" int me_token_shift(const void* x, int64_t x_stride, int dtype, const float* mu, int S, float* state, int64_t state_stride,
                              const int32_t* slots, const int32_t* cu, const int32_t* seq_of_token, void* out, int64_t T, int n,
                              hipStream_t stream) {
  if (T == 0 || n == 0) return 0;
  ME_CHECK(S >= 1 && T <= 2147483647ll, "token_shift: bad sizes");
  const dim3 block(n >= 256 ? 256 : 64);
  const unsigned gy = (unsigned)((n + block.x - 1) / block.x < 64 ? (n + block.x - 1) / block.x : 64);
  const dim3 grid((unsigned)T, gy);
  if (rows_by_fours(T, n) && by_fours(x, dtype, x_stride) && by_fours(mu, ME_F32, 0) && by_fours(out, dtype, 0)) {
    const int threads = threads_by_fours(n);
    const dim3 rows((unsigned)T, (n / 4 + threads - 1) / threads);
    if (dtype == ME_F32)
      token_shift_fours_kernel<float><<<rows, threads, 0, stream>>>((const float*)x, x_stride, mu, S, state, state_stride, slots, cu, seq_of_token, (float*)out, T, n);
    else
      token_shift_fours_kernel<bf16_t><<<rows, threads, 0, stream>>>((const bf16_t*)x, x_stride, mu, S, state, state_stride, slots, cu, seq_of_token, (bf16_t*)out, T, n);
    ME_LAUNCH_CHECK();
    return 0;
  }
  if (dtype == ME_F32)
    token_shift_kernel<float><<<grid, block, 0, stream>>>((const float*)x, x_stride, mu, S, state, state_stride, slots, cu, seq_of_token, (float*)out, T, n);
  else
    token_shift_kernel<bf16_t><<<grid, block, 0, stream>>>((const bf16_t*)x, x_stride, mu, S, state, state_stride, slots, cu, seq_of_token, (bf16_t*)out, T, n);
  ME_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------------ the recurrence with a decay per state row
// Per request and head a state S [N, P] in float32, walked over the request's tokens of this step in order.
//   RULE 0 (bonus):  d_n = exp(-exp(raw[t, h, n] + base[h, n]));
//                    y_p = sum_n q_n (S[n, p] + bonus[h, n] k_n v_p);   S[n, p] <- d_n S[n, p] + k_n v_p
//   RULE 1 (delta):  d_n = exp(-rate[h] softplus(raw[t, h, n] + base[h, n])),  beta = sigmoid(beta_raw[t, h]);
//                    S[n, p] <- d_n S[n, p];  u_p = beta (v_p - sum_n S[n, p] k_n);  S[n, p] <- S[n, p] + k_n u_p;
//                    y_p = sum_n S[n, p] q_n
//   RULE 2 (gated):  d_n = sigmoid(raw[t, h, n] + base[h, n]) ^ rate[h] = exp(-rate[h] softplus(-(raw + base)));
//                    S[n, p] <- d_n S[n, p] + k_n v_p;   y_p = sum_n S[n, p] q_n
//   RULE 3 (delta_head): RULE 1 with one decay per head and token, d = exp(-rate[h] softplus(raw[t, h] + base[h])): the
//                    decay then needs no LDS and multiplies a lane's rows from a register
// With `unit`: q and k are first divided by sqrt(sum of their squares + unit_eps) per head; q is multiplied by q_scale.
// Every sum runs over n only, so a column p of the state never meets another: a wave takes 64 / RG columns of one head
// and a lane NR / RG of a column's rows, kept in registers for the whole walk; with RG > 1 the RG lanes of a column,
// neighbours in the wave, add their partial sums by exchanges inside a row of 16 lanes. q, k and the decays of a token, which all columns share, are
// formed once per wave in LDS, eight tokens at a time into one of two buffers; the next eight tokens' raw values are on
// their way while the current eight are worked on, so a wave waits for memory once per eight tokens. The products
// and sums of the walk are written as explicit fused multiply-adds: a token's result then does not depend on its place
// among the eight (the compiler is free to fuse each unrolled copy otherwise).
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

#define DR_TB 8          // tokens whose shared values are formed at once and wait in LDS

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

// One wave per (token, head): the shaped values of every token at once, for a recurrence kernel that then only streams
// them (decay_walk_kernel): pre_q, pre_k, pre_d [T, H, NR] and pre_x [T, H], float32. The rows of a (token, head) lie in the
// order in which that kernel's lanes take them (walk_place).
// Lane rg of the RG lanes of a column keeps rows rg, rg + RG, ...: its i-th row lies among the i / 4-th four of all lanes, so that
// the lanes of a column read 16-byte pieces side by side (a lane's rows in one run met each bank RL / 4 times: 128 rows over 16
// lanes, 44 % of the LDS cycles).
template <int NR, int RG>
__host__ __device__ constexpr int walk_place(int rg, int i) {
  constexpr int RL = NR / RG;
  return RL < 4 ? rg * RL + i : i / 4 * (RG * 4) + rg * 4 + i % 4;
}
template <typename TX, int NR, int RULE>
__global__ void __launch_bounds__(64) decay_prepare_kernel(DrArgs a, int row_groups, float* __restrict__ pre_q, float* __restrict__ pre_k,
                                                           float* __restrict__ pre_d, float* __restrict__ pre_x) {
  constexpr int PER = (NR + 63) / 64;
  const int64_t t = blockIdx.x;
  const int h = blockIdx.y, lane = threadIdx.x;
  const int g = h / (a.H / a.G);
  const TX* qp = (const TX*)a.q; const TX* kp = (const TX*)a.k; const TX* rp = (const TX*)a.raw; const TX* bp = (const TX*)a.beta;
  float q[PER], k[PER], d[PER], base[PER], bonus[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int n = lane + 64 * i;
    const bool in = n < a.N && n < NR;
    base[i] = RULE == 3 ? a.base[h] : (in ? a.base[h * a.N + n] : 0.f);
    bonus[i] = (RULE == 0 && in) ? a.bonus[h * a.N + n] : 0.f;
    q[i] = in ? to_f32<TX>(qp[t * a.q_stride + g * a.N + n]) : 0.f;
    k[i] = in ? to_f32<TX>(kp[t * a.k_stride + g * a.N + n]) : 0.f;
    d[i] = RULE == 3 ? to_f32<TX>(rp[t * a.raw_stride + h]) : (in ? to_f32<TX>(rp[t * a.raw_stride + h * a.N + n]) : 0.f);
  }
  const float beta = (RULE == 1 || RULE == 3) ? to_f32<TX>(bp[t * a.beta_stride + h]) : 0.f;
  const float x = shape_token<PER, RULE>(a, lane, NR, q, k, d, base, bonus, RULE != 0 ? a.rate[h] : 0.f, beta);
  // each lane takes the value that belongs in its place, so that a wave's stores are whole lines
  const int64_t at = (t * a.H + h) * NR;
  const int from = row_groups == 16 ? (NR == 32 ? lane % 2 * 16 + lane / 2 : lane % 4 * 16 + lane / 4) : (lane & ~15) + lane % 4 * 4 + lane / 4 % 4;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const float qv = __shfl(q[i], from), kv = __shfl(k[i], from), dv = RULE == 3 ? 0.f : __shfl(d[i], from);
    const int64_t to = at + lane + 64 * i;
    if (lane + 64 * i < NR) {
      pre_q[to] = qv; pre_k[to] = kv;
      if (RULE != 3) pre_d[to] = dv;
    }
  }
  if (lane == 0) {
    pre_x[t * a.H + h] = x;
    if (RULE == 3) pre_d[t * a.H + h] = d[0];
  }
}

template <typename TX, int NR, int RG, int RULE>
__global__ void __launch_bounds__(64) decay_rows_kernel(DrArgs a) {
  constexpr int PC = 64 / RG;            // columns per wave
  constexpr int RL = NR / RG;            // rows per lane
  constexpr int PER = (NR + 63) / 64;    // rows of q, k and the decay that a lane brings to LDS for the wave
  __shared__ float sq[2][DR_TB][NR], sk[2][DR_TB][NR], sd[2][RULE == 3 ? 1 : DR_TB][RULE == 3 ? 1 : NR];
  const int lane = threadIdx.x;
  const int col_blocks = (a.P + PC - 1) / PC;
  const int cb = blockIdx.x % col_blocks;
  const int h = (blockIdx.x / col_blocks) % a.H;
  const int b = blockIdx.x / (col_blocks * a.H);
  const int g = h / (a.H / a.G);
  const int64_t first = a.cu[b];
  const int n_tok = (int)(a.cu[b + 1] - first);
  if (n_tok <= 0) return;
  // the RG lanes of a column are neighbours; lane rg of them keeps rows rg, rg + RG, ... (neighbours read neighbouring
  // words of LDS, the lanes of the wave's other columns the same words)
  const int p = cb * PC + lane / RG;
  const int rg = lane % RG;
  const bool live = p < a.P;
  const int pc = live ? p : a.P - 1;
  float* srow = a.state + (int64_t)a.slots[b] * a.state_stride + (int64_t)h * a.N * a.P;
  float S[RL];
#pragma unroll
  for (int i = 0; i < RL; ++i) S[i] = (i * RG + rg < a.N) ? srow[(int64_t)(i * RG + rg) * a.P + pc] : 0.f;

  const TX* qp = (const TX*)a.q; const TX* kp = (const TX*)a.k; const TX* vp = (const TX*)a.v;
  const TX* rp = (const TX*)a.raw; const TX* bp = (const TX*)a.beta;
  float base[PER], bonus[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int n = lane + 64 * i;
    const bool in = n < a.N && n < NR;
    base[i] = RULE == 3 ? a.base[h] : (in ? a.base[h * a.N + n] : 0.f);
    bonus[i] = (RULE == 0 && in) ? a.bonus[h * a.N + n] : 0.f;
  }
  const float rate = RULE != 0 ? a.rate[h] : 0.f;
  // a batch of tokens on its way (n*) and the batch being worked on (c*): a lane's own column's v and the token's own
  // number (the write strength, or under the bonus rule sum_n q_n bonus_n k_n)
  float nq[DR_TB][PER], nk[DR_TB][PER], nr[DR_TB][PER], nv[DR_TB], nb[DR_TB];
  float cv[DR_TB], cx[DR_TB], cd[DR_TB];        // cd: the token's decay (RULE 3)
  auto fetch = [&](int t0) {
#pragma unroll
    for (int j = 0; j < DR_TB; ++j) {
      if (t0 + j < n_tok) {
        const int64_t row = first + t0 + j;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          const int n = lane + 64 * i;
          const bool in = n < a.N && n < NR;
          nq[j][i] = in ? to_f32<TX>(qp[row * a.q_stride + g * a.N + n]) : 0.f;
          nk[j][i] = in ? to_f32<TX>(kp[row * a.k_stride + g * a.N + n]) : 0.f;
          if (RULE == 3) nr[j][i] = i == 0 ? to_f32<TX>(rp[row * a.raw_stride + h]) : 0.f;
          else nr[j][i] = in ? to_f32<TX>(rp[row * a.raw_stride + h * a.N + n]) : 0.f;
        }
        nv[j] = to_f32<TX>(vp[row * a.v_stride + h * a.P + pc]);
        nb[j] = (RULE == 1 || RULE == 3) ? to_f32<TX>(bp[row * a.beta_stride + h]) : 0.f;
      }
    }
  };
  // the fetched batch's shared values into LDS buffer `buf`, its per-lane values into c*
  auto settle = [&](int t0, int buf) {
#pragma unroll
    for (int j = 0; j < DR_TB; ++j) {
      if (t0 + j < n_tok) {
        const float x = shape_token<PER, RULE>(a, lane, NR, nq[j], nk[j], nr[j], base, bonus, rate, nb[j]);
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          const int n = lane + 64 * i;
          // row n belongs to lane n % RG of a column as its row n / RG: a lane's rows lie side by side in LDS, so that it
          // reads them four at a time
          const int at = (n % RG) * RL + n / RG;
          if (n < NR) {
            sq[buf][j][at] = nq[j][i]; sk[buf][j][at] = nk[j][i];
            if (RULE != 3) sd[buf][j][at] = nr[j][i];
          }
        }
        cd[j] = nr[j][0];
        cv[j] = nv[j];
        cx[j] = x;
      }
    }
  };
  fetch(0);
  for (int t0 = 0, buf = 0; t0 < n_tok; t0 += DR_TB, buf ^= 1) {
    settle(t0, buf);
    __syncthreads();      // the batch is in LDS; the other buffer, which the next batch will take, has been read by all
    if (t0 + DR_TB < n_tok) fetch(t0 + DR_TB);
#pragma unroll
    for (int j = 0; j < DR_TB; ++j) {
      if (t0 + j < n_tok) {
        const float v = cv[j];
        float y = 0.f;
        if (RULE == 0) {
#pragma unroll
          for (int i = 0; i < RL; ++i) {
            const int n = rg * RL + i;
            y = fmaf(sq[buf][j][n], S[i], y);
            S[i] = fmaf(sd[buf][j][n], S[i], sk[buf][j][n] * v);
          }
        } else if (RULE == 2) {
#pragma unroll
          for (int i = 0; i < RL; ++i) {
            const int n = rg * RL + i;
            S[i] = fmaf(sd[buf][j][n], S[i], sk[buf][j][n] * v);
            y = fmaf(sq[buf][j][n], S[i], y);
          }
        } else {
          float dot = 0.f;
#pragma unroll
          for (int i = 0; i < RL; ++i) {
            const int n = rg * RL + i;
            S[i] *= RULE == 3 ? cd[j] : sd[buf][j][n];
            dot = fmaf(S[i], sk[buf][j][n], dot);
          }
          dot = group_sum<RG>(dot);
          const float u = cx[j] * (v - dot);
#pragma unroll
          for (int i = 0; i < RL; ++i) {
            const int n = rg * RL + i;
            S[i] = fmaf(sk[buf][j][n], u, S[i]);
            y = fmaf(S[i], sq[buf][j][n], y);
          }
        }
        y = group_sum<RG>(y);
        if (RULE == 0) y = fmaf(cx[j], v, y);       // the current token's own term: v_p * sum_n q_n bonus_n k_n
        if (live && rg == 0) a.y[(first + t0 + j) * (int64_t)(a.H * a.P) + h * a.P + p] = y;
      }
    }
  }
  if (live) {
#pragma unroll
    for (int i = 0; i < RL; ++i)
      if (i * RG + rg < a.N) srow[(int64_t)(i * RG + rg) * a.P + p] = S[i];
  }
}

// The same walk over values that decay_prepare_kernel has shaped: portions of many tokens. What bounds it is the number of
// instructions of a wave per token (a request's tokens are a chain, and the chip has few waves per SIMD, each of which issues an instruction
// in four cycles), so a batch of eight tokens is one piece of code without a branch: the exchange
// and the output sum of a token overlap the next token's reads and updates, and shared values are brought in 16-byte pieces that
// go to LDS as they are. The sums are those of decay_rows_kernel in the same order.
template <typename TX, int NR, int RG, int RULE>
__device__ __forceinline__ void walk_alone(const DrArgs& a, const float* __restrict__ pre_q, const float* __restrict__ pre_k,
                                           const float* __restrict__ pre_d, const float* __restrict__ pre_x) {
  constexpr int TB = DR_TB;
  constexpr int AHEAD = NR <= 64 ? 3 : NR <= 128 ? 2 : 1;    // tokens whose shared values are read from LDS ahead
  constexpr int PC = 64 / RG;            // columns per wave
  constexpr int RL = NR / RG;            // rows per lane
  constexpr int PIECES = TB * NR / 4; // 16-byte pieces of a batch's q, k or decays
  constexpr int ROUNDS = (PIECES + 63) / 64;
  constexpr int VALUES = TB * PC, VROUNDS = (VALUES + 63) / 64;
  constexpr bool ROWS = RULE != 3;
  constexpr bool SHARED_V = NR <= 128;   // the columns' values go through LDS too; with 256 rows a lane asks for its own
  // A lane that holds 64 rows has no registers left over: the last batch shares the code around the others and the loads of a
  // batch's values their addresses (63 registers spilled otherwise, 32 so: 16 prompts of 512 tokens over 4 heads of 256 x 64, bonus rule
  // 463 -> 415 us, delta rule 529 -> 512); elsewhere a wave is level or slower with it (16 lanes to a column, delta rule 167 / 190).
  constexpr bool TIGHT = NR / RG > 32;
  __shared__ f32x4 sq[2][PIECES], sk[2][PIECES], sd[ROWS ? 2 : 1][ROWS ? PIECES : 1];
  __shared__ __align__(16) float sv[2][SHARED_V ? VALUES : 1];              // [column][token]
  __shared__ float sx[2][TB], sh[2][TB];               // the tokens' own numbers; their heads' decays (RULE 3)
  const int lane = threadIdx.x;
  const int col_blocks = (a.P + PC - 1) / PC;
  const int cb = blockIdx.x % col_blocks;
  const int h = (blockIdx.x / col_blocks) % a.H;
  const int b = blockIdx.x / (col_blocks * a.H);
  const int begin = __builtin_amdgcn_readfirstlane(a.cu[b]);
  const int n_tok = __builtin_amdgcn_readfirstlane(a.cu[b + 1]) - begin;
  if (n_tok <= 0) return;
  const int64_t first = begin;
  const int p = cb * PC + lane / RG;
  const int rg = lane % RG;
  const bool live = p < a.P;
  const int pc = live ? p : a.P - 1;
  float* srow = a.state + (int64_t)a.slots[b] * a.state_stride + (int64_t)h * a.N * a.P;
  float S[RL];
#pragma unroll
  for (int i = 0; i < RL; ++i) S[i] = (i * RG + rg < a.N) ? srow[(int64_t)(i * RG + rg) * a.P + pc] : 0.f;

  const TX* values = (const TX*)a.v + first * a.v_stride + h * a.P;
  const int64_t head0 = first * a.H + h;
  f32x4 nq[ROUNDS], nk[ROUNDS], nd[ROUNDS];
  float nx = 0.f, nh = 0.f;
  TX nv[SHARED_V ? VROUNDS : TB];
  // what a lane adds to a batch's first address, in bytes (the address itself is the same for all lanes)
  uint32_t piece[ROUNDS];
  int column[VROUNDS];                                       // of a value that a thread brings, and its place in sv
  int place[VROUNDS];
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int e = min(lane + 64 * r, PIECES - 1);
    piece[r] = (uint32_t)((e / (NR / 4) * a.H * (NR / 4) + e % (NR / 4)) * 16);
  }
#pragma unroll
  for (int r = 0; r < VROUNDS; ++r) {
    const int e = min(lane + 64 * r, VALUES - 1);
    column[r] = min(cb * PC + e % PC, a.P - 1);
    place[r] = e % PC * TB + e / PC;
  }
  const int my_token = lane & (TB - 1);
  const uint32_t own = (uint32_t)(my_token * a.H * 4);
  auto at = [](const void* base, uint32_t bytes) { return reinterpret_cast<const char*>(base) + bytes; };
  // the next batch on its way; of a batch that is not whole, tokens behind the last are read from the last one and not used
  auto fetch = [&](int t0) {
    if (!TIGHT && t0 >= n_tok) return;
    if (SHARED_V) {
#pragma unroll
      for (int r = 0; r < VROUNDS; ++r)
        nv[r] = values[(int64_t)min(t0 + min(lane + 64 * r, VALUES - 1) / PC, n_tok - 1) * a.v_stride + column[r]];
    } else if (!TIGHT) {
#pragma unroll
      for (int j = 0; j < TB; ++j) nv[j] = values[(int64_t)min(t0 + j, n_tok - 1) * a.v_stride + pc];
    }
    if (t0 + TB <= n_tok) {
      const int64_t row = head0 + (int64_t)t0 * a.H;
#pragma unroll
      for (int r = 0; r < ROUNDS; ++r) {
        nq[r] = *reinterpret_cast<const f32x4*>(at(pre_q + row * NR, piece[r]));
        nk[r] = *reinterpret_cast<const f32x4*>(at(pre_k + row * NR, piece[r]));
        if (ROWS) nd[r] = *reinterpret_cast<const f32x4*>(at(pre_d + row * NR, piece[r]));
      }
      nx = *reinterpret_cast<const float*>(at(pre_x + row, own));
      if (!ROWS) nh = *reinterpret_cast<const float*>(at(pre_d + row, own));
      if (TIGHT) {
        const TX* vt = values + t0 * a.v_stride;
#pragma unroll
        for (int j = 0; j < TB; ++j, vt += a.v_stride) nv[j] = *reinterpret_cast<const TX*>(at(vt, (uint32_t)(pc * sizeof(TX))));
      }
      return;
    }
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
      const int e = min(lane + 64 * r, PIECES - 1);
      const int64_t from = (head0 + (int64_t)min(t0 + e / (NR / 4), n_tok - 1) * a.H) * NR + e % (NR / 4) * 4;
      nq[r] = *reinterpret_cast<const f32x4*>(pre_q + from);
      nk[r] = *reinterpret_cast<const f32x4*>(pre_k + from);
      if (ROWS) nd[r] = *reinterpret_cast<const f32x4*>(pre_d + from);
    }
    const int64_t row = head0 + (int64_t)min(t0 + my_token, n_tok - 1) * a.H;
    nx = pre_x[row];
    if (!ROWS) nh = pre_d[row];
    if (TIGHT) {
#pragma unroll
      for (int j = 0; j < TB; ++j) nv[j] = values[(int64_t)min(t0 + j, n_tok - 1) * a.v_stride + pc];
    }
  };
  struct Shared { float q[RL], k[RL], d[RL], x; };
  auto read = [&](int buf, int j, Shared& o) {
    const float* aq = reinterpret_cast<const float*>(&sq[buf][0]) + j * NR + walk_place<NR, RG>(rg, 0);
    const float* ak = reinterpret_cast<const float*>(&sk[buf][0]) + j * NR + walk_place<NR, RG>(rg, 0);
    const float* ad = reinterpret_cast<const float*>(&sd[ROWS ? buf : 0][0]) + j * NR + walk_place<NR, RG>(rg, 0);
#pragma unroll
    for (int i = 0; i < RL; ++i) {
      const int e = walk_place<NR, RG>(0, i);
      o.q[i] = aq[e];
      o.k[i] = ak[e];
      if (ROWS) o.d[i] = ad[e];
    }
    if (!ROWS) o.d[0] = sh[buf][j];
    o.x = RULE == 2 ? 0.f : sx[buf][j];
  };
  // the state behind a token and the token's output
  auto token = [&](const Shared& o, float v) {
    float y = 0.f;
    if (RULE == 0) {
#pragma unroll
      for (int i = 0; i < RL; ++i) {
        y = fmaf(o.q[i], S[i], y);
        S[i] = fmaf(o.d[i], S[i], o.k[i] * v);
      }
    } else if (RULE == 2) {
#pragma unroll
      for (int i = 0; i < RL; ++i) {
        S[i] = fmaf(o.d[i], S[i], o.k[i] * v);
        y = fmaf(o.q[i], S[i], y);
      }
    } else {
      float dot = 0.f;
#pragma unroll
      for (int i = 0; i < RL; ++i) {
        S[i] *= o.d[ROWS ? i : 0];
        dot = fmaf(S[i], o.k[i], dot);
      }
      dot = group_sum<RG>(dot);
      const float u = o.x * (v - dot);
#pragma unroll
      for (int i = 0; i < RL; ++i) {
        S[i] = fmaf(o.k[i], u, S[i]);
        y = fmaf(S[i], o.q[i], y);
      }
    }
    y = group_sum<RG>(y);
    if (RULE == 0) y = fmaf(o.x, v, y);          // the current token's own term: v_p * sum_n q_n bonus_n k_n
    return y;
  };
  float* out = a.y + first * (int64_t)(a.H * a.P) + h * a.P + p;
  int t0 = 0, buf = 0;
  // the batch that has come goes to LDS, the next one is asked for, and the columns' values of the batch are read
  auto next_batch = [&](float (&v)[TB]) {
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
      const int e = lane + 64 * r;
      if (PIECES % 64 == 0 || e < PIECES) {
        sq[buf][e] = nq[r]; sk[buf][e] = nk[r];
        if (ROWS) sd[ROWS ? buf : 0][e] = nd[r];
      }
    }
    if (!SHARED_V) {
#pragma unroll
      for (int j = 0; j < TB; ++j) v[j] = to_f32<TX>(nv[j]);
    } else
#pragma unroll
    for (int r = 0; r < VROUNDS; ++r)
      if (VALUES % 64 == 0 || lane + 64 * r < VALUES) sv[buf][place[r]] = to_f32<TX>(nv[r]);
    if (lane < TB) {
      sx[buf][lane] = nx;
      if (!ROWS) sh[buf][lane] = nh;
    }
    asm volatile("" ::: "memory");
    fetch(t0 + TB);
    asm volatile("" ::: "memory");         // (one wave needs no barrier: what its lanes write to LDS, its lanes read behind it)
    if (SHARED_V) {
#pragma unroll
      for (int j = 0; j < TB; ++j) v[j] = sv[buf][lane / RG * TB + j];
    }
  };
// a last batch that is not whole (no lambda: the choice of a value would become an address, and v memory)
#define DR_LAST_BATCH                                             \
  _Pragma("unroll 1") for (int j = 0; t0 + j < n_tok; ++j) {      \
    Shared o;                                                     \
    read(buf, j, o);                                              \
    float vj = v[0];                                              \
    _Pragma("unroll") for (int i = 1; i < TB; ++i) vj = i == j ? v[i] : vj; \
    const float y = token(o, vj);                                 \
    if (live && rg == 0) out[(int64_t)(t0 + j) * (a.H * a.P)] = y; \
  }
  fetch(0);
  for (; t0 + (TIGHT ? 1 : TB) <= n_tok; t0 += TB, buf ^= 1) {
    float v[TB], y[TB];
    next_batch(v);
    if (TIGHT && t0 + TB > n_tok) {
      DR_LAST_BATCH
      continue;
    }
    Shared o[AHEAD + 1];                         // a token's values are read while those before it are worked on
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) read(buf, j, o[j]);
#pragma unroll
    for (int j = 0; j < TB; ++j) {
      if (j + AHEAD < TB) read(buf, j + AHEAD, o[(j + AHEAD) % (AHEAD + 1)]);
      y[j] = token(o[j % (AHEAD + 1)], v[j]);
    }
    // the first four lanes of a column hold the same bits (the others have added in another order): lane rg of them stores
    // output i0 + rg
    constexpr int ST = RG < 4 ? RG : 4;
    if (live && rg < ST) {
#pragma unroll
      for (int i0 = 0; i0 < TB; i0 += ST) {
        float mine = y[i0];
#pragma unroll
        for (int i = 1; i < ST; ++i) mine = rg == i ? y[i0 + i] : mine;
        out[(int64_t)(t0 + i0 + rg) * (a.H * a.P)] = mine;
      }
    }
  }
  if (!TIGHT && t0 < n_tok) {
    float v[TB];
    next_batch(v);
    DR_LAST_BATCH
  }
#undef DR_LAST_BATCH
  if (live) {
#pragma unroll
    for (int i = 0; i < RL; ++i)
      if (i * RG + rg < a.N) srow[(int64_t)(i * RG + rg) * a.P + p] = S[i];
  }
}

// 64 x 16 bytes from base + voff (bytes, per lane) to LDS at lds_addr + 16 * lane. The write to m0 needs one wait
// state before an instruction that reads it for an LDS address.
__device__ __forceinline__ void walk_request(uint32_t lds_addr, uint32_t voff, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voff), "s"(base) : "memory");
}

// The walk where compute units are left over: four waves hold the same four columns: each of them carries the state through every
// token, but forms, exchanges and stores the outputs of every fourth only, and brings a quarter of the shared values. What bounds it
// is a wave's instructions for a token, the delta rules' also the sum over the column's lanes, four exchanges of which each waits for the one
// before (152 cycles of a token's 200 at 128 rows); so everything else is kept out of the way. A batch's rows go to LDS past the registers, without
// a branch in front of what is waited for; reads from LDS run seven tokens ahead (three waited for them: 64 rows 157 us for one request of 2,048
// tokens, 109 so) and on into the next batch, behind the one barrier of a batch; the delta rules' reads and an output's exchanges stand between
// the sum's exchanges. With the kernel that shapes the values, 2,048 tokens beside 1,075, against register copies, two barriers' worth of waiting for
// a batch's outputs and values, and reads two or three tokens ahead: delta rule, 4 heads of 128 x 128, 262 -> 227 us, bonus rule, 16 heads of 64 x 64,
// 150 -> 134 (one wave to a column group 344 and 230). Up to 64 rows batches of 32 tokens, held to the registers that let three workgroups onto a
// compute unit (768 workgroups of 1,100 tokens 141 -> 130 us, 512 132 -> 135). What is left of a request behind its whole batches, or all of a
// short one, all four waves walk too, four tokens in a piece (16 heads of 64 x 64, bonus rule, one request of 16 / 31 / 63 / 127 tokens 9.5 / 12.0 / 14.3 /
// 18.5 us by one wave with nothing read ahead, 8.1 / 9.5 / 12.0 / 16.0 so; batches of 16 tokens through registers, which have nothing left of 16, 7.8 / 11.4
// / 13.6 / 18.1), and behind the last batch no rows are asked for (one of 2,048 tokens 118 -> 110 us).
template <typename TX, int NR, int RULE>
__device__ __forceinline__ void walk_shared(const DrArgs& a, const float* __restrict__ pre_q, const float* __restrict__ pre_k,
                                            const float* __restrict__ pre_d, const float* __restrict__ pre_x) {
  constexpr int RG = 16, W = 4, PC = 4, RL = NR / RG;
  constexpr int TB = NR <= 64 ? 32 : 16;      // tokens of a batch
  constexpr int AHEAD = 7;               // tokens whose shared values are read from LDS ahead
  constexpr int PIECES = TB * NR / 4, ROUNDS = (PIECES + 255) / 256;
  constexpr bool ROWS = RULE != 3;
  constexpr bool DELTA = RULE == 1 || RULE == 3;
  constexpr int KINDS = ROWS ? 3 : 2;
  __shared__ f32x4 rows[2][KINDS][PIECES];               // q, k, decays
  __shared__ f32x4 sv[2][PC][TB / 4], sx[2][TB / 4], sh[2][TB / 4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col_blocks = (a.P + PC - 1) / PC;
  const int cb = blockIdx.x % col_blocks;
  const int h = (blockIdx.x / col_blocks) % a.H;
  const int b = blockIdx.x / (col_blocks * a.H);
  const int begin = __builtin_amdgcn_readfirstlane(a.cu[b]);
  const int n_tok = __builtin_amdgcn_readfirstlane(a.cu[b + 1]) - begin;
  if (n_tok <= 0) return;
  const int64_t first = begin;
  const int p = cb * PC + lane / RG;
  const int rg = lane % RG;
  const bool live = p < a.P;
  const int pc = live ? p : a.P - 1;
  float* srow = a.state + (int64_t)a.slots[b] * a.state_stride + (int64_t)h * a.N * a.P;
  float S[RL];
#pragma unroll
  for (int i = 0; i < RL; ++i) S[i] = (i * RG + rg < a.N) ? srow[(int64_t)(i * RG + rg) * a.P + pc] : 0.f;

  // What a thread brings of a batch: pieces of the rows, which go to LDS past the registers; the first threads one column's
  // value of one token each, the third wave's (and the fourth's) one token's number (and decay). Addresses are a batch's own, the same
  // for all lanes, and a lane's bytes behind it; of a batch that is not whole, tokens behind the last are read from the last
  // one and not used.
  const int my_token = tid & (TB - 1), my_column = min(cb * PC + (tid / TB) % PC, a.P - 1);
  TX nv;
  float nx = 0.f;
  const uint32_t rows_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)&rows[0][0][0];
  auto request = [&](int t0, int buf) {
    const bool more = t0 < n_tok;                // (behind the last batch no rows, but the last token's values: a branch around them would wait for nv)
    t0 = min(t0, n_tok - 1);
    const int last = n_tok - 1 - t0;
    const int64_t row = (first + t0) * a.H + h;
    if (more)
#pragma unroll
      for (int r = 0; r < ROUNDS; ++r) {
        const int e0 = 64 * wave + 256 * r;
        if (PIECES % 256 == 0 || e0 < PIECES) {
          const int e = e0 + lane;
          const uint32_t from = (uint32_t)((min(e / (NR / 4), last) * a.H * (NR / 4) + e % (NR / 4)) * 16);
          const uint32_t to = rows_base + (uint32_t)((buf * KINDS * PIECES + e0) * 16);
          walk_request(to, from, pre_q + row * NR);
          walk_request(to + PIECES * 16, from, pre_k + row * NR);
          if (ROWS) walk_request(to + 2 * PIECES * 16, from, pre_d + row * NR);
        }
      }
    const int t = min(my_token, last);
    nv = ((const TX*)a.v + (first + t0) * a.v_stride + h * a.P)[(int64_t)t * a.v_stride + my_column];
    if (RULE != 2) nx = ((!ROWS && wave == 3 ? pre_d : pre_x) + row)[t * a.H];
  };
  // The requested batch is in LDS for all waves behind this, and nobody reads from the other buffer any more.
  auto arrive = [&](int buf) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (wave < TB * PC / 64) reinterpret_cast<float*>(&sv[buf][0][0])[tid] = to_f32<TX>(nv);
    if (wave == 2 && RULE != 2 && lane < TB) reinterpret_cast<float*>(&sx[buf][0])[lane] = nx;
    if (wave == 3 && !ROWS && lane < TB) reinterpret_cast<float*>(&sh[buf][0])[lane] = nx;
    __syncthreads();
  };
  struct Rows { float q[RL], k[RL], d[RL], x; };         // (x: RULE 0's number, which goes to the output)
  struct Numbers { float v[4], x[4], h[4]; };   // of four tokens: the column's value, the delta rules' number and (RULE 3) decay
  auto read_rows = [&](int buf, int j, float (&to)[RL], int kind) {
    const float* f = reinterpret_cast<const float*>(&rows[buf][kind][0]) + j * NR + walk_place<NR, RG>(rg, 0);
#pragma unroll
    for (int i = 0; i < RL; ++i) to[i] = f[walk_place<NR, RG>(0, i)];
  };
  auto read_x = [&](int buf, int j) { return RULE == 0 ? reinterpret_cast<const float*>(&sx[buf][0])[j] : 0.f; };
  auto read_numbers = [&](int buf, int g, Numbers& o) {
    const f32x4 v = sv[buf][lane / RG][g];
    f32x4 x = {0.f, 0.f, 0.f, 0.f}, hh = x;
    if (DELTA) x = sx[buf][g];           // (a register of a read that nobody uses is given away at once, and its next owner waits for the read)
    if (!ROWS) hh = sh[buf][g];
#pragma unroll
    for (int i = 0; i < 4; ++i) { o.v[i] = v[i]; o.x[i] = x[i]; o.h[i] = hh[i]; }
  };
  auto exchange = [&](float y, int step) {
    return y + (step == 0 ? dpp_f<0xB1>(y) : step == 1 ? dpp_f<0x4E>(y) : step == 2 ? dpp_f<0x124>(y) : dpp_f<0x128>(y));
  };
  // One token: the state behind it and, where this wave is to give it, the lane's part of its output. `beside(step)` is what
  // is issued in front of the exchanges of the delta rules' sum, each of which waits for the one before it.
  auto token = [&](const Rows& o, float v, float x, float hd, bool reads_out, auto beside) {
    float y = 0.f;
    if (!DELTA) {
      beside(0); beside(1); beside(2); beside(3);
#pragma unroll
      for (int i = 0; i < RL; ++i) {
        if (RULE == 0 && reads_out) y = fmaf(o.q[i], S[i], y);
        S[i] = fmaf(o.d[i], S[i], o.k[i] * v);
        if (RULE == 2 && reads_out) y = fmaf(o.q[i], S[i], y);
      }
    } else {
      float dot = 0.f;
#pragma unroll
      for (int i = 0; i < RL; ++i) {
        S[i] *= ROWS ? o.d[i] : hd;
        dot = fmaf(S[i], o.k[i], dot);
      }
#pragma unroll
      for (int step = 0; step < 4; ++step) {
        __builtin_amdgcn_sched_barrier(0);
        beside(step);
        __builtin_amdgcn_sched_barrier(0);
        dot = exchange(dot, step);
      }
      const float u = x * (v - dot);
#pragma unroll
      for (int i = 0; i < RL; ++i) {
        S[i] = fmaf(o.k[i], u, S[i]);
        if (reads_out) y = fmaf(S[i], o.q[i], y);
      }
    }
    return y;
  };
  float* out = a.y + first * (int64_t)(a.H * a.P) + h * a.P;
  int t0 = 0, buf = 0;
  request(0, 0);
  arrive(0);
  if (TB < n_tok) request(TB, 1);
  auto walk = [&](auto which) {                  // the whole batches; this wave gives the outputs of tokens ME, ME + W, ... of each
    constexpr int ME = decltype(which)::value;
    if (TB > n_tok) return;
    Rows o[AHEAD + 1];
    Numbers num[2];                              // of the four tokens under way and the next four
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      read_rows(0, j, o[j].k, 1);
      if (ROWS) read_rows(0, j, o[j].d, 2);
      if (j % W == ME) read_rows(0, j, o[j].q, 0), o[j].x = read_x(0, j);
    }
    read_numbers(0, 0, num[0]);
    const uint32_t to_mine = (uint32_t)((ME + W * rg) * (a.H * a.P) + p);
    for (; t0 + TB <= n_tok; t0 += TB, buf ^= 1) {
      float y[4], part = 0.f;
#pragma unroll
      for (int j = 0; j < TB; ++j) {
        if (j == TB - AHEAD) {                   // from here on the next batch is read
          arrive(buf ^ 1);
          request(t0 + 2 * TB, buf);
        }
        const int from = j + AHEAD < TB ? buf : buf ^ 1, jn = (j + AHEAD) % TB;
        Rows& next = o[(j + AHEAD) % (AHEAD + 1)];
        const bool waits = DELTA && j % 16 > 0 && (j - 1) % W == ME;     // an output whose exchanges go beside this token's
        const Numbers& n = num[j / 4 % 2];
        const float yj = token(o[j % (AHEAD + 1)], n.v[j % 4], n.x[j % 4], n.h[j % 4], j % W == ME, [&](int step) {
          if (step == 1) read_rows(from, jn, next.k, 1);
          if (step == 2 && ROWS) read_rows(from, jn, next.d, 2);
          if (step == 3 && jn % W == ME) read_rows(from, jn, next.q, 0), next.x = read_x(from, jn);
          if (step == (ROWS ? 3 : 2) && j % 4 == 0) read_numbers(j + 4 < TB ? buf : buf ^ 1, (j / 4 + 1) % (TB / 4), num[(j / 4 + 1) % 2]);
          asm volatile("" ::: "memory");         // the reads stay here (the compiler would sink them to where they are used)
          if (waits) part = exchange(part, step);
        });
        if (waits) y[(j - 1) / W % 4] = part;
        if (j % W == ME) {
          part = yj;
          if (!DELTA || j % 16 == 15) {
            part = group_sum<RG>(part);
            if (RULE == 0) part = fmaf(o[j % (AHEAD + 1)].x, n.v[j % 4], part);   // the token's own term: v_p * sum_n q_n bonus_n k_n
            y[j / W % 4] = part;
          }
        }
        // the first four lanes of a column hold the same bits (the others have added in another order): lane rg of them stores
        // the wave's output rg of sixteen tokens
        if (j % 16 == 15) {
          float mine = y[0];
#pragma unroll
          for (int i = 1; i < 4; ++i) mine = rg == i ? y[i] : mine;
          if (live && rg < 4) (out + (int64_t)(t0 + j - 15) * (a.H * a.P))[to_mine] = mine;
        }
      }
    }
  };
  if (wave == 0) walk(std::integral_constant<int, 0>{});
  else if (wave == 1) walk(std::integral_constant<int, 1>{});
  else if (wave == 2) walk(std::integral_constant<int, 2>{});
  else walk(std::integral_constant<int, 3>{});
  // A last batch that is not whole, which lies in LDS, four tokens at a time, whose rows are read while the four before them are
  // worked on; each wave gives the output of one of the four. (Rows behind the last token are there, and not used.)
  auto rest = [&](auto which) {
    constexpr int ME = decltype(which)::value;
    const int left = n_tok - t0;
    if (left <= 0) return;
    struct Four { float k[4][RL], d[4][RL], q[RL], x; };
    Four f[2];
    Numbers num[2];
    auto read_four = [&](int g, Four& o, Numbers& n) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        read_rows(buf, 4 * g + j, o.k[j], 1);
        if (ROWS) read_rows(buf, 4 * g + j, o.d[j], 2);
      }
      read_rows(buf, 4 * g + ME, o.q, 0);
      o.x = read_x(buf, 4 * g + ME);
      read_numbers(buf, g, n);
    };
    auto four = [&](int g, const Four& o, const Numbers& n) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (4 * g + j >= left) return;
        Rows r;
#pragma unroll
        for (int i = 0; i < RL; ++i) { r.k[i] = o.k[j][i]; if (ROWS) r.d[i] = o.d[j][i]; r.q[i] = o.q[i]; }
        float y = token(r, n.v[j], n.x[j], n.h[j], j == ME, [](int) {});
        if (j != ME) continue;
        y = group_sum<RG>(y);
        if (RULE == 0) y = fmaf(o.x, n.v[j], y);
        if (live && rg == 0) (out + (int64_t)(t0 + 4 * g + j) * (a.H * a.P))[p] = y;
      }
    };
    read_four(0, f[0], num[0]);
#pragma unroll 1
    for (int g = 0; 4 * g < left; g += 2) {
      read_four(g + 1, f[1], num[1]);
      asm volatile("" ::: "memory");
      four(g, f[0], num[0]);
      read_four(min(g + 2, TB / 4 - 1), f[0], num[0]);
      asm volatile("" ::: "memory");
      four(g + 1, f[1], num[1]);
    }
  };
  if (wave == 0) rest(std::integral_constant<int, 0>{});
  else if (wave == 1) rest(std::integral_constant<int, 1>{});
  else if (wave == 2) rest(std::integral_constant<int, 2>{});
  else rest(std::integral_constant<int, 3>{});
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // no request outlives its workgroup's LDS
  if (wave != 0) return;
  if (live) {
#pragma unroll
    for (int i = 0; i < RL; ++i)
      if (i * RG + rg < a.N) srow[(int64_t)(i * RG + rg) * a.P + p] = S[i];
  }
}

// W: the waves that hold a column group, one or four.
template <typename TX, int NR, int RG, int RULE, int W>
__global__ void __launch_bounds__(64 * W, W == 1 ? 1 : NR <= 64 ? 3 : 2) decay_walk_kernel(DrArgs a, const float* __restrict__ pre_q, const float* __restrict__ pre_k,
                                                                                           const float* __restrict__ pre_d, const float* __restrict__ pre_x) {
  if constexpr (W == 1) walk_alone<TX, NR, RG, RULE>(a, pre_q, pre_k, pre_d, pre_x);
  else walk_shared<TX, NR, RULE>(a, pre_q, pre_k, pre_d, pre_x);
}

// Workgroups up to which four waves share the walk of a column group: as many as are in flight at once by their LDS and registers, three
// to a compute unit up to 64 rows, two of 128. us with the kernel that shapes the values, requests of 1,100 tokens, one wave / four, bonus and
// delta rule: 64 rows, 512 workgroups 122 / 94 and 162 / 140, 768 146 / 126 and 185 / 185, 832 157 / 157 and 193 / 228; 128 rows, 256
// workgroups 150 / 104 and 179 / 139, 384 167 / 134 and 197 / 181, 512 169 / 144 and 202 / 199, 576 197 / 206 and 242 / 276. With 256 rows
// the batches' LDS leaves no room for longer ones, and without them four waves gain nothing (624 / 650). Of 128 rows requests of
// fewer than 64 tokens on average (`mean`) share up to 256 workgroups (384 of them, bonus rule, 16 tokens 11.3 / 12.4, 32 14.2 / 14.9, 48 17.1 /
// 17.2, 64 20.2 / 19.8, 95 27.2 / 24.9).
template <int NR> static unsigned dr_shared_max(int64_t mean) { return NR <= 64 ? 768 : NR > 128 ? 0 : mean >= 64 ? 512 : 256; }
template <typename TX, int NR, int RG, bool PRE>
static void launch_decay_rows(const DrArgs& a, int rule, int num_seqs, int64_t T, float* pre, hipStream_t stream) {
  constexpr int PC = 64 / RG;
  const dim3 grid((unsigned)(num_seqs * a.H * ((a.P + PC - 1) / PC))), block(64);
  if constexpr (PRE) {
    const int64_t each = T * a.H * NR;
    float *pq = pre, *pk = pre + each, *pd = pre + 2 * each, *px = pre + 3 * each;
    const dim3 pgrid((unsigned)T, a.H);
#define DR_RULE(R)                                                                       \
  do {                                                                                   \
    decay_prepare_kernel<TX, NR, R><<<pgrid, block, 0, stream>>>(a, RG, pq, pk, pd, px); \
    constexpr bool SHARES = RG == 16 && NR <= 128;                                       \
    if (SHARES && grid.x <= dr_shared_max<NR>(T / num_seqs) && (int64_t)a.H * a.P < (1 << 27))       \
      decay_walk_kernel<TX, NR, RG, R, SHARES ? 4 : 1><<<grid, SHARES ? 256 : 64, 0, stream>>>(a, pq, pk, pd, px); \
    else decay_walk_kernel<TX, NR, RG, R, 1><<<grid, block, 0, stream>>>(a, pq, pk, pd, px); \
  } while (0)
    if (rule == 0) DR_RULE(0); else if (rule == 1) DR_RULE(1); else if (rule == 2) DR_RULE(2); else DR_RULE(3);
#undef DR_RULE
  } else {
    if (rule == 0) decay_rows_kernel<TX, NR, RG, 0><<<grid, block, 0, stream>>>(a);
    else if (rule == 1) decay_rows_kernel<TX, NR, RG, 1><<<grid, block, 0, stream>>>(a);
    else if (rule == 2) decay_rows_kernel<TX, NR, RG, 2><<<grid, block, 0, stream>>>(a);
    else decay_rows_kernel<TX, NR, RG, 3><<<grid, block, 0, stream>>>(a);
  }
}

// row_groups: lanes that share a column: 1 or 4 (4 gives four times the waves with a quarter of the rows each) with the
// tokens' values shaped inside the kernel; 4 or 16 with `pre`, scratch of 3 T H NR + T H floats (NR: N rounded up to 32, 64,
// 128 or 256) that a first kernel fills with the shaped values of all tokens at once, so that the walk only streams them.
extern "C" int me_decay_rows_recurrence(const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v, int64_t v_stride,
                                        const void* raw, int64_t raw_stride, const void* beta, int64_t beta_stride, int dtype,
                                        const float* base, const float* rate, const float* bonus, float* state, int64_t state_stride,
                                        const int32_t* slots, const int32_t* cu, float* y, int num_seqs, int H, int G, int N, int P,
                                        int rule, int unit, float unit_eps, float q_scale, int row_groups, int64_t T, float* pre, hipStream_t stream) {
  if (num_seqs == 0) return 0;
  ME_CHECK(H >= 1 && G >= 1 && H % G == 0 && N >= 1 && N <= 256 && P >= 1, "decay_rows_recurrence: %d heads over %d groups, state %d x %d "
           "(up to 256 rows)", H, G, N, P);
  ME_CHECK(rule >= 0 && rule <= 3, "decay_rows_recurrence: unknown rule %d", rule);
  ME_CHECK(rule == 0 ? bonus != nullptr : (rate != nullptr && (rule == 2 || beta != nullptr)), "decay_rows_recurrence: the rule's constants are missing");
  ME_CHECK(pre == nullptr ? (row_groups == 1 || row_groups == 4) : (row_groups == 4 || row_groups == 16),
           "decay_rows_recurrence: 1 or 4 lanes to a column, 4 or 16 over prepared values");
  ME_CHECK(T >= 0 && T <= 2147483647ll && H <= 65535, "decay_rows_recurrence: too many tokens or heads");
  ME_CHECK((int64_t)num_seqs * H * ((P + 3) / 4) <= 2147483647ll && H <= 65535 && P <= (1 << 28), "decay_rows_recurrence: too many workgroups");
  DrArgs a;
  a.q = q; a.k = k; a.v = v; a.raw = raw; a.beta = beta;
  a.q_stride = q_stride; a.k_stride = k_stride; a.v_stride = v_stride; a.raw_stride = raw_stride; a.beta_stride = beta_stride;
  a.base = base; a.rate = rate; a.bonus = bonus; a.state = state; a.state_stride = state_stride; a.slots = slots; a.cu = cu; a.y = y;
  a.H = H; a.G = G; a.N = N; a.P = P; a.unit = unit; a.unit_eps = unit_eps; a.q_scale = q_scale;
#define DR_NR(TX, NR)                                                           \
  do {                                                                          \
    if (pre != nullptr && row_groups == 16) launch_decay_rows<TX, NR, 16, true>(a, rule, num_seqs, T, pre, stream); \
    else if (pre != nullptr) launch_decay_rows<TX, NR, 4, true>(a, rule, num_seqs, T, pre, stream);                 \
    else if (row_groups == 4) launch_decay_rows<TX, NR, 4, false>(a, rule, num_seqs, T, pre, stream);               \
    else launch_decay_rows<TX, NR, 1, false>(a, rule, num_seqs, T, pre, stream);                                    \
  } while (0)
#define DR(TX)                            \
  do {                                    \
    if (N <= 32) DR_NR(TX, 32);           \
    else if (N <= 64) DR_NR(TX, 64);      \
    else if (N <= 128) DR_NR(TX, 128);    \
    else DR_NR(TX, 256);                  \
  } while (0)
  if (dtype == ME_F32) DR(float); else DR(bf16_t);
#undef DR
#undef DR_NR
  ME_LAUNCH_CHECK();
  return 0;
}
