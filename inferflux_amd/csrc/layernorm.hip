// Layer norm with a weight and no bias, over rows of up to MAX_H columns, all math in float:
//   y = (x - mean(x)) / sqrt(mean((x - mean(x))^2) + eps) * w
// Two uses.  ifx_layernorm normalises rows of a tensor (the float32 stream before the head, optionally only the
// rows a list names, optionally with a delta added first).  ifx_add_layernorm is the arrangement in which the norm
// sits on a sub-block's output: stream[t] += LN(delta[t]) * w, and beside it the new stream rounded to the
// activation type, which is what the next sub-block reads.
//
// A workgroup takes a row, holds it in LDS as floats (read once from memory, partial sums of a sliced product added
// in slice order on the way), forms the mean and then the mean of the squared deviations from it, both by the
// fixed-order sums of common.h: a row's result never depends on the other rows of the launch.
#include "common.h"

IFX_DEFINE_LAST_ERROR()

#define MAX_H 16000      // (the row and the sums fit 64 KB of LDS)

template <typename TX>
__device__ __forceinline__ float sliced(const TX* __restrict__ x, int i, int n_slices, size_t stride) {
  float v = to_f(x[i]);
  for (int s = 1; s < n_slices; ++s) v += to_f(x[(size_t)s * stride + i]);
  return v;
}

// the row's mean and 1 / sqrt(variance + eps) from the floats in `row`
__device__ __forceinline__ void moments(const float* row, int H, float eps, float* red, float& mean, float& rstd) {
  float s = 0.f;
  for (int i = threadIdx.x; i < H; i += blockDim.x) s += row[i];
  mean = block_sum(s, red) / (float)H;
  float v = 0.f;
  for (int i = threadIdx.x; i < H; i += blockDim.x) {
    const float d = row[i] - mean;
    v = fmaf(d, d, v);
  }
  rstd = 1.0f / sqrtf(block_sum(v, red) / (float)H + eps);
}

template <typename TX, typename TD, typename TO>
__global__ __launch_bounds__(256) void layernorm_kernel(TX* __restrict__ x, const TD* __restrict__ delta, int n_slices,
                                                        size_t slice_stride, const void* __restrict__ weight, int w_dtype,
                                                        TO* __restrict__ out, const int* __restrict__ rows, int H, float eps,
                                                        int write_back) {
  extern __shared__ float row[];
  __shared__ float red[16];
  const int r = blockIdx.x;
  const size_t src = rows ? (size_t)rows[r] : (size_t)r;
  TX* xr = x + src * H;
  for (int i = threadIdx.x; i < H; i += blockDim.x) {
    float v = to_f(xr[i]);
    if (delta) {
      v += sliced(delta + src * H, i, n_slices, slice_stride);
      if (write_back) xr[i] = from_f<TX>(v);
    }
    row[i] = v;
  }
  __syncthreads();
  float mean, rstd;
  moments(row, H, eps, red, mean, rstd);
  TO* o = out + (size_t)r * H;
  for (int i = threadIdx.x; i < H; i += blockDim.x) o[i] = from_f<TO>((row[i] - mean) * rstd * load_dyn(weight, w_dtype, i));
}

template <typename TD, typename TC>
__global__ __launch_bounds__(256) void add_layernorm_kernel(float* __restrict__ stream, const TD* __restrict__ delta, int n_slices,
                                                            size_t slice_stride, const void* __restrict__ weight, int w_dtype,
                                                            TC* __restrict__ cast_out, int H, float eps) {
  extern __shared__ float row[];
  __shared__ float red[16];
  constexpr int NV = 8;          // rows of up to 256 NV columns: the stream and the weight are asked for before the sums
  const size_t t = blockIdx.x;
  float* s = stream + t * H;
  const bool ahead = H <= 256 * NV;
  float sv[NV], wv[NV];
  if (ahead) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int i = threadIdx.x + 256 * v;
      sv[v] = i < H ? s[i] : 0.f;
      wv[v] = i < H ? load_dyn(weight, w_dtype, i) : 0.f;
    }
  }
  for (int i = threadIdx.x; i < H; i += blockDim.x) row[i] = sliced(delta + t * H, i, n_slices, slice_stride);
  __syncthreads();
  float mean, rstd;
  moments(row, H, eps, red, mean, rstd);
  if (ahead) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int i = threadIdx.x + 256 * v;
      if (i < H) {
        const float x = sv[v] + (row[i] - mean) * rstd * wv[v];
        s[i] = x;
        if (cast_out) cast_out[t * H + i] = from_f<TC>(x);
      }
    }
    return;
  }
  for (int i = threadIdx.x; i < H; i += blockDim.x) {
    const float v = s[i] + (row[i] - mean) * rstd * load_dyn(weight, w_dtype, i);
    s[i] = v;
    if (cast_out) cast_out[t * H + i] = from_f<TC>(v);
  }
}

// The same for rows of a multiple of 4 columns, up to 1,024 NV: a thread holds NV runs of four columns in registers and asks for
// all it needs at once (the row, the weight, the delta's first slice, then up to seven further slices), where the kernel above
// takes a trip per slice and run of 256 columns: 2,048 columns, 8 rows, six slices 19 us, one slice 9.8.
template <typename T> struct Four;
template <> struct Four<float> { typedef float4 type; };
template <> struct Four<bf16_t> { typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 type; };
__device__ __forceinline__ void widen(const float4& t, float* v) { v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w; }
__device__ __forceinline__ void widen(const Four<bf16_t>::type& t, float* v) {
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = (float)t[e];
}

template <typename TD, typename TC, typename TW, int NV>
__global__ __launch_bounds__(256) void add_layernorm4_kernel(float* __restrict__ stream, const TD* __restrict__ delta, int n_slices,
                                                             size_t slice_stride, const TW* __restrict__ weight, TC* __restrict__ cast_out,
                                                             int H, float eps) {
  __shared__ float red[16];
  constexpr int AT_ONCE = NV <= 2 ? 7 : 3;
  const size_t t = blockIdx.x;
  float* s = stream + t * H;
  const TD* d = delta + t * H;
  float4 was[NV];
  typename Four<TW>::type wt[NV];
  typename Four<TD>::type d0[NV];
  float x[NV][4];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int i = 4 * (threadIdx.x + blockDim.x * v);
    if (i >= H) continue;
    d0[v] = *(const typename Four<TD>::type*)(d + i);
    was[v] = *(const float4*)(s + i);
    wt[v] = *(const typename Four<TW>::type*)(weight + i);
  }
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    x[v][0] = x[v][1] = x[v][2] = x[v][3] = 0.f;
    if (4 * (int)(threadIdx.x + blockDim.x * v) < H) widen(d0[v], x[v]);
  }
  for (int k0 = 1; k0 < n_slices; k0 += AT_ONCE) {          // partial sums, added in slice order
    typename Four<TD>::type p[AT_ONCE][NV];
#pragma unroll
    for (int u = 0; u < AT_ONCE; ++u)
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const int i = 4 * (threadIdx.x + blockDim.x * v);
        if (k0 + u < n_slices && i < H) p[u][v] = *(const typename Four<TD>::type*)(d + (size_t)(k0 + u) * slice_stride + i);
      }
#pragma unroll
    for (int u = 0; u < AT_ONCE; ++u)
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        if (k0 + u >= n_slices || 4 * (int)(threadIdx.x + blockDim.x * v) >= H) continue;
        float f[4];
        widen(p[u][v], f);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[v][e] += f[e];
      }
  }
  float sum = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int e = 0; e < 4; ++e) sum += x[v][e];
  const float mean = block_sum(sum, red) / (float)H;
  float sq = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v)
    if (4 * (int)(threadIdx.x + blockDim.x * v) < H)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[v][e] -= mean;
        sq = fmaf(x[v][e], x[v][e], sq);
      }
  const float rstd = 1.0f / sqrtf(block_sum(sq, red) / (float)H + eps);
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int i = 4 * (threadIdx.x + blockDim.x * v);
    if (i >= H) continue;
    float y[4], w[4];
    widen(was[v], y);
    widen(wt[v], w);
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] += x[v][e] * rstd * w[e];
    *(float4*)(s + i) = make_float4(y[0], y[1], y[2], y[3]);
    if (cast_out) {
      TC* c = cast_out + t * H + i;
      if constexpr (sizeof(TC) == 4) *(float4*)c = make_float4(y[0], y[1], y[2], y[3]);
      else {
        Four<bf16_t>::type o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (__bf16)y[e];
        *(Four<bf16_t>::type*)c = o;
      }
    }
  }
}

template <typename TO>
__global__ __launch_bounds__(256) void cast_rows_kernel(const float* __restrict__ x, TO* __restrict__ out, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = from_f<TO>(x[i]);
}

// out = the float32 rows of x rounded to bfloat16 (what a sub-block that reads the stream itself is given first)
extern "C" int ifx_cast_rows(const float* x, void* out, int out_dtype, long long n, void* stream) {
  IFX_REQUIRE(n >= 0 && out_dtype == DT_BF16, "cast_rows: to bfloat16 only (dtype %d)", out_dtype);
  if (n == 0) return 0;
  hipLaunchKernelGGL(cast_rows_kernel<bf16_t>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, x, (bf16_t*)out, (size_t)n);
  IFX_LAUNCH_CHECK();
}

// out[r, :] = LN(x[src] (+ delta[src])) * weight, src = rows ? rows[r] : r.  x is float32 or bfloat16; with a delta
// and no row list the sum is written back to x.
extern "C" int ifx_layernorm(void* x, int x_dtype, const void* delta, int delta_dtype, int n_slices, long long slice_stride,
                             const void* weight, int w_dtype, void* out, int out_dtype, const int* rows, int n, int H,
                             float eps, void* stream) {
  IFX_REQUIRE(n >= 0 && H > 0 && H <= MAX_H, "layernorm: %d rows of %d columns (at most %d)", n, H, MAX_H);
  IFX_REQUIRE(n_slices >= 1, "layernorm: %d slices", n_slices);
  IFX_REQUIRE(w_dtype == DT_F32 || w_dtype == DT_BF16, "layernorm: unknown weight dtype %d", w_dtype);
  if (n == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const int wb = (delta && !rows) ? 1 : 0;
  const size_t lds = (size_t)H * sizeof(float);
#define LN_LAUNCH(TX, TD, TO) \
  hipLaunchKernelGGL((layernorm_kernel<TX, TD, TO>), dim3(n), dim3(256), lds, s, (TX*)x, (const TD*)delta, n_slices, \
                     (size_t)slice_stride, weight, w_dtype, (TO*)out, rows, H, eps, wb)
  const int dd = delta ? delta_dtype : DT_F32;
  if (x_dtype == DT_F32 && dd == DT_F32 && out_dtype == DT_F32) LN_LAUNCH(float, float, float);
  else if (x_dtype == DT_F32 && dd == DT_F32 && out_dtype == DT_BF16) LN_LAUNCH(float, float, bf16_t);
  else if (x_dtype == DT_F32 && dd == DT_BF16 && out_dtype == DT_BF16) LN_LAUNCH(float, bf16_t, bf16_t);
  else if (x_dtype == DT_BF16 && dd == DT_BF16 && out_dtype == DT_BF16) LN_LAUNCH(bf16_t, bf16_t, bf16_t);
  else if (x_dtype == DT_BF16 && dd == DT_F32 && out_dtype == DT_BF16) LN_LAUNCH(bf16_t, float, bf16_t);
  else IFX_FAIL("layernorm: unsupported types x=%d delta=%d out=%d", x_dtype, delta_dtype, out_dtype);
#undef LN_LAUNCH
  IFX_LAUNCH_CHECK();
}

// stream[t, :] += LN(delta[t, :]) * weight for every row; cast_out (or null) receives the new stream in cast_dtype.
extern "C" int ifx_add_layernorm(float* stream_rows, const void* delta, int delta_dtype, int n_slices, long long slice_stride,
                                 const void* weight, int w_dtype, void* cast_out, int cast_dtype, int T, int H, float eps,
                                 void* stream) {
  IFX_REQUIRE(T >= 0 && H > 0 && H <= MAX_H, "add_layernorm: %d rows of %d columns (at most %d)", T, H, MAX_H);
  IFX_REQUIRE(n_slices >= 1 && delta, "add_layernorm: needs a delta in at least one slice");
  IFX_REQUIRE(w_dtype == DT_F32 || w_dtype == DT_BF16, "add_layernorm: unknown weight dtype %d", w_dtype);
  if (T == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const size_t lds = (size_t)H * sizeof(float);
  // (operands on 16 bytes and slices a multiple of 4 apart, for loads of four elements)
  const bool fours = H % 4 == 0 && H <= 4096 && slice_stride % 4 == 0 && ((uintptr_t)stream_rows | (uintptr_t)delta | (uintptr_t)weight | (uintptr_t)cast_out) % 16 == 0;
  const int threads4 = min(256, (H / 4 + WAVE - 1) / WAVE * WAVE);      // (a run of four columns to a thread: narrow rows fill fewer)
#define ALN4(TD, TC, TW, NV) hipLaunchKernelGGL((add_layernorm4_kernel<TD, TC, TW, NV>), dim3(T), dim3(threads4), 0, s, stream_rows, (const TD*)delta, \
                                                n_slices, (size_t)slice_stride, (const TW*)weight, (TC*)cast_out, H, eps)
#define ALN_ROWS(TD, TC)                                                \
  do {                                                                  \
    if (!fours) ALN_LAUNCH(TD, TC);                                     \
    else if (w_dtype == DT_F32 && H <= 2048) ALN4(TD, TC, float, 2);    \
    else if (w_dtype == DT_F32) ALN4(TD, TC, float, 4);                 \
    else if (H <= 2048) ALN4(TD, TC, bf16_t, 2);                        \
    else ALN4(TD, TC, bf16_t, 4);                                       \
  } while (0)
#define ALN_LAUNCH(TD, TC) \
  hipLaunchKernelGGL((add_layernorm_kernel<TD, TC>), dim3(T), dim3(256), lds, s, stream_rows, (const TD*)delta, n_slices, \
                     (size_t)slice_stride, weight, w_dtype, (TC*)cast_out, H, eps)
  const int cd = cast_out ? cast_dtype : DT_BF16;
  if (delta_dtype == DT_F32 && cd == DT_BF16) ALN_ROWS(float, bf16_t);
  else if (delta_dtype == DT_F32 && cd == DT_F32) ALN_ROWS(float, float);
  else if (delta_dtype == DT_BF16 && cd == DT_BF16) ALN_ROWS(bf16_t, bf16_t);
  else if (delta_dtype == DT_BF16 && cd == DT_F32) ALN_ROWS(bf16_t, float);
  else IFX_FAIL("add_layernorm: unsupported types delta=%d cast=%d", delta_dtype, cast_dtype);
#undef ALN_LAUNCH
#undef ALN_ROWS
#undef ALN4
  IFX_LAUNCH_CHECK();
}
