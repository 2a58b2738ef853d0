// Helper kernels of attention through a latent: what lies between the mixer's matrix products and the paged
// attention kernels.
//
// The mixer projects its input down to a query latent, a key/value latent c (kv_rank wide) and one rotated key part
// k_r (rot_dim wide) that every head shares.  Per head the unrotated key is W_uk c and the value W_uv c, so the score
//   (q_n . W_uk c + q_r . k_r) * scale = ([W_uk^T q_n | q_r] . [c | k_r]) * scale
// and the head's output W_uv (sum_j a_j c_j): attention runs over one shared "kv head" whose key is [c | k_r]
// and whose value is c, with queries of kv_rank + rot_dim elements, and only c and k_r are cached.
//
//   ifx_latent_finish   after the down projections: RMS norm of the query latent (handed on), RMS norm of c and
//                       rotation of k_r, both written into the paged cache (K rows [c | k_r], V columns c; or V
//                       columns [c | k_r] too, for attention kernels that want values as wide as keys: the sums
//                       over k_r that they then return behind a head's kv_rank outputs are not used by anyone)
//   ifx_headwise        out[t, h, :] = W[h] x[t, h, :] for every head (W [H][N][K]), the products by W_uk^T and
//                       W_uv; optionally a tail of each head's input is rotated and appended to the head's output
//                       (the rotated query part); optionally out[t, h, n] is multiplied by sigmoid of a column of a wider
//                       projected row, one column per output element (the output gate on W_uv's product)
//
//   ifx_headwise_splits the same from the row kernel's splits of attention (split_rows.h): W_uv's product of up to 16 rows
//   ifx_latent_query    ifx_headwise of the queries and ifx_latent_finish of the latent without a query latent, in one launch
//
// All sums in float in ascending k, one output element per thread: a row's result does not depend on the batch.
#include "common.h"
#include "column_gate.h"
#include "split_rows.h"

IFX_DEFINE_LAST_ERROR()

template <typename TY>
__device__ __forceinline__ float sliced(const TY* __restrict__ y, int i, int n_slices, size_t stride) {
  float v = to_f(y[i]);
  for (int s = 1; s < n_slices; ++s) v += to_f(y[(size_t)s * stride + i]);
  return v;
}

// y [T][ld], a row's q_rank + kv_rank + rot_dim numbers from ``y`` on (n_slices partial sums, slice_stride elements apart)
template <typename TY, typename T>
struct FinishArgs {
  const TY* y;
  int n_slices;
  size_t slice_stride;
  const void* wq; const void* wkv;
  int w_dtype;
  const float* cs; const float* sn;
  int rot_dims;
  const int* slots;
  T* cq; T* k_cache; T* v_cache;
  int q_rank, kv_rank, rot_dim, page_size;
  float eps;
  int v_rows, ld;
};

// Row t by the workgroup's 256 threads.  LF_EACH: numbers of each latent that a thread keeps in registers (wider latents are read
// again); ``red``: 32 floats of LDS.
template <typename TY, typename T, int LF_EACH>
__device__ __forceinline__ void finish_row(const FinishArgs<TY, T>& a, size_t t, float* red) {
  const int n_slices = a.n_slices, rot_dims = a.rot_dims, q_rank = a.q_rank, kv_rank = a.kv_rank, rot_dim = a.rot_dim, page_size = a.page_size;
  const int v_rows = a.v_rows, w_dtype = a.w_dtype;
  const size_t slice_stride = a.slice_stride;
  const float eps = a.eps, *cs = a.cs, *sn = a.sn;
  const int* slots = a.slots;
  const void *wq = a.wq, *wkv = a.wkv;
  T *cq = a.cq, *k_cache = a.k_cache, *v_cache = a.v_cache;
  const TY* yr = a.y + t * a.ld;
  const TY* yc = yr + q_rank;
  const TY* yk = yc + kv_rank;
  const int slot = slots ? slots[t] : -1, half = rot_dims / 2, tid = threadIdx.x;
  const int n_kv = slots ? kv_rank : 0, n_rot = slots ? rot_dim : 0;
  // A thread's numbers of both latents and of the key part, every load on its way before the first is used.  (Where a thread
  // has no number the last one is read again and counts as zero: loads without branches.)
  float q[LF_EACH], c[LF_EACH], k = 0.f, k_other = 0.f, cv = 1.f, sv = 0.f;
  const int other = tid < half ? tid + half : tid - half;
  const int ki = n_rot > 0 ? min(tid, n_rot - 1) : 0, ko = n_rot > 0 ? min(max(tid < rot_dims ? other : tid, 0), n_rot - 1) : 0;
  const TY* yk_safe = n_rot > 0 ? yk : yr;
  const TY* yc_safe = n_kv > 0 ? yc : yr;
#pragma unroll
  for (int e = 0; e < LF_EACH; ++e) { q[e] = 0.f; c[e] = 0.f; }
#pragma unroll 4
  for (int s = 0; s < n_slices; ++s) {
    const size_t at = (size_t)s * slice_stride;
#pragma unroll
    for (int e = 0; e < LF_EACH; ++e) {
      q[e] += to_f(yr[at + min(tid + 256 * e, max(q_rank - 1, 0))]);
      c[e] += to_f(yc_safe[at + min(tid + 256 * e, max(n_kv - 1, 0))]);
    }
    k += to_f(yk_safe[at + ki]);
    k_other += to_f(yk_safe[at + ko]);
  }
#pragma unroll
  for (int e = 0; e < LF_EACH; ++e) {
    if (tid + 256 * e >= q_rank) q[e] = 0.f;
    if (tid + 256 * e >= n_kv) c[e] = 0.f;
  }
  if (tid < n_rot && tid < rot_dims) {
    const int p = tid < half ? tid : other;
    cv = cs[t * half + p]; sv = sn[t * half + p];
  }
  float sq = 0.f, sc = 0.f;
#pragma unroll
  for (int e = 0; e < LF_EACH; ++e) { sq = fmaf(q[e], q[e], sq); sc = fmaf(c[e], c[e], sc); }
  for (int i = tid + 256 * LF_EACH; i < q_rank; i += 256) { const float v = sliced(yr, i, n_slices, slice_stride); sq = fmaf(v, v, sq); }
  for (int i = tid + 256 * LF_EACH; i < n_kv; i += 256) { const float v = sliced(yc, i, n_slices, slice_stride); sc = fmaf(v, v, sc); }
  // both sums over the workgroup's four waves in one meeting
  sq = wave_sum(sq); sc = wave_sum(sc);
  if (tid % WAVE == 0) { red[tid / WAVE] = sq; red[16 + tid / WAVE] = sc; }
  __syncthreads();
  sq = (red[0] + red[1]) + (red[2] + red[3]);
  sc = (red[16] + red[17]) + (red[18] + red[19]);
  if (q_rank > 0) {
    const float r = 1.0f / sqrtf(sq / (float)q_rank + eps);
#pragma unroll
    for (int e = 0; e < LF_EACH; ++e) {
      const int i = tid + 256 * e;
      if (i < q_rank) cq[t * q_rank + i] = from_f<T>(q[e] * r * load_dyn(wq, w_dtype, i));
    }
    for (int i = tid + 256 * LF_EACH; i < q_rank; i += 256) cq[t * q_rank + i] = from_f<T>(sliced(yr, i, n_slices, slice_stride) * r * load_dyn(wq, w_dtype, i));
  }
  if (!slots) return;
  const int page = slot / page_size, off = slot % page_size;
  const int d = kv_rank + rot_dim;
  T* krow = k_cache + (size_t)slot * d;                       // K [page][1][offset][d]
  T* vcol = v_cache + (size_t)page * v_rows * page_size + off;    // V [page][1][v_rows][offset], v_rows = kv_rank or d
  const float r = 1.0f / sqrtf(sc / (float)kv_rank + eps);
  auto put = [&](int i, float v) {
    const T x = from_f<T>(v * r * load_dyn(wkv, w_dtype, i));
    krow[i] = x;
    vcol[(size_t)i * page_size] = x;
  };
#pragma unroll
  for (int e = 0; e < LF_EACH; ++e)
    if (tid + 256 * e < kv_rank) put(tid + 256 * e, c[e]);
  for (int i = tid + 256 * LF_EACH; i < kv_rank; i += 256) put(i, sliced(yc, i, n_slices, slice_stride));
  auto put_k = [&](int i, float v) {
    krow[kv_rank + i] = from_f<T>(v);
    if (v_rows > kv_rank) vcol[(size_t)(kv_rank + i) * page_size] = from_f<T>(v);   // values as wide as keys: see the entry point
  };
  if (tid < rot_dim) put_k(tid, tid >= rot_dims ? k : (tid < half ? k * cv - k_other * sv : k * cv + k_other * sv));
  for (int i = tid + 256; i < rot_dim; i += 256) {      // (a key part wider than the workgroup)
    float v = sliced(yk, i, n_slices, slice_stride);
    if (i < rot_dims) {
      const int p = i < half ? i : i - half;
      const float cp = cs[t * half + p], sp = sn[t * half + p];
      const float o = sliced(yk, i < half ? i + half : i - half, n_slices, slice_stride);
      v = i < half ? v * cp - o * sp : v * cp + o * sp;
    }
    put_k(i, v);
  }
}

template <typename TY, typename T, int LF_EACH>
__global__ __launch_bounds__(256) void latent_finish_kernel(FinishArgs<TY, T> a) {
  __shared__ float red[32];
  finish_row<TY, T, LF_EACH>(a, blockIdx.x, red);
}

extern "C" int ifx_latent_finish(const void* y, int y_dtype, int n_slices, long long slice_stride, const void* wq, const void* wkv,
                                 int w_dtype, const float* cs, const float* sn, int rot_dims, const int* slots, void* cq,
                                 void* k_cache, void* v_cache, int dtype, int T, int q_rank, int kv_rank, int rot_dim,
                                 int page_size, float eps, int v_rows, int ld, void* stream) {
  IFX_REQUIRE(ld >= q_rank + (slots ? kv_rank + rot_dim : 0), "latent_finish: rows of %d are too short", ld);
  IFX_REQUIRE(T >= 0 && q_rank >= 0 && kv_rank > 0 && rot_dim >= 0, "latent_finish: bad sizes T=%d q_rank=%d kv_rank=%d rot_dim=%d", T, q_rank, kv_rank, rot_dim);
  IFX_REQUIRE(rot_dims >= 0 && rot_dims % 2 == 0 && rot_dims <= rot_dim, "latent_finish: %d of %d dimensions rotate", rot_dims, rot_dim);
  IFX_REQUIRE(rot_dims == 0 || (cs && sn), "latent_finish: a rotation needs its table");
  IFX_REQUIRE(!slots || (k_cache && v_cache && page_size > 0), "latent_finish: slots but no cache");
  IFX_REQUIRE(v_rows == kv_rank || v_rows == kv_rank + rot_dim, "latent_finish: values of %d rows (the latent's %d, or %d with the key part)", v_rows, kv_rank, kv_rank + rot_dim);
  IFX_REQUIRE(n_slices >= 1 && (n_slices == 1 || y_dtype == DT_F32), "latent_finish: partial sums are float32");
  IFX_REQUIRE(w_dtype == DT_F32 || w_dtype == DT_BF16, "latent_finish: unknown weight dtype %d", w_dtype);
  if (T == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const int widest = max(q_rank, slots ? kv_rank : 0);
#define LF_LAUNCH(TY, TT)                                                \
  do {                                                                   \
    if (widest <= 256) LF_GO(TY, TT, 1);                                 \
    else if (widest <= 512) LF_GO(TY, TT, 2);                            \
    else if (widest <= 1024) LF_GO(TY, TT, 4);                           \
    else LF_GO(TY, TT, 6);                                               \
  } while (0)
#define LF_GO(TY, TT, EACH) \
  hipLaunchKernelGGL((latent_finish_kernel<TY, TT, EACH>), dim3(T), dim3(256), 0, s,                                                          \
                     FinishArgs<TY, TT>{(const TY*)y, n_slices, (size_t)slice_stride, wq, wkv, w_dtype, cs, sn, rot_dims, slots, (TT*)cq,       \
                                        (TT*)k_cache, (TT*)v_cache, q_rank, kv_rank, rot_dim, page_size, eps, v_rows, ld})
  if (y_dtype == DT_F32 && dtype == DT_F32) LF_LAUNCH(float, float);
  else if (y_dtype == DT_F32 && dtype == DT_BF16) LF_LAUNCH(float, bf16_t);
  else if (y_dtype == DT_BF16 && dtype == DT_BF16) LF_LAUNCH(bf16_t, bf16_t);
  else IFX_FAIL("latent_finish: unsupported types y=%d out=%d", y_dtype, dtype);
#undef LF_LAUNCH
#undef LF_GO
  IFX_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------------------
// out[t][h][n] = sum_k W[h][n][k] * x[t][h * x_head + k]   (n < N), and for a tail of `tail` elements that follow
// the K inputs of each head, out[t][h][N + e] = the tail turned by the step's rotation table (its first rot_dims
// elements in split-half pairs, the rest as they are).  x rows are x_row apart, out rows H * (N + tail) wide.
struct HeadwiseArgs {
  const void* x; const void* w; void* out;
  const float* cs; const float* sn;
  int T, H, K, N, x_row, x_head, tail, rot_dims;
  ColumnGate gate;   // columns col + h * N + n of row t
  int tile0;      // the launch's first tile (the tail's, when only the tails are wanted)
};

#define HW_TM 16
#define HW_TN 64
#define HW_TK 32

template <typename T>
__global__ __launch_bounds__(256) void headwise_kernel(HeadwiseArgs a) {
  __shared__ float xs[HW_TM][HW_TK];
  __shared__ float ws[HW_TN][HW_TK + 1];
  const int n_tiles = (a.N + HW_TN - 1) / HW_TN;
  const int h = blockIdx.y, t0 = blockIdx.x * HW_TM, tile = blockIdx.z + a.tile0;
  const int out_head = a.N + a.tail;
  const T* x = (const T*)a.x;
  T* out = (T*)a.out;
  if (tile == n_tiles) {      // the tail: rotate and copy
    const int half = a.rot_dims / 2;
    for (int idx = threadIdx.x; idx < HW_TM * a.tail; idx += blockDim.x) {
      const int t = t0 + idx / a.tail, e = idx % a.tail;
      if (t >= a.T) continue;
      const T* xt = x + (size_t)t * a.x_row + (size_t)h * a.x_head + a.K;
      float v = to_f(xt[e]);
      if (e < a.rot_dims) {
        const int p = e < half ? e : e - half;
        const float c = a.cs[(size_t)t * half + p], s = a.sn[(size_t)t * half + p];
        const float other = to_f(xt[e < half ? e + half : e - half]);
        v = e < half ? v * c - other * s : v * c + other * s;
      }
      out[((size_t)t * a.H + h) * out_head + a.N + e] = from_f<T>(v);
    }
    return;
  }
  const int n0 = tile * HW_TN;
  const int tx = threadIdx.x % HW_TN, ty = threadIdx.x / HW_TN;     // output column, group of four rows
  const T* w = (const T*)a.w + (size_t)h * a.N * a.K;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < a.K; k0 += HW_TK) {
    for (int idx = threadIdx.x; idx < HW_TM * HW_TK; idx += blockDim.x) {
      const int m = idx / HW_TK, kk = idx % HW_TK, t = t0 + m, k = k0 + kk;
      xs[m][kk] = (t < a.T && k < a.K) ? to_f(x[(size_t)t * a.x_row + (size_t)h * a.x_head + k]) : 0.f;
    }
    for (int idx = threadIdx.x; idx < HW_TN * HW_TK; idx += blockDim.x) {
      const int n = idx / HW_TK, kk = idx % HW_TK, k = k0 + kk;
      ws[n][kk] = (n0 + n < a.N && k < a.K) ? to_f(w[(size_t)(n0 + n) * a.K + k]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < HW_TK; ++kk) {
      const float wv = ws[tx][kk];
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[m] = fmaf(xs[ty * 4 + m][kk], wv, acc[m]);
    }
    __syncthreads();
  }
  if (n0 + tx < a.N)
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int t = t0 + ty * 4 + m;
      if (t < a.T) out[((size_t)t * a.H + h) * out_head + n0 + tx] = from_f<T>(a.gate.rows ? acc[m] * a.gate.at<T>(t, h * a.N + n0 + tx) : acc[m]);
    }
}

// The same for steps of few rows: a thread owns one output element of one (row, head) and reads its weight row in
// 16-byte pieces, all asked for at once (a wave's rows are one contiguous run of memory); no LDS, no barrier.  The sum
// runs over k in the tiled kernel's order, so both give the same bits.
// The row of x, the same for all threads, is read through the constant address space: scalar loads, which no vector load waits for.  Where workgroups beside these write
// (latent_query_kernel) the compiler read it by vector loads otherwise, each of which waited for itself and for the weights asked for before it.
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 hw_bf16x8;
#define HW_CONSTANT __attribute__((address_space(4)))
__device__ __forceinline__ void hw_widen(hw_bf16x8 t, float* v) {
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = (float)t[i];
}
__device__ __forceinline__ void hw_load8(const HW_CONSTANT bf16_t* p, float* v) { hw_widen(*(const HW_CONSTANT hw_bf16x8*)p, v); }
__device__ __forceinline__ void hw_load8(const HW_CONSTANT float* p, float* v) {
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = p[i];
}
__device__ __forceinline__ void hw_load8(const bf16_t* p, float* v) { hw_widen(*(const hw_bf16x8*)p, v); }
__device__ __forceinline__ void hw_load8(const float* p, float* v) {
  const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

template <typename T>
__device__ __forceinline__ void headwise_row(const HeadwiseArgs& a, int t, int h, int n) {
  const int out_head = a.N + a.tail;
  const T* xt = (const T*)a.x + (size_t)t * a.x_row + (size_t)h * a.x_head;
  T* out = (T*)a.out + ((size_t)t * a.H + h) * out_head;
  if (n < a.N) {
    const T* w = (const T*)a.w + ((size_t)h * a.N + n) * a.K;
    const HW_CONSTANT T* xc = (const HW_CONSTANT T*)xt;
    float acc = 0.f;
#pragma unroll 4
    for (int k = 0; k < a.K; k += 8) {
      float xv[8], wv[8];
      hw_load8(xc + k, xv);
      hw_load8(w + k, wv);
#pragma unroll
      for (int i = 0; i < 8; ++i) acc = fmaf(xv[i], wv[i], acc);
    }
    out[n] = from_f<T>(a.gate.rows ? acc * a.gate.at<T>(t, h * a.N + n) : acc);
  } else if (n < out_head) {
    const int e = n - a.N, half = a.rot_dims / 2;
    float v = to_f(xt[a.K + e]);
    if (e < a.rot_dims) {
      const int p = e < half ? e : e - half;
      const float c = a.cs[(size_t)t * half + p], s = a.sn[(size_t)t * half + p];
      const float other = to_f(xt[a.K + (e < half ? e + half : e - half)]);
      v = e < half ? v * c - other * s : v * c + other * s;
    }
    out[n] = from_f<T>(v);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void headwise_rows_kernel(HeadwiseArgs a) {
  headwise_row<T>(a, blockIdx.x, blockIdx.y, blockIdx.z * 256 + threadIdx.x);
}

// The queries' side of a step and the cache's, which do not need each other: workgroups (row, head) for the product, and one a row
// behind them for ``finish_row``.  Bound by the launch and a chain of two trips, or W_uk: us in one launch / two, 4 rows of 32 heads of 96 x 512 5.2 / 4.2 + 3.6, 8 rows
// 6.7 / 6.2 + 3.7, of 96 x 96 4.0 / 3.7 + 3.3, 8 rows of 64 heads of 128 x 512 13.7 / 13.3 + 4.1.
template <int LF_EACH>
__global__ __launch_bounds__(256) void latent_query_kernel(HeadwiseArgs a, FinishArgs<bf16_t, bf16_t> f) {
  __shared__ float red[32];
  if ((int)blockIdx.y < a.H) headwise_row<bf16_t>(a, blockIdx.x, blockIdx.y, blockIdx.z * 256 + threadIdx.x);
  else if (blockIdx.z == 0) finish_row<bf16_t, bf16_t, LF_EACH>(f, blockIdx.x, red);
}

// W_uv's product from attention's splits: a workgroup's four waves join a head's splits (in float, no rounding between) while the
// weights, a thread its whole row, are on their way.  Bound by its launch and one trip to memory: 8 rows of 16 heads in 16 splits 4.8 us, where
// the launch that joined them took 5.1 and the product from rows 4.7.
__global__ __launch_bounds__(256) void headwise_splits_kernel(HeadwiseArgs a, SplitRows p) {
  typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
  __shared__ __attribute__((aligned(16))) float xs[SPLITS_MAX_WIDTH];
  __shared__ float sums[4][SPLITS_MAX_WIDTH];
  const int t = blockIdx.x, h = blockIdx.y, n = blockIdx.z * 256 + threadIdx.x, wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const size_t at = (size_t)t * a.H + h;
  SplitMerge<4> m;
  m.ask(p, at, a.K, wave, lane);
  const bf16_t* w = (const bf16_t*)a.w + ((size_t)h * a.N + min(n, a.N - 1)) * a.K;
  bf16x8 wv[SPLITS_MAX_WIDTH / 8];
#pragma unroll
  for (int i = 0; i < SPLITS_MAX_WIDTH / 8; ++i) wv[i] = *(const bf16x8*)(w + min(8 * i, a.K - 8));
  const float gate = a.gate.rows && n < a.N ? a.gate.at<bf16_t>(t, h * a.N + n) : 1.f;
  const float inv = m.weigh(p, at, a.H);
  m.sums(wave, sums[wave], lane);
  __syncthreads();
  const int e = threadIdx.x;
  if (e < SPLITS_MAX_WIDTH) xs[e] = ((sums[0][e] + sums[1][e]) + (sums[2][e] + sums[3][e])) * inv;
  __syncthreads();
  if (n >= a.N) return;
  float y = 0.f;
#pragma unroll
  for (int i = 0; i < SPLITS_MAX_WIDTH / 8; ++i)
    if (8 * i < a.K) {
      float x[8];
      hw_load8(xs + 8 * i, x);
#pragma unroll
      for (int j = 0; j < 8; ++j) y = fmaf(x[j], (float)wv[i][j], y);
    }
  ((bf16_t*)a.out)[at * a.N + n] = (bf16_t)(y * gate);
}

#define HW_ROWS_MAX_T 16

extern "C" int ifx_headwise(const void* x, const void* w, void* out, int dtype, int T, int H, int K, int N, int x_row, int x_head,
                            int tail, const float* cs, const float* sn, int rot_dims, int tail_only, const void* gate, int gate_ld,
                            int gate_col, int gate_slices, long long gate_stride, void* stream) {
  IFX_REQUIRE(T >= 0 && H > 0 && K > 0 && N > 0 && tail >= 0, "headwise: bad sizes T=%d H=%d K=%d N=%d tail=%d", T, H, K, N, tail);
  IFX_REQUIRE(x_head >= K + tail && x_row >= (H - 1) * x_head + K + tail, "headwise: the heads do not fit the rows of x");
  IFX_REQUIRE(rot_dims >= 0 && rot_dims % 2 == 0 && rot_dims <= tail, "headwise: %d of a tail of %d rotate", rot_dims, tail);
  IFX_REQUIRE(rot_dims == 0 || (cs && sn), "headwise: a rotation needs its table");
  IFX_REQUIRE(H <= 65535, "headwise: %d heads", H);
  if (T == 0) return 0;
  HeadwiseArgs a{x, w, out, cs, sn, T, H, K, N, x_row, x_head, tail, rot_dims,
                 ColumnGate{gate, gate_ld, gate_col, gate_slices, (size_t)gate_stride}, 0};
  IFX_REQUIRE(!gate || (gate_col >= 0 && gate_col + H * N <= gate_ld && gate_slices >= 0), "headwise: %d gates from column %d on do not fit rows of %d", H * N, gate_col, gate_ld);
  // tail_only: the products are somebody else's (the grouped matrix-core kernel's); only the tails are turned and copied
  IFX_REQUIRE(!tail_only || tail > 0, "headwise: tail_only without a tail");
  a.tile0 = tail_only ? (N + HW_TN - 1) / HW_TN : 0;
  hipStream_t s = (hipStream_t)stream;
  if (!tail_only && T <= HW_ROWS_MAX_T && K % 8 == 0 && x_row % 8 == 0 && x_head % 8 == 0 && (uintptr_t)x % 4 == 0) {      // (scalar loads: on 4 bytes)
    const dim3 grid(T, H, (N + tail + 255) / 256);
    if (dtype == DT_F32) hipLaunchKernelGGL(headwise_rows_kernel<float>, grid, dim3(256), 0, s, a);
    else if (dtype == DT_BF16) hipLaunchKernelGGL(headwise_rows_kernel<bf16_t>, grid, dim3(256), 0, s, a);
    else IFX_FAIL("headwise: unknown dtype %d", dtype);
    IFX_LAUNCH_CHECK();
  }
  const dim3 grid((T + HW_TM - 1) / HW_TM, H, tail_only ? 1 : (N + HW_TN - 1) / HW_TN + (tail > 0 ? 1 : 0));
  if (dtype == DT_F32) hipLaunchKernelGGL(headwise_kernel<float>, grid, dim3(256), 0, s, a);
  else if (dtype == DT_BF16) hipLaunchKernelGGL(headwise_kernel<bf16_t>, grid, dim3(256), 0, s, a);
  else IFX_FAIL("headwise: unknown dtype %d", dtype);
  IFX_LAUNCH_CHECK();
}

extern "C" int ifx_headwise_splits(const float* part_o, const float* part_ml, const float* sinks, int splits, int D, const void* w, void* out, int T,
                                   int H, int K, int N, const void* gate, int gate_ld, int gate_col, int gate_slices, long long gate_stride, void* stream) {
  IFX_REQUIRE(T >= 0 && T <= HW_ROWS_MAX_T && H > 0 && H <= 65535 && N > 0, "headwise_splits: bad sizes T=%d H=%d N=%d", T, H, N);
  IFX_REQUIRE(K > 0 && K % 8 == 0 && K <= SPLITS_MAX_WIDTH && K <= D, "headwise_splits: K=%d (a multiple of 8 up to %d) of heads of %d", K, SPLITS_MAX_WIDTH, D);
  IFX_REQUIRE(part_o && part_ml && splits > 0 && splits <= SPLITS_MAX, "headwise_splits: %d splits (1-%d)", splits, SPLITS_MAX);
  IFX_REQUIRE(!gate || (gate_col >= 0 && gate_col + H * N <= gate_ld && gate_slices >= 0), "headwise_splits: %d gates from column %d on do not fit rows of %d", H * N, gate_col, gate_ld);
  if (T == 0) return 0;
  HeadwiseArgs a{nullptr, w, out, nullptr, nullptr, T, H, K, N, 0, 0, 0, 0, ColumnGate{gate, gate_ld, gate_col, gate_slices, (size_t)gate_stride}, 0};
  hipLaunchKernelGGL(headwise_splits_kernel, dim3(T, H, (N + 255) / 256), dim3(256), 0, (hipStream_t)stream, a, SplitRows{part_o, part_ml, sinks, splits, D});
  IFX_LAUNCH_CHECK();
}

// x [T][x_row]: the queries; y [T][ld]: a row's kv_rank + rot_dim numbers, the latent and the key part (columns of the same rows or of others).
extern "C" int ifx_latent_query(const void* x, int x_row, const void* y, int ld, const void* w, void* out, int T, int H, int K, int N, int x_head,
                                int tail, const float* cs, const float* sn, int rot_dims, const void* wkv, int w_dtype, const int* slots,
                                void* k_cache, void* v_cache, int kv_rank, int rot_dim, int page_size, float eps, int v_rows, void* stream) {
  IFX_REQUIRE(T >= 0 && T <= HW_ROWS_MAX_T && H > 0 && H < 65535 && K > 0 && N > 0 && tail >= 0 && x_head >= K + tail, "latent_query: bad sizes T=%d H=%d K=%d N=%d tail=%d", T, H, K, N, tail);
  IFX_REQUIRE(K % 8 == 0 && x_head % 8 == 0 && x_row % 8 == 0 && (uintptr_t)x % 16 == 0, "latent_query: K=%d, heads of %d and rows of %d must be multiples of 8", K, x_head, x_row);
  IFX_REQUIRE(x_row >= (H - 1) * x_head + K + tail, "latent_query: the heads do not fit the rows of x");
  IFX_REQUIRE(kv_rank > 0 && rot_dim >= 0 && kv_rank <= 1536 && ld >= kv_rank + rot_dim, "latent_query: rows of %d are too short", ld);
  IFX_REQUIRE(rot_dims >= 0 && rot_dims % 2 == 0 && rot_dims <= rot_dim && rot_dims <= tail, "latent_query: %d of %d dimensions rotate", rot_dims, rot_dim);
  IFX_REQUIRE(rot_dims == 0 || (cs && sn), "latent_query: a rotation needs its table");
  IFX_REQUIRE(slots && k_cache && v_cache && page_size > 0, "latent_query: no cache");
  IFX_REQUIRE(v_rows == kv_rank || v_rows == kv_rank + rot_dim, "latent_query: values of %d rows (the latent's %d, or %d with the key part)", v_rows, kv_rank, kv_rank + rot_dim);
  IFX_REQUIRE(w_dtype == DT_F32 || w_dtype == DT_BF16, "latent_query: unknown weight dtype %d", w_dtype);
  if (T == 0) return 0;
  HeadwiseArgs a{x, w, out, cs, sn, T, H, K, N, x_row, x_head, tail, rot_dims, ColumnGate{nullptr, 0, 0, 0, 0}, 0};
  FinishArgs<bf16_t, bf16_t> f{(const bf16_t*)y, 1, 0, nullptr, wkv, w_dtype, cs, sn, rot_dims, slots, nullptr, (bf16_t*)k_cache,
                               (bf16_t*)v_cache, 0, kv_rank, rot_dim, page_size, eps, v_rows, ld};
  const dim3 grid(T, H + 1, (N + tail + 255) / 256);
  if (kv_rank <= 256) hipLaunchKernelGGL(latent_query_kernel<1>, grid, dim3(256), 0, (hipStream_t)stream, a, f);
  else if (kv_rank <= 512) hipLaunchKernelGGL(latent_query_kernel<2>, grid, dim3(256), 0, (hipStream_t)stream, a, f);
  else hipLaunchKernelGGL(latent_query_kernel<6>, grid, dim3(256), 0, (hipStream_t)stream, a, f);
  IFX_LAUNCH_CHECK();
}
