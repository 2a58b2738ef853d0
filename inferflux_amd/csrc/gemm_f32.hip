// True 32-bit matrix product:  C[M,N] = A[M,K] * W[N,K]^T (+ bias[N]).
//
// The weight is float and every multiply-add is one of the 32-bit matrix instruction (v_mfma_f32_16x16x4_f32: float
// products, float sums, no reduced-precision mode).  An element's sum does not depend on M, on the element's place in the
// batch or on what else runs: K is cut into the same sixteen slices whatever M and N are, a slice is summed in one chain of
// matrix instructions in ascending steps of 16 (instruction j of a step takes k = 4 q + j of the step's 16 for q = 0 .. 3,
// which is how four consecutive floats per lane lie in registers), and the slices' sums are added in ascending order.  Both
// kernels below keep that order, so rows computed alone and in a batch of thousands are the same bits.
// This is the matrix product of the 32-bit path; the reference has no 32-bit path
// (runtime/backends/cuda/native/transformer_forward.cu:4600-4601 instantiates half and bf16
// only), its library call with float accumulation is runtime/backends/cuda/native/cublas_gemm.cpp:99-117.
#include "common.h"
#include "f32_loads.h"
#include "product_tiles.h"

IFX_DEFINE_LAST_ERROR()

#define N_SLICES 16

__device__ __forceinline__ int slice_len(int K) { return ((K + N_SLICES - 1) / N_SLICES + 15) / 16 * 16; }

// ---- the results ---------------------------------------------------------------------------------------------------------
// Either the sums as they are, C [M][N], or, with an activation, weight rows of gate and up in turn and C [M][N / 2] = act(gate) * up:
// neighbouring lanes hold neighbouring columns, the even one stores for both.  Called by all lanes of a wave that hold a sum (an even
// number of them); `in`: whether this lane's is within C.  The formula is that of the kernel that would read the sums back
// (swiglu, 4.9 us a launch of few rows), so the bits are the same.
struct Gated {
  int act;                  // -1: none
  float limit;
};
template <typename TO>
__device__ __forceinline__ void put(TO* __restrict__ C, int m, int n, int N, float v, bool in, const Gated& g) {
  if (g.act < 0) {
    if (in) C[(size_t)m * N + n] = from_f<TO>(v);
    return;
  }
  const float up = __shfl_down(v, 1);
  if (in && n % 2 == 0) C[(size_t)m * (N / 2) + n / 2] = from_f<TO>(gated_act(v, up, g.act, g.limit));
}

// ---- few rows: the weight is streamed once -----------------------------------------------------------------------------
// A workgroup takes NT x 16 weight rows and MT x 16 rows of A; its sixteen waves take a slice of K each and meet in LDS.
// Bound by the weight's bytes where N is large (5.6 TB/s at 151,936 x 896) and by the few workgroups where it is not (56 for
// 896 rows: 1.2 TB/s at K = 4,864): a wave has STEPS steps of 16 k-values (STEPS x (NT + MT) loads of 16 bytes a lane) in
// flight, and as many waves as a workgroup can hold do more than longer runs of loads in fewer (8 and 10 steps, eight waves:
// 15.1 to 17.5 us where these take 14.5).
template <typename TA, typename TO, int MT, int NT, int STEPS, bool VEC>
__global__ __launch_bounds__(1024) void gemm_f32_few_kernel(const TA* __restrict__ A, const float* __restrict__ W,
                                                           const float* __restrict__ bias, TO* __restrict__ C,
                                                           int M, int N, int K, Gated gated) {
  __shared__ float part[N_SLICES][MT * NT][256];
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
  const int i = lane % 16, q = lane / 16;
  const int n0 = blockIdx.x * (16 * NT), m0 = blockIdx.y * (16 * MT);
  const int len = slice_len(K), k_lo = wave * len, k_hi = min(K, k_lo + len);
  const float* wrow[NT];
  const TA* arow[MT];
  bool a_in[MT];
#pragma unroll
  for (int n = 0; n < NT; ++n) wrow[n] = W + (size_t)min(n0 + 16 * n + i, N - 1) * K;      // (columns beyond N are computed and dropped)
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    a_in[m] = m0 + 16 * m + i < M;
    arow[m] = A + (size_t)min(m0 + 16 * m + i, M - 1) * K;
  }
  f32x4 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = (f32x4){0.f, 0.f, 0.f, 0.f};

  f32x4 w[STEPS][NT], a[STEPS][MT];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int k = k0 + 16 * s + 4 * q;
#pragma unroll
      for (int n = 0; n < NT; ++n) w[s][n] = load4<VEC>(wrow[n], k, k_hi);
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        a[s][m] = (f32x4){0.f, 0.f, 0.f, 0.f};
        if (a_in[m]) a[s][m] = load4<VEC>(arow[m], k, k_hi);
      }
    }
  };
  for (int k0 = k_lo; k0 < k_hi; k0 += 16 * STEPS) {
    fetch(k0);
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int n = 0; n < NT; ++n)
            acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s][m][j], w[s][n][j], acc[m][n], 0, 0, 0);
  }
  // lane (i, q) holds rows 4 q + r of column i
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) part[wave][m * NT + n][(4 * q + r) * 16 + i] = acc[m][n][r];
  __syncthreads();
  for (int e = threadIdx.x; e < MT * NT * 256; e += 1024) {
    const int t = e / 256, at = e % 256, m = m0 + 16 * (t / NT) + at / 16, n = n0 + 16 * (t % NT) + at % 16;
    float v = part[0][t][at];
#pragma unroll
    for (int s = 1; s < N_SLICES; ++s) v += part[s][t][at];
    if (bias && n < N) v += bias[n];
    put(C, m, n, N, v, m < M && n < N, gated);
  }
}

// ---- up to 8 rows: SP slices of K to a wave ------------------------------------------------------------------------------
// With up to 16 / SP rows of A the matrix instruction's 16 x 16 outputs hold as many rows of W for SP slices at once: lane i's
// row of W and of A is i % B of slice SP wave + i / B (B = 16 / SP), and of the B x B blocks of outputs those on the diagonal are
// a slice's (the others, one slice's rows of A by another's of W, are left).  So a workgroup takes B weight rows instead of 16,
// every load still has work for all lanes, and the order of an element's sum is the one of the other kernels.  Taken where 16
// weight rows to a workgroup leave compute units without one (us at 4 rows, 16 rows : 8 rows : 4 rows to a workgroup)
//   896 x 896 4.5 : 3.5 : 3.1     896 x 4,864 17.2 : 10.5 : 8.8     1,024 x 2,816 11.6 : 7.2 : 6.6    1,536 x 1,536 7.6 : 5.5 : 6.1
//   2,048 x 11,008 38.0 : 23.1 : 27.3     2,560 x 2,048 8.6 : 8.8 : 9.1      4,096 x 4,096 16.7 : 17.5 : 20.3
// or where their last round is far from full and A is little to read (6,144 x 2,048 15.0 : 13.6, 9,728 x 896 11.1 : 10.4; but
// 11,264 x 2,048 22.7 : 25.6).  More than four steps in flight a wave (5, 10, 20) gain at K = 4,864 only (8.0 at 20) and lose elsewhere.
template <typename TA, typename TO, int SP, int STEPS, bool VEC>
__global__ __launch_bounds__(64 * N_SLICES / SP) void gemm_f32_narrow_kernel(const TA* __restrict__ A, const float* __restrict__ W,
                                                                             const float* __restrict__ bias, TO* __restrict__ C,
                                                                             int M, int N, int K, Gated gated) {
  constexpr int B = 16 / SP;
  __shared__ float part[N_SLICES][B * B];
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
  const int i = lane % 16, q = lane / 16, r = i % B, slice = SP * wave + i / B;
  const int n0 = blockIdx.x * B;
  const int len = slice_len(K), k_lo = slice * len, k_hi = min(K, k_lo + len);
  const float* wrow = W + (size_t)min(n0 + r, N - 1) * K;      // (columns beyond N are computed and dropped)
  const TA* arow = A + (size_t)min(r, M - 1) * K;
  const int a_hi = r < M ? k_hi : 0;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < len; k0 += 16 * STEPS) {
    f32x4 w[STEPS], a[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int k = k_lo + k0 + 16 * s + 4 * q;
      w[s] = load4<VEC>(wrow, k, k_hi);
      a[s] = load4<VEC>(arow, k, a_hi);
    }
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s][j], w[s][j], acc, 0, 0, 0);
  }
  // lane (i, q) holds rows 4 q + j of column i
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if ((4 * q + j) / B == i / B) part[slice][(4 * q + j) % B * B + r] = acc[j];
  __syncthreads();
  const int e = threadIdx.x, m = e / B, n = n0 + e % B;
  if (e < B * B) {
    float v = part[0][e];
#pragma unroll
    for (int s = 1; s < N_SLICES; ++s) v += part[s][e];
    if (bias && n < N) v += bias[n];
    put(C, m, n, N, v, m < M && n < N, gated);
  }
}

// ---- the same of q, k and v -------------------------------------------------------------------------------------------------
// A workgroup takes both halves of B / 2 rotation pairs, and bias, rotation (split-half pairs over the whole head) and the write into the paged cache
// are its end, bit for bit those of rope_append, whose launch it saves.  us with the norm's launch before it, two launches / this: 4 rows of 896 in 14 heads of 64
// on 2 8.3 / 6.2, 1 row 7.8 / 5.7, 8 rows 8.7 / 6.5, 4 rows of 1,536 in 12 heads of 128 on 2 10.9 / 8.5, of 2,048 in 6 on 2 10.7 / 8.5.  (That norm, formed by every
// workgroup for itself from the stream, gives 0.1 to 0.3 more here, and costs gate/up with its many workgroups 3; a product that adds to the stream itself instead
// of leaving it to the norm gives nothing.)
struct QkvArgs {
  const float *A, *W, *bias;
  float* q;                 // [M][nH][d]
  int M, N, K;
  const int* slots;         // [M] or null: W holds q alone
  const float *cs, *sn;     // [M][d / 2]
  int nH, nKV, d, page_size;
  float *k_cache, *v_cache;
};

template <int SP>
__global__ __launch_bounds__(64 * N_SLICES / SP) void narrow_qkv_kernel(QkvArgs a) {
  constexpr int B = 16 / SP, STEPS = 4;
  __shared__ float part[N_SLICES][B * B];
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
  const int i = lane % 16, q = lane / 16, r = i % B, slice = SP * wave + i / B;
  const int M = a.M, K = a.K, half = a.d / 2;
  // the weight row of column c of this workgroup, its head and where it stands in it (pairs beyond the last are computed and dropped)
  auto row_at = [&](int c, int& head, int& at) {
    const int p = min((int)blockIdx.x * (B / 2) + c % (B / 2), a.N / 2 - 1);
    head = p / half;
    at = p % half + (c >= B / 2 ? half : 0);
    return head * a.d + at;
  };
  int its_head, its_place;
  const int len = slice_len(K), k_lo = slice * len, k_hi = min(K, k_lo + len), a_hi = r < M ? k_hi : 0;
  const float* wrow = a.W + (size_t)row_at(r, its_head, its_place) * K;
  const float* arow = a.A + (size_t)min(r, M - 1) * K;
  f32x4 w[STEPS], x[STEPS];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      w[s] = load4<true>(wrow, k_lo + k0 + 16 * s + 4 * q, k_hi);
      x[s] = load4<true>(arow, k_lo + k0 + 16 * s + 4 * q, a_hi);
    }
  };
  fetch(0);
  // what the end needs, for the threads that write
  const int e = threadIdx.x, m = e / B, c = e % B;
  int head, at;
  const int n = row_at(c, head, at);
  const bool in = e < B * B && m < M && (int)blockIdx.x * (B / 2) + c % (B / 2) < a.N / 2;
  float bias = 0.f, cs = 0.f, sn = 0.f;
  int slot = -1;
  if (in) {
    if (a.bias) bias = a.bias[n];
    cs = a.cs[(size_t)m * half + at % half], sn = a.sn[(size_t)m * half + at % half];
    if (a.slots) slot = a.slots[m];
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < len; k0 += 16 * STEPS) {
    if (k0 > 0) fetch(k0);
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[s][j], w[s][j], acc, 0, 0, 0);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if ((4 * q + j) / B == i / B) part[slice][(4 * q + j) % B * B + r] = acc[j];
  __syncthreads();
  if (e >= B * B) return;
  float v = part[0][e];
#pragma unroll
  for (int s = 1; s < N_SLICES; ++s) v += part[s][e];
  if (a.bias) v += bias;
  const float other = __shfl_xor(v, B / 2);
  if (!in) return;
  const float turned = other * sn;
  const float y = __builtin_fmaf(v, cs, c < B / 2 ? -turned : turned);
  if (head < a.nH) {
    a.q[(size_t)m * a.nH * a.d + n] = y;
    return;
  }
  if (slot < 0) return;
  const int page = slot / a.page_size, off = slot % a.page_size, h = (head - a.nH) % a.nKV;
  if (head < a.nH + a.nKV) a.k_cache[(((size_t)page * a.nKV + h) * a.page_size + off) * a.d + at] = y;
  else a.v_cache[(((size_t)page * a.nKV + h) * a.d + at) * a.page_size + off] = v;
}

// The slices to a wave with which the products of up to 8 rows take this size, 0: another kernel does.
static int narrow_slices(int M, int N) {
  const double b16 = (N + 15) / 16, full16 = 256.0 * (double)((N + 4095) / 4096);
  if (M <= 4 && N <= 1024) return 4;
  return (M <= 8 && N <= 2048) || (M <= 4 && b16 > 256.0 && b16 < 0.85 * full16) ? 2 : 0;
}
extern "C" int ifx_gemm_f32_narrow_slices(int M, int N) { return M > 0 && N > 0 ? narrow_slices(M, N) : 0; }

// q, k and v of the rows A [M][K] by W [N][K] (both on 16 bytes, K a multiple of 4, sizes that narrow_slices takes) and ``bias`` [N] or null: q to q [M][nH][d],
// k and v at ``slots`` [M] (page * page_size + offset, below 0: not) into the cache; slots null: N holds q alone, nKV 0.
extern "C" int ifx_qkv_rope_f32(const float* A, const float* W, const float* bias, float* q, int M, int N, int K, const int* slots, const float* cs, const float* sn,
                                int nH, int nKV, int d, int page_size, float* k_cache, float* v_cache, void* stream) {
  IFX_REQUIRE(M > 0 && N > 0 && K > 0 && K % 4 == 0 && narrow_slices(M, N) > 0, "qkv_rope_f32: not for M=%d N=%d K=%d", M, N, K);
  IFX_REQUIRE(((uintptr_t)A | (uintptr_t)W) % 16 == 0, "qkv_rope_f32: rows and weight must lie on 16 bytes");
  IFX_REQUIRE(cs && sn && nH > 0 && nKV >= 0 && d > 0 && d % 2 == 0 && N == (nH + 2 * nKV) * d && (slots ? nKV > 0 && page_size > 0 && k_cache && v_cache : nKV == 0),
              "qkv_rope_f32: %d rows of weight for %d + %d heads of %d", N, nH, nKV, d);
  const QkvArgs a{A, W, bias, q, M, N, K, slots, cs, sn, nH, nKV, d, page_size, k_cache, v_cache};
  const int sp = narrow_slices(M, N);
  const dim3 grid((N + 16 / sp - 1) / (16 / sp)), threads(64 * N_SLICES / sp);
  hipStream_t s = (hipStream_t)stream;
  if (sp == 4) hipLaunchKernelGGL((narrow_qkv_kernel<4>), grid, threads, 0, s, a);
  else hipLaunchKernelGGL((narrow_qkv_kernel<2>), grid, threads, 0, s, a);
  IFX_LAUNCH_CHECK();
}

// ---- many rows: tiles of A and W through LDS -----------------------------------------------------------------------------
// A workgroup of four waves makes (32 TM) x (32 TN) outputs, two waves by two; a step of 32 k-values goes through LDS, the next
// one is on its way from memory meanwhile.  Bound by the matrix units: a wave reads TM + TN fragments of 16 bytes a lane for
// 4 TM TN instructions of 32 cycles.  LDS rows of 32 floats, the eight pieces of 16 bytes of a row placed by piece ^ (row % 8):
// the 16 lanes of a fragment's quarter then lie in different banks without padding.
template <typename TA, typename TO, int TM, int TN, bool VEC>
__global__ __launch_bounds__(256) void gemm_f32_tiles_kernel(const TA* __restrict__ A, const float* __restrict__ W,
                                                             const float* __restrict__ bias, TO* __restrict__ C,
                                                             int M, int N, int K, Gated gated) {
  constexpr int BM = 32 * TM, BN = 32 * TN, BK = 32;
  __shared__ f32x4 As[BM][BK / 4], Ws[BN][BK / 4];
  const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
  const int i = lane % 16, q = lane / 16;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int wm = (wave / 2) * 16 * TM, wn = (wave % 2) * 16 * TN;
  const int len = slice_len(K);
  const int pr = tid / 8, pp = tid % 8;                    // the row (of 32) and the piece this thread brings in
  f32x4 acc[TM][TN], total[TM][TN], na[TM], nw[TN];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) acc[m][n] = total[m][n] = (f32x4){0.f, 0.f, 0.f, 0.f};
  auto fetch = [&](int k0, int k_hi) {
    const int k = k0 + 4 * pp;
#pragma unroll
    for (int r = 0; r < TM; ++r) {
      const int m = m0 + 32 * r + pr;
      na[r] = (f32x4){0.f, 0.f, 0.f, 0.f};
      if (m < M) na[r] = load4<VEC>(A + (size_t)m * K, k, k_hi);
    }
#pragma unroll
    for (int r = 0; r < TN; ++r) {
      const int n = n0 + 32 * r + pr;
      nw[r] = (f32x4){0.f, 0.f, 0.f, 0.f};
      if (n < N) nw[r] = load4<VEC>(W + (size_t)n * K, k, k_hi);
    }
  };
  fetch(0, min(K, len));
  for (int k_lo = 0, s = 0; k_lo < K; k_lo += len, ++s) {
    const int k_hi = min(K, k_lo + len);
    for (int k0 = k_lo; k0 < k_hi; k0 += BK) {
      __syncthreads();
#pragma unroll
      for (int r = 0; r < TM; ++r) As[32 * r + pr][pp ^ (pr % 8)] = na[r];
#pragma unroll
      for (int r = 0; r < TN; ++r) Ws[32 * r + pr][pp ^ (pr % 8)] = nw[r];
      __syncthreads();
      if (k0 + BK < k_hi) fetch(k0 + BK, k_hi);
      else if (k_hi < K) fetch(k_hi, min(K, k_hi + len));
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (k0 + 16 * h >= k_hi) break;                    // (a slice may end in the middle of a step: its length is a multiple of 16)
        f32x4 a[TM], w[TN];
#pragma unroll
        for (int m = 0; m < TM; ++m) a[m] = As[wm + 16 * m + i][(4 * h + q) ^ (i % 8)];
#pragma unroll
        for (int n = 0; n < TN; ++n) w[n] = Ws[wn + 16 * n + i][(4 * h + q) ^ (i % 8)];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int m = 0; m < TM; ++m)
#pragma unroll
            for (int n = 0; n < TN; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m][j], w[n][j], acc[m][n], 0, 0, 0);
      }
    }
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        total[m][n] = s == 0 ? acc[m][n] : total[m][n] + acc[m][n];
        acc[m][n] = (f32x4){0.f, 0.f, 0.f, 0.f};
      }
  }
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      const int col = n0 + wn + 16 * n + i;
      const float b = bias && col < N ? bias[col] : 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + 16 * m + 4 * q + r;
        put(C, row, col, N, bias ? total[m][n][r] + b : total[m][n][r], row < M && col < N, gated);
      }
    }
}

// The same of float rows on 16 bytes: a step's rows go straight to LDS, two steps ahead of their use and with one barrier a step, and three workgroups share a compute unit.
// 470 rows of 9,728 x 896 108 -> 94 us, 2,000 366 -> 315, 4,000 of 896 x 4,864 413 -> 348 (100 to 113 TFLOP/s).
template <typename TO, int TM, int TN>
__global__ __launch_bounds__(256) void gemm_f32_walk_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                                                            TO* __restrict__ C, int M, int N, int K, Gated gated) {
  constexpr int BM = 32 * TM, BN = 32 * TN, BK = 32, ROWS = BM + BN, SLOTS = 3, LOADS = ROWS / 32;      // direct loads of a wave and a step, 8 rows of 128 bytes each
  __shared__ __attribute__((aligned(1024))) f32x4 stage[SLOTS][ROWS][BK / 4];
  const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int i = lane % 16, q = lane / 16;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int wm = (wave / 2) * 16 * TM, wn = (wave % 2) * 16 * TN;
  const int len = slice_len(K), steps = (len + BK - 1) / BK;
  // (rows beyond the last lie beyond the buffer's end and are zeros)
  const tile_uintx4 ab = tile_buffer(A + (size_t)m0 * K, (unsigned)min(BM, M - m0) * (unsigned)K * 4u), wb = tile_buffer(W + (size_t)n0 * K, (unsigned)min(BN, N - n0) * (unsigned)K * 4u);
  const unsigned base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)&stage[0][0][0];
  int offset[LOADS];                                      // of this lane's piece (of a row's eight the one that lands at lane % 8) in step 0
  const int piece = 4 * (lane % 8 ^ lane / 8);
#pragma unroll
  for (int l = 0; l < LOADS; ++l) {
    const int row = 8 * (wave * LOADS + l) + lane / 8;
    offset[l] = ((row < BM ? row : row - BM) * K + piece) * 4;
  }
  int ask_lo = 0, ask_step = 0;                           // the slice and the step in it to ask for next
  auto ask = [&](int slot) {
    const int k_hi = min(K, ask_lo + len), k = ask_lo + BK * ask_step;
#pragma unroll
    for (int l = 0; l < LOADS; ++l) {
      const int eight = wave * LOADS + l;
      tile_direct_load(eight < BM / 8 ? ab : wb, k + piece < k_hi ? offset[l] + 4 * k : TILE_NO_ROW, base + slot * (ROWS * 128) + eight * 1024);
    }
    if (++ask_step == steps) ask_step = 0, ask_lo += len;
  };
  f32x4 acc[TM][TN], total[TM][TN];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) acc[m][n] = total[m][n] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < SLOTS - 1; ++s) ask(s);
  int slot = 0;
  for (int k_lo = 0; k_lo < K; k_lo += len) {
    const int k_hi = min(K, k_lo + len);
    for (int step = 0; step < steps; ++step) {
      tile_meet<(SLOTS - 2) * LOADS>();                   // the step is there, and everyone has read the one before it
      ask(slot == 0 ? SLOTS - 1 : slot - 1);
      f32x4(*As)[BK / 4] = stage[slot], (*Ws)[BK / 4] = stage[slot] + BM;
      slot = slot == SLOTS - 1 ? 0 : slot + 1;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (k_lo + BK * step + 16 * h >= k_hi) break;      // (the end of the slice, whose length is a multiple of 16, or of K)
        f32x4 a[TM], w[TN];
#pragma unroll
        for (int m = 0; m < TM; ++m) a[m] = As[wm + 16 * m + i][(4 * h + q) ^ (i % 8)];
#pragma unroll
        for (int n = 0; n < TN; ++n) w[n] = Ws[wn + 16 * n + i][(4 * h + q) ^ (i % 8)];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int m = 0; m < TM; ++m)
#pragma unroll
            for (int n = 0; n < TN; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m][j], w[n][j], acc[m][n], 0, 0, 0);
      }
    }
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        total[m][n] = k_lo == 0 ? acc[m][n] : total[m][n] + acc[m][n];
        acc[m][n] = (f32x4){0.f, 0.f, 0.f, 0.f};
      }
  }
  tile_meet<0>();                                         // (the loads beyond the end have landed before the workgroup leaves)
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      const int col = n0 + wn + 16 * n + i;
      const float b = bias && col < N ? bias[col] : 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + 16 * m + 4 * q + r;
        put(C, row, col, N, bias ? total[m][n][r] + b : total[m][n][r], row < M && col < N, gated);
      }
    }
}

// ---- hundreds of rows: tiles of A and W through LDS, the slices of K side by side --------------------------------------------------
// Four groups of four waves take four slices of K each and all of them the same (32 TM) x (32 TN) outputs, with a stage of LDS of their own, in step; the slices' sums
// stay apart, 16 TM TN registers of them, and are added up in their order by the groups one after the other.  Sixteen waves keep the matrix units of a compute unit busy
// where the walk of the kernel above, four waves through all of K, waits at its barriers, and a step's rows are read once for 32 TM or 32 TN outputs, where the kernel of
// sixteen slices without LDS reads them from the caches for 16 or 32.  A step of 32 k-values of all groups goes straight to LDS, two or three ahead of its use (one with
// tiles of 64 x 64; by way of registers, one step ahead, a step took 1.3 to 1.7 times as long).  us, the others' best / here: 470 rows of 896 x 4,864 97 / 56, 1,536 x 8,960
// 255 / 160, 2,048 x 1,536 51 / 35, 1,152 x 896 28 / 24, 896 x 896 21 / 16; 200 rows of 896 x 4,864 52 / 36, 2,048 x 2,048 42 / 27; 64 of 9,728 x 896 31 / 24; many
// rounds of them are no faster (470 of 9,728 x 896 101 / 105).
template <typename TO, int TM, int TN>
__global__ __launch_bounds__(1024) void gemm_f32_groups_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                                                               TO* __restrict__ C, int M, int N, int K, Gated gated) {
  constexpr int BM = 32 * TM, BN = 32 * TN, BK = 32, GROUPS = 4, PER = N_SLICES / GROUPS, ROWS = BM + BN;
  constexpr int SLOTS = TM * TN == 1 ? 4 : TM * TN == 2 ? 3 : 2, LOADS = ROWS / 32;      // direct loads of a wave and a step, 8 rows of 128 bytes each
  __shared__ __attribute__((aligned(1024))) f32x4 stage[SLOTS][GROUPS][ROWS][BK / 4];
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / 256), lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x % 256 / WAVE);
  const int i = lane % 16, q = lane / 16;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int wm = (wave / 2) * 16 * TM, wn = (wave % 2) * 16 * TN;
  const int len = slice_len(K), steps = (len + BK - 1) / BK;
  // (rows beyond the last lie beyond the buffer's end and are zeros)
  const tile_uintx4 ab = tile_buffer(A + (size_t)m0 * K, (unsigned)min(BM, M - m0) * (unsigned)K * 4u), wb = tile_buffer(W + (size_t)n0 * K, (unsigned)min(BN, N - n0) * (unsigned)K * 4u);
  const unsigned base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)&stage[0][group][0][0];
  const int piece = 4 * (lane % 8 ^ lane / 8);            // of a row's eight the one that lands at lane % 8
  int ask_slice = 0, ask_step = 0;                        // the next step to ask for
  auto ask = [&](int slot) {
    const int k_lo = (PER * group + ask_slice) * len, k_hi = ask_slice < PER ? min(K, k_lo + len) : 0, k = k_lo + BK * ask_step + piece;
#pragma unroll
    for (int l = 0; l < LOADS; ++l) {
      const int eight = wave * LOADS + l, row = 8 * eight + lane / 8;
      const bool of_a = eight < BM / 8;
      tile_direct_load(of_a ? ab : wb, k < k_hi ? ((of_a ? row : row - BM) * K + k) * 4 : TILE_NO_ROW, base + slot * (GROUPS * ROWS * 128) + eight * 1024);
    }
    if (++ask_step == steps) ask_step = 0, ++ask_slice;
  };
  f32x4 acc[PER][TM][TN];
#pragma unroll
  for (int s = 0; s < PER; ++s)
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int n = 0; n < TN; ++n) acc[s][m][n] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < SLOTS - 1; ++s) ask(s);
  int slot = 0;
#pragma unroll
  for (int s = 0; s < PER; ++s) {
    const int k_lo = (PER * group + s) * len, k_hi = min(K, k_lo + len);
    for (int step = 0; step < steps; ++step) {
      tile_meet<(SLOTS - 2) * LOADS>();                   // the step is there, and everyone has read the one before it
      ask(slot == 0 ? SLOTS - 1 : slot - 1);
      f32x4(*As)[BK / 4] = stage[slot][group], (*Ws)[BK / 4] = stage[slot][group] + BM;
      slot = slot == SLOTS - 1 ? 0 : slot + 1;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (k_lo + BK * step + 16 * h >= k_hi) break;      // (the end of the slice, whose length is a multiple of 16, or of K)
        f32x4 a[TM], w[TN];
#pragma unroll
        for (int m = 0; m < TM; ++m) a[m] = As[wm + 16 * m + i][(4 * h + q) ^ (i % 8)];
#pragma unroll
        for (int n = 0; n < TN; ++n) w[n] = Ws[wn + 16 * n + i][(4 * h + q) ^ (i % 8)];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int m = 0; m < TM; ++m)
#pragma unroll
            for (int n = 0; n < TN; ++n) acc[s][m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m][j], w[n][j], acc[s][m][n], 0, 0, 0);
      }
    }
  }
  tile_meet<0>();                                         // (the loads beyond the end)
  // the groups in turn: what the ones before have added up, and this one's slices in ascending order
  f32x4* sums = &stage[0][0][0][0];          // [wave][TM][TN][lane]
  static_assert(4 * TM * TN * WAVE <= GROUPS * ROWS * (BK / 4), "the sums fit the stages' place");
#pragma unroll 1
  for (int g = 0; g < GROUPS; ++g) {
    __syncthreads();
    if (g != group) continue;
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        f32x4& at = sums[((wave * TM + m) * TN + n) * WAVE + lane];
        f32x4 total = g == 0 ? acc[0][m][n] : at + acc[0][m][n];
#pragma unroll
        for (int s = 1; s < PER; ++s) total = total + acc[s][m][n];
        if (g < GROUPS - 1) at = total;
        else acc[0][m][n] = total;
      }
  }
  if (group < GROUPS - 1) return;
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      const int col = n0 + wn + 16 * n + i;
      const float b = bias && col < N ? bias[col] : 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + 16 * m + 4 * q + r;
        put(C, row, col, N, bias ? acc[0][m][n][r] + b : acc[0][m][n][r], row < M && col < N, gated);
      }
    }
}

// Which kernel: the one with the lowest estimate of its time, all but the groups' in proportion to K (of more than 3,000 a fifth less).  A kernel's grid runs in rounds of
// 256 workgroups (one for each compute unit; sixteen waves fill it, and two workgroups of the tile kernel share one).  A round
// at K = 896 was measured at 5.6 us for 16 x 16 outputs, 7.5 for 32 x 16 and 10.3 for 32 x 32 with the slices side by side; the
// tile kernel, which walks K in one go, takes 31 us for up to 256 tiles of 64 x 64 and 0.083 us a tile beyond that (but not
// less than 44), with direct loads 12 us and 16 for each 256 tiles.  Before these kernels (one thread summing an output, tiles of 64 x 64, scalar loads) a product took 83 us at
// 1 row and 102 at 475 of 896 x 896 (now, in a graph, 2.8 and 14.4), 449 and 559 of 896 x 4,864 (8.5 and 54), 90 and 266 of 9,728 x 896 (10.0
// and 87), 410 at one row of 151,936 x 896 (103: 5.3 TB/s); 2,048 rows of 22,016 x 2,048 run at 121 TFLOP/s.  Errors against 64
// bits fell to a third (5.4e-7 to 2.0e-7 at K = 896, 1.9e-6 to 6.6e-7 at 11,008): shorter chains.
template <typename TA, typename TO, bool VEC>
static void launch(const TA* A, const float* W, const float* bias, TO* C, int M, int N, int K, Gated gated, hipStream_t s) {
  auto blocks = [&](int m, int n) { return (double)((M + m - 1) / m) * ((N + n - 1) / n); };
  auto rounds = [&](int m, int n) { return (double)(long long)((blocks(m, n) + 255.0) / 256.0); };
  const double t11 = 5.6 * rounds(16, 16), t21 = 7.5 * rounds(32, 16), t22 = 10.3 * rounds(32, 32);
  constexpr bool direct = VEC && sizeof(TA) == 4;          // (rows that may go straight to LDS)
  const double b64 = blocks(64, 64), tiles = direct ? 12.0 + 16.0 * rounds(64, 64) : b64 <= 256.0 ? 31.0 : (b64 < 530.0 ? 44.0 : 0.083 * b64);
#define FEW(MT, NT)                                                                                              \
  hipLaunchKernelGGL((gemm_f32_few_kernel<TA, TO, MT, NT, 4, VEC>),                                              \
                     dim3((N + 16 * NT - 1) / (16 * NT), (M + 16 * MT - 1) / (16 * MT)), dim3(1024), 0, s, A, W, bias, C, M, N, K, gated)
  // (a grid has at most 65,535 rows: millions of rows by a handful of columns are the tile kernel's, whose limit the caller checks)
  const bool in16 = (M + 15) / 16 <= 65535, in32 = (M + 31) / 32 <= 65535;
#define GROUPS_(TM, TN)                                                                                          \
  hipLaunchKernelGGL((gemm_f32_groups_kernel<TO, TM, TN>), dim3((N + 32 * TN - 1) / (32 * TN), (M + 32 * TM - 1) / (32 * TM)), dim3(1024), 0, s, (const float*)A, W, bias, C, M, N, K, gated)
#define NARROW(SP, STEPS)                                                                                        \
  hipLaunchKernelGGL((gemm_f32_narrow_kernel<TA, TO, SP, STEPS, VEC>), dim3((N + 16 / SP - 1) / (16 / SP)),      \
                     dim3(64 * N_SLICES / SP), 0, s, A, W, bias, C, M, N, K, gated)
  // the groups' tiles: a round of them, and each 1,000 k-values of it (which of them, -1: another kernel)
  static const struct { int bm, bn; double round, per_k; } kinds[4] = {{32, 32, 5.4, 5.75}, {64, 32, 6.2, 9.65}, {32, 64, 6.2, 9.65}, {64, 64, 7.7, 16.7}};
  int groups = -1;
  if (direct && in32 && K <= 1 << 22) {
    double least = fmin(fmin(in16 ? t11 : 1e30, fmin(t21, t22)), tiles) * (K / 896.0) * (K > 3000 ? 0.82 : 1.0);
    for (int k = 0; k < 4; ++k) {
      const double us = rounds(kinds[k].bm, kinds[k].bn) * (kinds[k].round + kinds[k].per_k * K / 1000.0);
      if (us < least) least = us, groups = k;
    }
  }
  const int narrow = narrow_slices(M, N);
  if (narrow == 4) NARROW(4, 4);
  else if (narrow == 2) NARROW(2, 4);
  else if (M > 16 && groups == 0) GROUPS_(1, 1);
  else if (M > 16 && groups == 1) GROUPS_(2, 1);
  else if (M > 16 && groups == 2) GROUPS_(1, 2);
  else if (M > 16 && groups == 3) GROUPS_(2, 2);
  else if (M <= 16 || (in16 && t11 <= t21 && t11 <= t22 && t11 <= tiles)) FEW(1, 1);
  else if (in32 && t21 <= t22 && t21 <= tiles) FEW(2, 1);
  else if (in32 && t22 <= tiles) FEW(2, 2);
  else if (direct && K <= 1 << 22)
    hipLaunchKernelGGL((gemm_f32_walk_kernel<TO, 2, 2>), dim3((N + 63) / 64, (M + 63) / 64), dim3(256), 0, s, (const float*)A, W, bias, C, M, N, K, gated);
  else
    // (float rows beyond 4M k-values, whose tiles no buffer's offsets reach, go with those that do not lie on 16 bytes)
    hipLaunchKernelGGL((gemm_f32_tiles_kernel<TA, TO, 2, 2, VEC && !direct>), dim3((N + 63) / 64, (M + 63) / 64), dim3(256), 0, s, A, W, bias, C, M, N, K, gated);
#undef FEW
#undef GROUPS_
#undef NARROW
}

// act: -1, or the activation of gate and up rows in turn (N even, no bias, C [M][N / 2] of A's type)
extern "C" int ifx_gemm_f32(const void* A, int a_dtype, const float* W, const float* bias, void* C,
                            int c_dtype, int M, int N, int K, int act, float limit, void* stream) {
  IFX_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
  IFX_REQUIRE(act < 0 || (N % 2 == 0 && !bias && a_dtype == DT_F32 && c_dtype == DT_F32 &&
                          (act == ACT_SILU || act == ACT_GELU_TANH || (act == ACT_CLAMPED_SWISH && limit > 0.f))),
              "gemm_f32: gated activation %d (limit %g) of %d columns", act, (double)limit, N);
  const Gated gated{act, limit};
  if (M == 0) return 0;
  IFX_REQUIRE((M + 63) / 64 <= 65535, "gemm_f32: M=%d too large for one launch", M);
  hipStream_t s = (hipStream_t)stream;
  const bool vec = K % 4 == 0 && (uintptr_t)W % 16 == 0 && (uintptr_t)A % (a_dtype == DT_BF16 ? 8 : 16) == 0;
#define LAUNCH(TA, TO)                                                              \
  do {                                                                              \
    if (vec) launch<TA, TO, true>((const TA*)A, W, bias, (TO*)C, M, N, K, gated, s);       \
    else launch<TA, TO, false>((const TA*)A, W, bias, (TO*)C, M, N, K, gated, s);          \
  } while (0)
  if (a_dtype == DT_F32 && c_dtype == DT_F32) LAUNCH(float, float);
  else if (a_dtype == DT_BF16 && c_dtype == DT_BF16) LAUNCH(bf16_t, bf16_t);
  else if (a_dtype == DT_BF16 && c_dtype == DT_F32) LAUNCH(bf16_t, float);
  else if (a_dtype == DT_F32 && c_dtype == DT_BF16) LAUNCH(float, bf16_t);
  else IFX_FAIL("gemm_f32: unknown dtypes a=%d c=%d", a_dtype, c_dtype);
#undef LAUNCH
  IFX_LAUNCH_CHECK();
}
