// A mixture of experts for steps of few rows (up to 64, bfloat16), on the matrix cores: every chosen expert's weights are
// streamed once, whatever the number of rows that chose it.
//
//   ifx_moe_logits         the router's logits, as partial sums over slices of K
//   ifx_moe_choose         scores, choice and weights of every row from the logits (the same function as ifx_moe_route of
//                          moe.hip)
//   ifx_moe_few_gate_up    act[item][:] = activation(Wg[e] x, Wu[e] x) for the (row, choice) items and their experts e, from
//                          weights whose rows alternate 16 of Wg with 16 of Wu
//   ifx_moe_few_down       parts[choice][row][:] = weight[item] * Wd[e] act[item] in float; the kernel that adds the result to
//                          the stream sums the choices in order
// Rows may come up to a norm's factor (row_scale.h, up to 16 rows): the logits' product forms it beside its own loads, multiplies
// the logits by it and leaves it for the experts' products, which multiply their sums by it; the norm's own launch is saved.
// Identity experts (ids from `n_real` on) and weights on the experts' inputs are those of grouped_gemm.hip.  A shared expert, which
// every row takes with weight 1, runs in the same launches: its rows are workgroups of their own ahead of the experts', its output
// one more part.  As two products, an activation's launch and the launch that added it, one row of 2,048 values to a shared
// expert of 1,408 took 19.5 us beside its experts, now 7.5.
//
// The products are bound by the chosen experts' bytes.  A workgroup takes an expert and NT x 16 of its weight rows and finds the
// expert's items itself, from the step's few ids (no ordered list, no launch that makes one); its waves split K, meet in LDS in
// wave order, and a wave has U x 64 k-values of the rows in flight.  The items are the columns of the matrix instruction (MT x 16
// at a time), so an item's sums depend on its own row and on how K is dealt to the waves: by twos of 64 k-values, or in gate/up of
// up to 16 rows by threes, so there the bits of a row may differ from those in a step of more rows.  The weights lie in tiles (1 KB of contiguous memory to a wave's
// load): from plain rows the same kernels take 1.1 to 1.3 times as long.
//
// Experts of 2,048 x 1,408 (us for a whole mixture: router, choice, both products; against a wave per output element that reads
// an expert again for every item, and from 64 items on tiles of 64 items of one expert through LDS, with the router's launches):
// 64 experts of which a row takes 6, at 1 / 8 / 16 / 64 rows 30 / 102 / 150 / 180 (53 / 142 / 230 / 264; the chosen experts'
// bytes at 6.5 TB/s: 16 / 93 / 141 / 170); 32 experts, 4 to a row, 23 / 66 / 86 / 99 (32 / 97 / 125 / 153; 11 / 53 / 77 / 85).
#include "common.h"
#include "row_scale.h"

IFX_DEFINE_LAST_ERROR()

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

#define MAX_E 256
#define MAX_TOP 32
#define MAX_ROWS 64

// ---- logits, scores, choice, lists ----------------------------------------------------------------------------------------
__device__ __forceinline__ bf16x8 zero8() {
  bf16x8 z;
#pragma unroll
  for (int i = 0; i < 8; ++i) z[i] = (__bf16)0.f;
  return z;
}

// The router's logits as partial sums over up to LOGIT_SLICES slices of K: z[slice][row][expert] in float.  A workgroup takes 16
// experts and one slice, a wave 16 rows of x.  A router is a handful of weight rows, so what counts is the number of trips to
// memory: with 128 k-values to a slice a wave asks for all it needs at once and stores what comes out, nothing is added up
// here (the kernel that chooses reads the slices side by side).
#define LOGIT_SLICES 16
__global__ __launch_bounds__(256) void moe_logits_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, float* __restrict__ z,
                                                         int T, int K, int E, int slice_blocks, RowScale scale, float* __restrict__ factor) {
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE, col = lane & 15, g = lane >> 4;
  const int e0 = 16 * blockIdx.x, m = 16 * wave + col;
  const bf16_t* wrow = w + (size_t)min(e0 + col, E - 1) * K;
  const bf16_t* xrow = x + (size_t)min(m, T - 1) * K;
  floatx4 acc{0.f, 0.f, 0.f, 0.f};
  // (its loads go out ahead of the first of W, which are waited for together)
  const float f = scale.pieces ? row_factor(scale, lane) : 1.f;
  const int kb_end = min((K + 63) / 64, (int)(blockIdx.y + 1) * slice_blocks);
  for (int kb0 = blockIdx.y * slice_blocks; kb0 < kb_end; kb0 += 2) {
    bf16x8 wv[4], xv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = (kb0 + i / 2) * 64 + 16 * g + 8 * (i % 2);
      const bool in = kb0 + i / 2 < kb_end && k < K;
      wv[i] = in ? *(const bf16x8*)(wrow + k) : zero8();
      xv[i] = in ? *(const bf16x8*)(xrow + k) : zero8();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[i], xv[i], acc, 0, 0, 0);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (m < T && e0 + 4 * g + r < E) z[((size_t)blockIdx.y * T + m) * E + e0 + 4 * g + r] = acc[r] * f;
  if (scale.pieces && blockIdx.x == 0 && blockIdx.y == 0 && lane < T) factor[lane] = f;
}

static int logit_slice_blocks(int K) {                  // blocks of 64 k-values to a slice
  const int nkb = (K + 63) / 64, per = (nkb + LOGIT_SLICES - 1) / LOGIT_SLICES;
  return per < 2 ? 2 : per;
}
extern "C" int ifx_moe_logit_slices(int K) { return ((K + 63) / 64 + logit_slice_blocks(K) - 1) / logit_slice_blocks(K); }

extern "C" int ifx_moe_logits(const void* x, const void* w, float* z, int T, int K, int E, const float* pieces, int n_pieces,
                              float width, float eps, float* factor, void* stream) {
  IFX_REQUIRE(!pieces || (T <= 16 && n_pieces > 0 && width > 0.f && factor), "moe_logits: bad row factors (%d rows, %d pieces, width %g)", T, n_pieces, (double)width);
  IFX_REQUIRE(T > 0 && T <= MAX_ROWS && E > 0 && K > 0 && K % 8 == 0, "moe_logits: %d rows (at most %d), %d experts, K=%d (a multiple of 8)", T, MAX_ROWS, E, K);
  hipLaunchKernelGGL(moe_logits_kernel, dim3((E + 15) / 16, ifx_moe_logit_slices(K)), dim3((T + 15) / 16 * WAVE), 0, (hipStream_t)stream,
                     (const bf16_t*)x, (const bf16_t*)w, z, T, K, E, logit_slice_blocks(K), RowScale{pieces, n_pieces, width, eps}, factor);
  IFX_LAUNCH_CHECK();
}

struct ChooseArgs {
  const float* z;            // [slices][T][E] the router's logits as partial sums
  const float* bias;         // [E] added to them, or null
  const float* choice_bias;  // [E] added to the scores for the choice alone, or null
  int* ids; float* weights;  // [T][top]
  int T, E, slices, top, groups, keep, group_top, softmax, renorm;
  float scale;
};

// The largest of a wave's 64 values, the same in every lane (data-parallel moves between neighbouring lanes, no trip to LDS).
__device__ __forceinline__ float lanes_max(float v) {
#define STEP(CTRL, ROWS) v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL, ROWS, 0xf, false)))
  STEP(0x111, 0xf);          // lane l takes lane l - 1 of its row of 16, then l - 2, - 4, - 8
  STEP(0x112, 0xf);
  STEP(0x114, 0xf);
  STEP(0x118, 0xf);
  STEP(0x142, 0xa);          // a row's last lane to the next row, then the first half's last lane to the second half
  STEP(0x143, 0xc);
#undef STEP
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// The number of the highest of the values v (number l + 64 r in lane l's r-th register), the lowest among equals.
template <int R>
__device__ __forceinline__ int highest(const float (&v)[R]) {
  float m = v[0];
#pragma unroll
  for (int r = 1; r < R; ++r) m = fmaxf(m, v[r]);
  m = lanes_max(m);
  int at = 0;
#pragma unroll
  for (int r = R - 1; r >= 0; --r) {
    const unsigned long long has = __ballot(v[r] == m);
    if (has) at = WAVE * r + __ffsll(has) - 1;
  }
  return at;
}

// A wave to a row, lane l its experts l + 64 r.  A choice is `top` times the highest that is left (after `keep` times the best
// group that is left).  Bound by its own chain of instructions: 3.9 to 4.6 us with eight groups of eight experts, where a workgroup that
// counted for every expert how many beat it, through LDS, took 18 (the logits' product included).
template <int R>
__global__ __launch_bounds__(WAVE) void moe_choose_kernel(ChooseArgs a) {
  __shared__ float key[WAVE * R];
  const int t = blockIdx.x, lane = threadIdx.x;
  float s[R], c[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int e = lane + WAVE * r;
    s[r] = -INFINITY;
    if (e < a.E) {
      const float* z = a.z + (size_t)t * a.E + e;
      float p[LOGIT_SLICES];
#pragma unroll
      for (int i = 0; i < LOGIT_SLICES; ++i) p[i] = i < a.slices ? z[(size_t)i * a.T * a.E] : 0.f;
      float v = p[0];
#pragma unroll
      for (int i = 1; i < LOGIT_SLICES; ++i) v += p[i];
      s[r] = v + (a.bias ? a.bias[e] : 0.f);
    }
  }
  if (a.softmax) {
    float m = s[0], l = 0.f;
#pragma unroll
    for (int r = 1; r < R; ++r) m = fmaxf(m, s[r]);
    m = lanes_max(m);
#pragma unroll
    for (int r = 0; r < R; ++r) l += lane + WAVE * r < a.E ? expf(s[r] - m) : 0.f;
    l = wave_sum(l);
#pragma unroll
    for (int r = 0; r < R; ++r) s[r] = expf(s[r] - m) / l;
  } else {
#pragma unroll
    for (int r = 0; r < R; ++r) s[r] = 1.0f / (1.0f + expf(-s[r]));
  }
  // what the choice goes by: always a number above -infinity, which stands for an expert that cannot be chosen (any more)
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int e = lane + WAVE * r;
    c[r] = e < a.E ? fmaxf(a.choice_bias ? s[r] + a.choice_bias[e] : s[r], -3.0e38f) : -INFINITY;
  }
  if (a.keep < a.groups) {
    const int per = a.E / a.groups;
#pragma unroll
    for (int r = 0; r < R; ++r) key[lane + WAVE * r] = c[r];
    __syncthreads();
    float worth[R];                                // a group is worth the sum of its group_top highest, added in falling order
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int g = lane + WAVE * r;
      worth[r] = -INFINITY;
      if (g < a.groups) {
        float best[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) best[i] = -INFINITY;
        for (int i0 = 0; i0 < per; i0 += 8) {
          float v[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) v[i] = i0 + i < per ? key[g * per + i0 + i] : -INFINITY;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            if (j >= a.group_top) break;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const float hi = fmaxf(best[j], v[i]);
              v[i] = fminf(best[j], v[i]);
              best[j] = hi;
            }
          }
        }
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) sum += j < a.group_top && j < per ? best[j] : 0.f;
        worth[r] = fmaxf(sum, -3.0e38f);
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) key[lane + WAVE * r] = 0.f;
    __syncthreads();
    for (int i = 0; i < a.keep; ++i) {
      const int g = highest(worth);
      if (lane == 0) key[g] = 1.f;
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (lane + WAVE * r == g) worth[r] = -INFINITY;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (lane + WAVE * r < a.E && key[(lane + WAVE * r) / per] == 0.f) c[r] = -INFINITY;
  }
  float mine = 0.f, total = 0.f;
  int my_id = 0;
  for (int j = 0; j < a.top; ++j) {
    const int e = highest(c);
    float v = s[0];
#pragma unroll
    for (int r = 1; r < R; ++r) v = e / WAVE == r ? s[r] : v;
    v = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), e % WAVE));
    total += v;
    if (lane == j) { mine = v; my_id = e; }
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (lane + WAVE * r == e) c[r] = -INFINITY;
  }
  if (lane < a.top) {
    a.ids[t * a.top + lane] = my_id;
    a.weights[t * a.top + lane] = (a.renorm ? mine / total : mine) * a.scale;
  }
}

extern "C" int ifx_moe_choose(const float* z, int slices, int* ids, float* weights, int T, int E, int top, int groups, int keep,
                              int group_top, int softmax, int renorm, float scale, const float* bias, const float* choice_bias, void* stream) {
  IFX_REQUIRE(T > 0 && T <= MAX_ROWS && E > 0 && E <= MAX_E, "moe_choose: %d rows (at most %d), %d experts (at most %d)", T, MAX_ROWS, E, MAX_E);
  IFX_REQUIRE(groups > 0 && E % groups == 0 && keep > 0 && keep <= groups, "moe_choose: %d experts in %d groups of which %d are kept", E, groups, keep);
  IFX_REQUIRE(group_top > 0 && group_top <= 8, "moe_choose: a group's score sums its %d largest (1-8)", group_top);
  IFX_REQUIRE(top > 0 && top <= MAX_TOP && top <= keep * (E / groups), "moe_choose: top %d of %d x %d experts", top, keep, E / groups);
  IFX_REQUIRE(slices > 0 && slices <= LOGIT_SLICES, "moe_choose: logits in %d slices (1-%d)", slices, LOGIT_SLICES);
  ChooseArgs a{z, bias, choice_bias, ids, weights, T, E, slices, top, groups, keep, group_top, softmax, renorm, scale};
  if (E <= WAVE) hipLaunchKernelGGL(moe_choose_kernel<1>, dim3(T), dim3(WAVE), 0, (hipStream_t)stream, a);
  else hipLaunchKernelGGL(moe_choose_kernel<4>, dim3(T), dim3(WAVE), 0, (hipStream_t)stream, a);
  IFX_LAUNCH_CHECK();
}

// ---- the products ------------------------------------------------------------------------------------------------------------
struct FewArgs {
  const bf16_t* x;          // item i reads K values from x + (i / x_div) * K
  const bf16_t* w;          // [experts][N][K], or its tiled form (k_tiles > 0; see ifx_tile_weights in gemm_bf16.hip, tiles of 16 rows)
  void* out;
  const int* ids;           // [items] the items' experts
  const float* weights;     // [items]
  const bf16_t* identity;   // DOWN: [T][N], what an identity expert hands back
  int K, N, x_div, T, top, n_real, act;
  int by_item;              // blockIdx.y counts items, not experts: the first item that chose an expert stands for it
  float limit;
  int weigh_input;          // the weight is on an expert's input: gate/up multiplies its sums by it, down leaves it out
  int k_tiles;              // tiled: tiles of 32 k-values to a row tile, an even number; 0: plain rows
  // the shared expert: the first shared_y rows of workgroups (0: there is none), all T rows its items
  int shared_y, shared_k, shared_n, shared_k_tiles;
  const bf16_t* shared_x;   // [T][shared_k]
  const bf16_t* shared_w;   // [shared_n][shared_k], in the experts' form
  void* shared_out;         // gate/up: [T][shared_n / 2]; down: [T][N]
  float shared_limit;
  const float* factor;      // [T] a factor on the rows (gate/up: x; down: identity), or null
};

template <bool DOWN, bool TILED, int MT, int NT, int U>
__global__ __launch_bounds__(256) void moe_few_kernel(FewArgs a) {
  extern __shared__ float red[];      // [waves - 1][NT * MT][64 lanes][4], then the list
  const int wave = threadIdx.x / WAVE, nw = blockDim.x / WAVE, lane = threadIdx.x % WAVE, col = lane & 15, g = lane >> 4;
  const bool shared = (int)blockIdx.y < a.shared_y;
  const int n0 = (shared ? blockIdx.y * gridDim.x + blockIdx.x : blockIdx.x) * (16 * NT), n_items = a.T * a.top, y = blockIdx.y - a.shared_y;
  const int K = shared ? a.shared_k : a.K, N = shared ? a.shared_n : a.N, k_tiles = shared ? a.shared_k_tiles : a.k_tiles;
  int* list = (int*)(red + (size_t)(nw - 1) * NT * MT * WAVE * 4);      // (room for all items: a row may name an expert twice)
  // The expert's items in rising order.  Every wave finds all of them and writes the same list.
  int group = 0, count = 0;
  if (shared) {
    if (n0 >= N) return;
    count = a.T;
  } else {
    group = a.by_item ? a.ids[y] : y;
    int first = n_items;
    for (int i0 = 0; i0 < n_items; i0 += WAVE) {
      const int i = i0 + lane;
      const unsigned long long has = __ballot(i < n_items && a.ids[min(i, n_items - 1)] == group);
      if (has & (1ull << lane)) list[count + __popcll(has & ((1ull << lane) - 1))] = i;
      if (has && first == n_items) first = i0 + __ffsll(has) - 1;
      count += __popcll(has);
    }
    if (count == 0 || (a.by_item && first != y)) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
  if (!shared && group >= a.n_real) {             // an identity expert (the whole workgroup)
    if (DOWN)
      for (int i = threadIdx.x; i < count * 16 * NT; i += blockDim.x) {
        const int m = list[i / (16 * NT)], n = n0 + i % (16 * NT);
        if (n < a.N)
          ((float*)a.out)[((size_t)(m % a.top) * a.T + m / a.top) * a.N + n] = a.weights[m] * (a.factor ? a.factor[m / a.top] : 1.f) * (float)a.identity[(size_t)(m / a.top) * a.N + n];
      }
    return;
  }
  const bf16_t *w = shared ? a.shared_w : a.w, *x = shared ? a.shared_x : a.x;
  const bf16_t* wrow[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)      // (rows past N are read again, never stored)
    wrow[nt] = TILED ? w + ((size_t)(group * (N / 16) + min(n0 / 16 + nt, N / 16 - 1)) * k_tiles * WAVE + lane) * 8
                     : w + ((size_t)group * N + min(n0 + 16 * nt + col, N - 1)) * K;
  for (int start = 0; start < count; start += 16 * MT) {      // (more items than columns: the rows are streamed again, from the L2)
  int item[MT];
  const bf16_t* xrow[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int at = start + 16 * mt + col;
    item[mt] = at < count ? (shared ? at : list[at]) : -1;
    xrow[mt] = x + (size_t)(item[mt] < 0 ? 0 : shared ? item[mt] : item[mt] / a.x_div) * K;
  }
  floatx4 acc[NT][MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int nkb = (K + 63) / 64;
  for (int kb0 = wave * U; kb0 < nkb; kb0 += nw * U) {
    bf16x8 wv[U][NT][2], xv[U][MT][2];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        // plain rows: a lane's two pieces are 32 contiguous bytes, four lanes cover a line; tiles: a wave's piece is 1 KB of contiguous memory
        const int k = (kb0 + u) * 64 + 16 * g + 8 * h;
        const bool in = TILED ? kb0 + u < nkb : k < K;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const bf16x8* p = (const bf16x8*)(wrow[nt] + (TILED ? (size_t)(2 * (kb0 + u) + h) * WAVE * 8 : (size_t)k));
          wv[u][nt][h] = in ? (TILED ? __builtin_nontemporal_load(p) : *p) : zero8();
        }
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int k = TILED ? (kb0 + u) * 64 + 32 * h + 8 * g : (kb0 + u) * 64 + 16 * g + 8 * h;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) xv[u][mt][h] = (k < K && item[mt] >= 0) ? *(const bf16x8*)(xrow[mt] + k) : zero8();
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[u][nt][h], xv[u][mt][h], acc[nt][mt], 0, 0, 0);
  }
  if (nw > 1) {
    if (start > 0) __syncthreads();      // wave 0 is done with the last columns' sums
    if (wave > 0)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          *(floatx4*)(red + ((size_t)((wave - 1) * NT * MT + nt * MT + mt) * WAVE + lane) * 4) = acc[nt][mt];
    __syncthreads();
    if (wave > 0) continue;
    for (int v = 1; v < nw; ++v)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const floatx4 o = *(const floatx4*)(red + ((size_t)((v - 1) * NT * MT + nt * MT + mt) * WAVE + lane) * 4);
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[nt][mt][r] += o[r];
        }
  }
  // acc[nt][mt][r]: weight row n0 + 16 nt + 4 g + r of item column 16 mt + col
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = item[mt];
    if (m < 0) continue;
    if constexpr (!DOWN) {             // NT = 2: 16 rows of Wg and the same 16 of Wu
      const float wi = (a.weigh_input && !shared ? a.weights[m] : 1.f) * (a.factor ? a.factor[shared ? m : m / a.top] : 1.f), limit = shared ? a.shared_limit : a.limit;
      bf16x4 y;
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = (__bf16)gated_act(wi * acc[0][mt][r], wi * acc[1][mt][r], a.act, limit);
      *(bf16x4*)((bf16_t*)(shared ? a.shared_out : a.out) + (size_t)m * (N / 2) + n0 / 2 + 4 * g) = y;
    } else {
      const float wgt = a.weigh_input || shared ? 1.f : a.weights[m];
      float* o = shared ? (float*)a.shared_out + (size_t)m * N : (float*)a.out + ((size_t)(m % a.top) * a.T + m / a.top) * N;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int n = n0 + 16 * nt + 4 * g;
        if (n + 3 < N && N % 4 == 0) {
          *(floatx4*)(o + n) = floatx4{wgt * acc[nt][mt][0], wgt * acc[nt][mt][1], wgt * acc[nt][mt][2], wgt * acc[nt][mt][3]};
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n + r < N) o[n + r] = wgt * acc[nt][mt][r];
        }
      }
    }
  }
  }
}

template <bool DOWN, int MT, int NT, int U>
static int launch_few(FewArgs a, int n_groups, int waves, hipStream_t s) {
  const int columns = (a.N + 16 * NT - 1) / (16 * NT);
  if (a.shared_w) a.shared_y = ((a.shared_n + 16 * NT - 1) / (16 * NT) + columns - 1) / columns;
  const dim3 grid(columns, a.shared_y + (a.by_item ? a.T * a.top : n_groups));
  const size_t lds = (size_t)(waves - 1) * NT * MT * WAVE * 4 * sizeof(float) + (size_t)a.T * a.top * sizeof(int);
  if (a.k_tiles > 0) hipLaunchKernelGGL((moe_few_kernel<DOWN, true, MT, NT, U>), grid, dim3(waves * WAVE), lds, s, a);
  else hipLaunchKernelGGL((moe_few_kernel<DOWN, false, MT, NT, U>), grid, dim3(waves * WAVE), lds, s, a);
  IFX_LAUNCH_CHECK();
}

// Four waves to a workgroup (fewer where K is short): more workgroups on a compute unit, each finding its list and meeting in LDS
// while others stream, beat eight waves that take K in one round (mixtures of 64 rows: 180 against 246 us at 64 experts).
static int few_waves(int K) {
  int waves = 4;
  while (waves > 1 && (K + 63) / 64 < waves * 2) waves /= 2;
  return waves;
}

// E: the experts and the identity experts that ids name; T rows, at most MAX_ROWS.  shared_w (or null): a shared expert of
// shared_ff inner values, in the experts' form, its activations to shared_act [T][shared_ff].
extern "C" int ifx_moe_few_gate_up(const void* x, const void* w, void* act, const int* ids, int T, int E, int K, int ff, int top, int n_real,
                                   int act_kind, float limit, const float* in_weights, int tiled, const void* shared_w, void* shared_act,
                                   int shared_ff, float shared_limit, const float* factor, void* stream) {
  IFX_REQUIRE(K > 0 && K % 8 == 0 && ff > 0 && ff % 16 == 0, "moe_few_gate_up: K=%d must be a multiple of 8, ff=%d of 16", K, ff);
  IFX_REQUIRE(T > 0 && T <= MAX_ROWS && top > 0 && top <= MAX_TOP && E > 0 && E <= MAX_E, "moe_few_gate_up: %d rows (at most %d) of %d of %d experts", T, MAX_ROWS, top, E);
  IFX_REQUIRE(!shared_w || (shared_act && shared_ff > 0 && shared_ff % 16 == 0 && shared_ff <= 1 << 20), "moe_few_gate_up: a shared expert of %d (a multiple of 16)", shared_ff);
  const int k_tiles = tiled ? (K + 63) / 64 * 2 : 0;
  FewArgs a{(const bf16_t*)x, (const bf16_t*)w, act, ids, in_weights, nullptr, K, 2 * ff, top, T, top, n_real, act_kind,
            T * top < E ? 1 : 0, limit, in_weights ? 1 : 0, k_tiles, 0, K, 2 * shared_ff, k_tiles, (const bf16_t*)x, (const bf16_t*)shared_w, shared_act, shared_limit, factor};
  const int waves = few_waves(K);
  if (T <= 16) return launch_few<false, 1, 2, 3>(a, E, waves, (hipStream_t)stream);
  return launch_few<false, 2, 2, 2>(a, E, waves, (hipStream_t)stream);
}

// parts [top][T][N], and with a shared expert [top + 1][T][N], its output the last.
extern "C" int ifx_moe_few_down(const void* act, const void* w, float* parts, const float* weights, const int* ids, int T, int E, int N,
                                int ff, int top, int n_real, const void* identity, int weigh_input, int tiled, const void* shared_act,
                                const void* shared_w, int shared_ff, const float* factor, void* stream) {
  IFX_REQUIRE(ff > 0 && ff % 8 == 0 && N > 0 && (!tiled || N % 16 == 0), "moe_few_down: ff=%d must be a multiple of 8, N=%d of 16 if tiled", ff, N);
  IFX_REQUIRE(T > 0 && T <= MAX_ROWS && top > 0 && top <= MAX_TOP && E > 0 && E <= MAX_E, "moe_few_down: %d rows (at most %d) of %d of %d experts", T, MAX_ROWS, top, E);
  IFX_REQUIRE(!shared_w || (shared_act && shared_ff > 0 && shared_ff % 8 == 0 && shared_ff <= 1 << 20), "moe_few_down: a shared expert of %d (a multiple of 8)", shared_ff);
  FewArgs a{(const bf16_t*)act, (const bf16_t*)w, parts, ids, weights, (const bf16_t*)identity, ff, N, 1, T, top, n_real, 0,
            T * top < E ? 1 : 0, 0.f, weigh_input, tiled ? (ff + 63) / 64 * 2 : 0, 0, shared_ff, N, tiled ? (shared_ff + 63) / 64 * 2 : 0,
            (const bf16_t*)shared_act, (const bf16_t*)shared_w, parts + (size_t)top * T * N, 0.f, factor};
  const int waves = few_waves(shared_w && shared_ff > ff ? shared_ff : ff);
  hipStream_t s = (hipStream_t)stream;
  // (two row tiles to a wave halve its reads of the items; up to 64 items one is better: twice the workgroups)
  if (T <= 16) return T * top <= 64 ? launch_few<true, 1, 1, 2>(a, E, waves, s) : launch_few<true, 1, 2, 2>(a, E, waves, s);
  return T * top <= 64 ? launch_few<true, 2, 1, 2>(a, E, waves, s) : launch_few<true, 2, 2, 2>(a, E, waves, s);
}
