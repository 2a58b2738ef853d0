// The experts' products in 32 bits, on the 32-bit matrix instruction: every (row, choice) item takes the weights of the expert it chose.
//
//   gate_up   a[item][:] = act(Wg[e] x, Wu[e] x), both sums times the item's weight first where it is on the expert's input
//   down      parts[choice][row][:] = weight[item] * Wd[e] a[item] (1 * where it was on the input): the choices of a row are the slices of a sum
//             that its reader forms in order.  An id from n_real upwards names an identity expert, whose output is the row itself.
//
// An element's sum has one order, in both ways to it, so a row's results are the same bits in steps of one row and of thousands: four neighbouring
// k-values are one matrix instruction's, and the 64 of them in a block of 256 k-values are added up in pairs: neighbours, then pairs of
// neighbours (a step of 16), steps two apart, steps (a group of 64), groups, pairs of groups; the blocks are added in ascending order and places
// beyond K add zeros.  With the slices of gemm_f32.hip, chains of 64 products at 1,024 k-values, errors against 64 bits were 1.6 times
// those of a wave's 64 partial sums, which were there before (3.0e-7 of the result for 1.9e-7); like this they are 1.7e-7.
//
//   few    a wave takes four columns of an item (of gate and of up) by vector instructions: the matrix instruction adds its four products to the
//          sum one after the other, each rounded once, so fmaf() in its order gives the same bits.  (By matrix instructions, of whose 256
//          sums an item wants 16, 16 items of 1,024 x 1,408 took 57 us where these take 43.)  Every item streams its expert's weights: for steps of few rows, which rarely share
//          an expert.  Bound by the caches then (227 us for the 1.66 GB that 192 items of 704 ask for).
//   four   the same for up to four items of an expert at a time (ifx_moe_sort's tiles of four), whose weights are asked for once: for experts of one to
//          eight items, of which tiles of 64 would be empty for the most part.
//   tiles  items ordered by expert (ifx_moe_sort), 64 items by 64 weight rows through LDS as in gemm_f32_tiles_kernel; a wave's two tiles of
//          weight rows are gate's and up's of the same columns.
//
// Before, a wave of moe.hip formed the outputs of an item and the weights were read again for every row.  us of both products, that way : few : four : tiles (16
// experts 1,024 wide and 1,408 inner, two to a row) 1 row 15 : 12 : 21 : 93, 8 45 : 43 : 35 : 112, 32 132 : 151 : 79 : 145, 64 212 : 274 : 114 : 145, 128 351 : 555 : 180 : 149, 1,720
// 3,298 : - : - : 468 (93 TFLOP/s); 64 of 704, six to a row, 1 21 : 15 : 36 : 71, 8 68 : 67 : 75 : 133, 16 122 : 122 : 112 : 217, 32 199 : 227 : 146 : 240, 64 365 : 443 : 213 : 242, 1,720 6,354 :
// - : - : 744; 32 2,048 wide and 1,408 inner, four to a row, 4 90 : 94 : 100 : 246, 8 163 : 175 : 149 : 331, 64 859 : 1,217 : 425 : 460.
#include "common.h"
#include "f32_loads.h"

IFX_DEFINE_LAST_ERROR()

enum { MODE_GATE_UP = 0, MODE_DOWN = 1 };

struct ExpertsF32 {
  const float* x;            // MODE_GATE_UP: rows [T][K]; MODE_DOWN: activations [items][K] (few: by item; tiles: in the items' order)
  const float* w;            // MODE_GATE_UP: Wg [n_real][N][K]; MODE_DOWN: Wd [n_real][N][K]
  const float* up;           // MODE_GATE_UP: Wu
  float* out;                // MODE_GATE_UP: activations [items][N]; MODE_DOWN: [top][T][N]
  const int* ids;            // [items] (few)
  const float* weights;      // [items]
  const float* identity;     // MODE_DOWN: the rows [T][N]
  const int* sorted; const int* tile_expert; const int* tile_start; const int* tile_count; const int* n_tiles;      // (tiles)
  int T, top, K, N, n_real, act;
  float limit;
  int weigh_input;
  int items_first;           // (few) the grid's x runs over the items, not the columns
};

// ---- few items ------------------------------------------------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}

// Two rows' sums over a pair of lanes each, the first in the lane where `odd` is false: CTRL brings the other lane's.
template <int CTRL>
__device__ __forceinline__ float halve(float first, float second, bool odd) {
  return (odd ? second : first) + dpp<CTRL>(odd ? first : second);
}

// total[j] = x[j] . w[r] for R (4 or 8) rows of K values and the first `count` of ITEMS rows of x; lane l takes the k-values 4 l ... 4 l + 3 of a block of
// 256, AT_ONCE blocks asked for at a time, and is left with the sum of row (l & 3) + (l & 4): of 8 rows the lanes of bit 2 have the later four.
template <int R, bool VEC, int ITEMS>
__device__ __forceinline__ void dots(const float* const (&x)[ITEMS], int count, const float* const (&w)[R], int K, int lane, float (&total)[ITEMS]) {
  constexpr int AT_ONCE = R > 4 ? 2 : 4;
  const bool one = lane & 1, two = lane & 2, four = lane & 4;
  for (int k0 = 0; k0 < K; k0 += 256 * AT_ONCE) {
    f32x4 xv[AT_ONCE][ITEMS], wv[AT_ONCE][R];
    if (VEC && k0 + 256 * AT_ONCE <= K) {          // (no lane's place lies beyond K)
#pragma unroll
      for (int b = 0; b < AT_ONCE; ++b) {
        const int k = k0 + 256 * b + 4 * lane;
#pragma unroll
        for (int j = 0; j < ITEMS; ++j)
          if (j < count) xv[b][j] = *(const f32x4*)(x[j] + k);
#pragma unroll
        for (int r = 0; r < R; ++r) wv[b][r] = *(const f32x4*)(w[r] + k);
      }
    } else {
#pragma unroll
      for (int b = 0; b < AT_ONCE; ++b) {
        const int k = k0 + 256 * b + 4 * lane;
#pragma unroll
        for (int j = 0; j < ITEMS; ++j)
          if (j < count) xv[b][j] = load4<VEC>(x[j], k, K);
#pragma unroll
        for (int r = 0; r < R; ++r) wv[b][r] = load4<VEC>(w[r], k, K);
      }
    }
#pragma unroll
    for (int b = 0; b < AT_ONCE; ++b) {
      if (k0 + 256 * b >= K) break;
#pragma unroll
      for (int j = 0; j < ITEMS; ++j) {
        if (j >= count) break;
        float v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {          // (the matrix instruction adds its four products one after the other, each rounded once: so does this)
          v[r] = 0.f;
#pragma unroll
          for (int q = 0; q < 4; ++q) v[r] = fmaf(xv[b][j][q], wv[b][r][q], v[r]);
        }
        float u[R / 2], t[R / 4];
#pragma unroll
        for (int r = 0; r < R / 2; ++r) u[r] = halve<0xb1>(v[2 * r], v[2 * r + 1], one);             // lanes l and l ^ 1
#pragma unroll
        for (int r = 0; r < R / 4; ++r) {
          t[r] = halve<0x4e>(u[2 * r], u[2 * r + 1], two);                                          // ... ^ 2: steps of 16
          t[r] += dpp<0x128>(t[r]);                                                                 // ... ^ 8 (a rotation of a row of 16 by 8)
        }
        // ... ^ 4: by a rotation by 4, which is right where lanes 8 apart hold the same
        float g = R > 4 ? halve<0x124>(t[0], t[R / 4 - 1], four) : t[0] + dpp<0x124>(t[0]);        // groups of 64
        const auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(g), __float_as_uint(g), false, false);
        g = __uint_as_float(s16[0]) + __uint_as_float(s16[1]);
        const auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(g), __float_as_uint(g), false, false);
        g = __uint_as_float(s32[0]) + __uint_as_float(s32[1]);                                     // a block
        total[j] = k0 + b == 0 ? g : total[j] + g;
      }
    }
  }
}

#define COLUMNS 4          // of a wave
#define ITEMS_FIRST 12
#define TOGETHER 4         // items of one expert that a wave takes at a time
// ITEMS 1: the grid's items one by one.  TOGETHER: the lists' tiles of up to so many.
template <int MODE, bool VEC, int ITEMS>
__global__ __launch_bounds__(256) void experts_f32_few_kernel(ExpertsF32 a) {
  const int nth = a.items_first ? blockIdx.x : blockIdx.y, lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
  if (ITEMS > 1 && nth >= *a.n_tiles) return;
  const int n0 = ((a.items_first ? blockIdx.y : blockIdx.x) * 4 + wave) * COLUMNS, K = a.K;
  const int e = ITEMS > 1 ? a.tile_expert[nth] : a.ids[nth];
  if (n0 >= a.N || (MODE == MODE_GATE_UP && e >= a.n_real)) return;
  const int count = ITEMS > 1 ? min(a.tile_count[nth], ITEMS) : 1, start = ITEMS > 1 ? a.tile_start[nth] : 0;
  int item[ITEMS];
  float weight[ITEMS];
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    item[j] = ITEMS > 1 ? a.sorted[start + min(j, count - 1)] : nth;
    weight[j] = a.weights[item[j]];
  }
  const auto place = [&](int m) {        // of an item's row of results
    const int t = m / a.top;
    return a.out + (MODE == MODE_GATE_UP ? (size_t)m : (size_t)(m - t * a.top) * a.T + t) * a.N;
  };
  if (e >= a.n_real) {
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
      if (j < count && lane < COLUMNS && n0 + lane < a.N) place(item[j])[n0 + lane] = weight[j] * a.identity[(size_t)(item[j] / a.top) * a.N + n0 + lane];
    return;
  }
  constexpr int R = MODE == MODE_GATE_UP ? 2 * COLUMNS : COLUMNS;
  const float* rows[R];
  const float* x[ITEMS];
#pragma unroll
  for (int c = 0; c < COLUMNS; ++c) {
    const size_t at = ((size_t)e * a.N + min(n0 + c, a.N - 1)) * K;          // (columns beyond N are computed and dropped)
    rows[c] = a.w + at;
    if (MODE == MODE_GATE_UP) rows[R / 2 + c] = a.up + at;
  }
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) x[j] = a.x + (size_t)(MODE == MODE_GATE_UP ? item[j] / a.top : item[j]) * K;
  float v[ITEMS] = {};
  dots<R, VEC, ITEMS>(x, count, rows, K, lane, v);
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    if (j >= count) break;
    const float up = MODE == MODE_GATE_UP ? __shfl(v[j], lane ^ 4) : 0.f;
    if (lane >= COLUMNS || n0 + lane >= a.N) continue;
    if (MODE == MODE_GATE_UP) {
      const float wi = a.weigh_input ? weight[j] : 1.f;
      place(item[j])[n0 + lane] = gated_act(wi * v[j], wi * up, a.act, a.limit);
    } else {
      place(item[j])[n0 + lane] = (a.weigh_input ? 1.f : weight[j]) * v[j];
    }
  }
}

// ---- tiles ---------------------------------------------------------------------------------------------------------------
#define TILE_ITEMS 64

// MODE_GATE_UP: 32 columns a workgroup, of which wave w takes 16 (w % 2) ...: its first tile of weight rows is gate's, its second up's.
template <int MODE, bool VEC>
__global__ __launch_bounds__(256, 2) void experts_f32_tiles_kernel(ExpertsF32 a) {
  constexpr int BK = 32, COLS = MODE == MODE_GATE_UP ? 32 : 64;
  __shared__ f32x4 As[TILE_ITEMS][BK / 4], Ws[64][BK / 4];
  if ((int)blockIdx.y >= *a.n_tiles) return;
  const int e = a.tile_expert[blockIdx.y], start = a.tile_start[blockIdx.y], count = min(a.tile_count[blockIdx.y], TILE_ITEMS);
  const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE, i = lane % 16, q = lane / 16;
  const int n0 = blockIdx.x * COLS, K = a.K;
  const int* items = a.sorted + start;
  if (e >= a.n_real) {
    if (MODE == MODE_DOWN)
      for (int j = tid; j < count * COLS; j += 256) {
        const int m = items[j / COLS], t = m / a.top, n = n0 + j % COLS;
        if (n < a.N) a.out[((size_t)(m - t * a.top) * a.T + t) * a.N + n] = a.weights[m] * a.identity[(size_t)t * a.N + n];
      }
    return;
  }
  const int wm = wave / 2 * 32, wn = wave % 2 * 32;
  const int pr = tid / 8, pp = tid % 8;                    // the row (of 32) and the piece this thread brings in
  const float* arow[2];
  const float* wrow[2];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int m = 32 * r + pr;
    arow[r] = m >= count ? nullptr : a.x + (size_t)(MODE == MODE_GATE_UP ? items[m] / a.top : start + m) * K;
    // row m of the tile in LDS: 16 of gate, the same 16 of up, in turn
    const int n = MODE == MODE_GATE_UP ? n0 + m / 32 * 16 + m % 16 : n0 + m;
    wrow[r] = n >= a.N ? nullptr : (MODE == MODE_GATE_UP && m % 32 >= 16 ? a.up : a.w) + ((size_t)e * a.N + n) * K;
  }
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 total[2][2], na[2], nw[2];
  auto fetch = [&](int k0) {
    const int k = k0 + 4 * pp;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      na[r] = nw[r] = zero;
      if (arow[r]) na[r] = load4<VEC>(arow[r], k, K);
      if (wrow[r]) nw[r] = load4<VEC>(wrow[r], k, K);
    }
  };
  // the 32 k-values from k0 on: two steps' sums, alone or (ADD) added to those in `step`; the next 32 are asked for meanwhile
  auto stage = [&](int k0, f32x4 (&step)[2][2][2], bool ADD) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c) {          // (element c of this piece, the instruction pp % 4 of its step)
        ((float*)&As[32 * r + pr][(pp / 4 * 4 + c) ^ (pr % 8)])[pp % 4] = na[r][c];
        ((float*)&Ws[32 * r + pr][(pp / 4 * 4 + c) ^ (pr % 8)])[pp % 4] = nw[r][c];
      }
    __syncthreads();
    if (k0 + BK < K) fetch(k0 + BK);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4 x[2], w[2];
#pragma unroll
      for (int m = 0; m < 2; ++m) x[m] = As[wm + 16 * m + i][(4 * h + q) ^ (i % 8)];
#pragma unroll
      for (int n = 0; n < 2; ++n) w[n] = Ws[wn + 16 * n + i][(4 * h + q) ^ (i % 8)];
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          f32x4 c[4];
#pragma unroll
          for (int l = 0; l < 4; ++l) c[l] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[m][l], w[n][l], zero, 0, 0, 0);
          const f32x4 sum = (c[0] + c[1]) + (c[2] + c[3]);
          step[h][m][n] = ADD ? step[h][m][n] + sum : sum;
        }
    }
  };
  fetch(0);
  for (int kb = 0; kb < K; kb += 256) {
    f32x4 pairs[2][2][2];          // of the block's groups
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int k0 = kb + 64 * g;
      if (k0 < K) {
        f32x4 step[2][2][2];
        stage(k0, step, false);
        if (k0 + BK < K) stage(k0 + BK, step, true);
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int n = 0; n < 2; ++n) {
            const f32x4 sum = step[0][m][n] + step[1][m][n];
            pairs[g / 2][m][n] = g % 2 == 0 ? sum : pairs[g / 2][m][n] + sum;
          }
      } else if (g == 2) {
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int n = 0; n < 2; ++n) pairs[1][m][n] = zero;
      }
    }
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        const f32x4 block = pairs[0][m][n] + pairs[1][m][n];
        total[m][n] = kb == 0 ? block : total[m][n] + block;
      }
  }
  // lane (i, q) holds items 4 q + r of weight row i
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int at = wm + 16 * m + 4 * q + r;
      if (at >= count) continue;
      const int item = items[at], t = item / a.top;
      const float weight = a.weights[item];
      if (MODE == MODE_GATE_UP) {
        const int n = n0 + wave % 2 * 16 + i;
        const float wi = a.weigh_input ? weight : 1.f;
        if (n < a.N) a.out[(size_t)(start + at) * a.N + n] = gated_act(wi * total[m][0][r], wi * total[m][1][r], a.act, a.limit);
      } else {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const int n = n0 + wn + 16 * c + i;
          if (n < a.N) a.out[((size_t)(item - t * a.top) * a.T + t) * a.N + n] = (a.weigh_input ? 1.f : weight) * total[m][c][r];
        }
      }
    }
}

static bool check_act(int act, float limit) { return act == ACT_SILU || act == ACT_GELU_TANH || (act == ACT_CLAMPED_SWISH && limit > 0.f); }
static bool on16(const void* p) { return (uintptr_t)p % 16 == 0; }

// Both products.  act [items][ff] is scratch; parts [top][T][N].  sorted ... n_tiles: the lists of ifx_moe_sort with tiles of tile_items items, 64 for the matrix
// instruction's tiles or 4 for the vector instructions' that share their weights, or null: few items, each with its expert's weights for itself.
extern "C" int ifx_moe_f32(const float* h, const float* gate, const float* up, const float* down, const int* ids, const float* weights,
                           float* act, float* parts, const int* sorted, const int* tile_expert, const int* tile_start, const int* tile_count,
                           const int* n_tiles, int max_tiles, int tile_items, int T, int K, int ff, int N, int top, int n_real, int n_identity, int act_kind,
                           float limit, int weigh_input, void* stream) {
  IFX_REQUIRE(T >= 0 && K > 0 && ff > 0 && N > 0 && top > 0 && n_real > 0, "moe_f32: bad sizes T=%d K=%d ff=%d N=%d top=%d", T, K, ff, N, top);
  IFX_REQUIRE(check_act(act_kind, limit), "moe_f32: gated activation %d (limit %g)", act_kind, (double)limit);
  IFX_REQUIRE(n_identity == 0 || N == K, "moe_f32: identity experts hand back the row itself, so N=%d must equal K=%d", N, K);
  IFX_REQUIRE((sorted ? (long long)max_tiles : (long long)T * top) <= 65535, "moe_f32: %lld items or tiles are too many for one launch", sorted ? (long long)max_tiles : (long long)T * top);
  IFX_REQUIRE(sorted ? tile_items == TILE_ITEMS || tile_items == TOGETHER : tile_items == 1, "moe_f32: tiles of %d items", tile_items);
  if (T == 0) return 0;
  // (us with the items : the columns running fastest, 16 experts of 704: 4 items 11.9 : 14.1, 8 16.2 : 18.0, 16 27.9 : 24.6, 32 46 : 38, 64 84 : 65;
  // 64 experts: 12 21 : 24, 24 42 : 37.  With 1,000,000 columns the grid's second dimension is at its end.)
  const int items_first = !sorted && T * top <= ITEMS_FIRST && ff <= 1 << 20 && N <= 1 << 20;
  ExpertsF32 g{h, gate, up, act, ids, weights, nullptr, sorted, tile_expert, tile_start, tile_count, n_tiles, T, top, K, ff, n_real, act_kind, limit, weigh_input, items_first};
  ExpertsF32 d{act, down, nullptr, parts, ids, weights, h, sorted, tile_expert, tile_start, tile_count, n_tiles, T, top, ff, N, n_real, act_kind, limit, weigh_input, items_first};
  const bool vec_g = K % 4 == 0 && on16(h) && on16(gate) && on16(up), vec_d = ff % 4 == 0 && on16(act) && on16(down);
  hipStream_t s = (hipStream_t)stream;
#define GO(KERNEL, ARGS, COLS) \
  hipLaunchKernelGGL(KERNEL, items_first ? dim3(T * top, (ARGS.N + COLS - 1) / COLS) : dim3((ARGS.N + COLS - 1) / COLS, sorted ? max_tiles : T * top), dim3(256), 0, s, ARGS)
#define FEW(ITEMS) \
  if (vec_g) GO((experts_f32_few_kernel<MODE_GATE_UP, true, ITEMS>), g, 4 * COLUMNS); \
  else GO((experts_f32_few_kernel<MODE_GATE_UP, false, ITEMS>), g, 4 * COLUMNS); \
  if (vec_d) GO((experts_f32_few_kernel<MODE_DOWN, true, ITEMS>), d, 4 * COLUMNS); \
  else GO((experts_f32_few_kernel<MODE_DOWN, false, ITEMS>), d, 4 * COLUMNS)
  if (!sorted) {
    FEW(1);
  } else if (tile_items == TOGETHER) {
    FEW(TOGETHER);
  } else {
    if (vec_g) GO((experts_f32_tiles_kernel<MODE_GATE_UP, true>), g, 32);
    else GO((experts_f32_tiles_kernel<MODE_GATE_UP, false>), g, 32);
    if (vec_d) GO((experts_f32_tiles_kernel<MODE_DOWN, true>), d, 64);
    else GO((experts_f32_tiles_kernel<MODE_DOWN, false>), d, 64);
  }
#undef FEW
#undef GO
  IFX_LAUNCH_CHECK();
}
