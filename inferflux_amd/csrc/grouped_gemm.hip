// Products of many rows with one of several weights each, on the matrix cores (bfloat16 in, float sums): the experts of
// a mixture, where every (row, choice) takes the weight of the expert it chose, and the per-head products of attention
// through a latent, where every head has a weight of its own.
//
//   ifx_moe_sort       the (row, choice) items of a step ordered by expert, cut into tiles of TM items of one expert
//                      each; everything stays on the device (the grid of the products is sized by the most tiles
//                      there can be, and a workgroup without a tile leaves at once)
//   ifx_moe_gate_up_grouped   act[place] = silu(Wg[e] x) * (Wu[e] x) for the item at a place of that order, from weights whose
//                      rows alternate 16 of Wg with 16 of Wu, so that a lane holds a gate and its up and the activation is
//                      the epilogue; the second product then reads its tiles' rows one after the other
//   ifx_moe_down_grouped      parts[choice][row] = weight[item] * Wd[e] act[place] in float: the choices of a row are
//                      the "slices" of a sum that the kernel which adds the result to the stream takes in order, so a
//                      row's result does not depend on where its items lay in the order
//                      An expert from `n_real` upwards is an identity expert without weights: the first product leaves its
//                      tiles alone and the second writes weight[item] * x[row] (`identity`, the rows as the first product
//                      read them; N is then the rows' width).  The first product's activation is `act` of common.h.
//                      With in_weights / weigh_input the weight is on the expert's input: the first product multiplies its sums
//                      by it before the activation and the second leaves it out.
//   ifx_headwise_grouped      out[t][h][:N] = W[h] x[t][h], tiles of TM rows of one head; optionally times sigmoid of a column
//                      of a wider projected row, one per output element
//
// The experts' products stand on product_tiles.h and wave_tiles.h (which of them: grouped_wave_items in ops.py), an item's result whatever shares its tile.  The heads' product, whose
// matrices are small (K of a hundred), is heads_kernel below.
#include "common.h"
#include "column_gate.h"
#include "product_tiles.h"
#include "wave_tiles.h"
#include "tile_acts.h"

IFX_DEFINE_LAST_ERROR()

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;

#define TM 128         // items to a tile of the eight-wave kernel,
#define FEW_ITEMS 64   // where experts have few,
#define WAVE_ITEMS 192 // ... of the kernel by four large waves
#define EXPERTS_GROUP 4          // tiles of items that meet a tile of W one after the other
#define MAX_EXPERTS 1024


// ---------------------------------------------------------------------------------------
// ids [n_items] -> sorted [n_items] (items of expert 0, then of expert 1, ...), tiles (expert, first place in sorted,
// count) and their number.  One workgroup.  The order of an expert's items among themselves is not fixed; no result
// depends on it.  A wave adds the experts' counts up and cuts the tiles (one thread did), and
// a thread asks for eight ids at a time: 22,800 items took 33 us with a trip for each.
__global__ __launch_bounds__(1024) void moe_sort_kernel(const int* __restrict__ ids, int n_items, int E, int n_real, int tile_items,
                                                        int* __restrict__ sorted, int* __restrict__ tile_expert, int* __restrict__ tile_start,
                                                        int* __restrict__ tile_count, int* __restrict__ n_tiles) {
  constexpr int AT_ONCE = 8;          // ids that a thread asks for at a time: the launch is a chain of trips to memory
  __shared__ int cnt[MAX_EXPERTS];
  __shared__ int offs[MAX_EXPERTS];
  const int tid = threadIdx.x;
  for (int e = tid; e < E; e += 1024) cnt[e] = 0;
  __syncthreads();
  for (int i0 = tid; i0 < n_items; i0 += 1024 * AT_ONCE) {
    int id[AT_ONCE];
#pragma unroll
    for (int j = 0; j < AT_ONCE; ++j) id[j] = i0 + 1024 * j < n_items ? ids[i0 + 1024 * j] : -1;
#pragma unroll
    for (int j = 0; j < AT_ONCE; ++j)
      if (id[j] >= 0) atomicAdd(&cnt[id[j]], 1);
  }
  __syncthreads();
  if (tid < WAVE) {          // sums over the experts before, of items and of tiles, an expert to a lane
    int at = 0, n = 0;
    for (int e0 = 0; e0 < E; e0 += WAVE) {
      const int e = e0 + tid, c = e < E ? cnt[e] : 0, t = (c + tile_items - 1) / tile_items;
      int items = c, tiles = t;
#pragma unroll
      for (int d = 1; d < WAVE; d *= 2) {
        const int i = __shfl_up(items, d), u = __shfl_up(tiles, d);
        if (tid >= d) { items += i; tiles += u; }
      }
      if (e < E) {
        const int start = at + items - c, first = n + tiles - t;
        offs[e] = start;
        for (int k = 0; k < t; ++k) {
          tile_expert[first + k] = e;
          tile_start[first + k] = start + k * tile_items;
          tile_count[first + k] = min(tile_items, c - k * tile_items);
        }
        if (e == n_real - 1) n_tiles[1] = first + t;
      }
      at += __shfl(items, WAVE - 1);
      n += __shfl(tiles, WAVE - 1);
    }
    if (tid == 0) *n_tiles = n;
  }
  __syncthreads();
  for (int i0 = tid; i0 < n_items; i0 += 1024 * AT_ONCE) {
    int id[AT_ONCE];
#pragma unroll
    for (int j = 0; j < AT_ONCE; ++j) id[j] = i0 + 1024 * j < n_items ? ids[i0 + 1024 * j] : -1;
#pragma unroll
    for (int j = 0; j < AT_ONCE; ++j)
      if (id[j] >= 0) sorted[atomicAdd(&offs[id[j]], 1)] = i0 + 1024 * j;
  }
}

// n_tiles [2]: all tiles, and those of the n_real experts with weights, which come first
extern "C" int ifx_moe_sort(const int* ids, int n_items, int E, int n_real, int tile_items, int* sorted, int* tile_expert, int* tile_start,
                            int* tile_count, int* n_tiles, void* stream) {
  IFX_REQUIRE(n_items >= 0 && E > 0 && E <= MAX_EXPERTS, "moe_sort: %d items, %d experts (at most %d)", n_items, E, MAX_EXPERTS);
  IFX_REQUIRE(n_real > 0 && n_real <= E && tile_items >= 1, "moe_sort: %d of %d experts, %d items to a tile", n_real, E, tile_items);
  hipLaunchKernelGGL(moe_sort_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, ids, n_items, E, n_real, tile_items, sorted, tile_expert,
                     tile_start, tile_count, n_tiles);
  IFX_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------------------
enum { MODE_GATE_UP = 0, MODE_DOWN = 1 };

struct ExpertsArgs {
  const bf16_t* x;          // MODE_GATE_UP: rows [T][K], an item's is row item / top; MODE_DOWN: [n_items][K] in the items' order
  const bf16_t* w;          // [n_real][NW][K], or its tiled form (TILED; see ifx_tile_weights in gemm_bf16.hip, tiles of 16 rows)
  void* out;                // MODE_GATE_UP: [n_items][NW / 2] in the items' order; MODE_DOWN: [top][T][NW] float
  const int* sorted; const int* tile_expert; const int* tile_start; const int* tile_count; const int* n_tiles;
  const float* weights;     // [n_items]
  const bf16_t* identity;   // MODE_DOWN: [T][NW], what an identity expert hands back
  int T, top, K, NW;
  int n_real;               // experts with weights; tiles of later ones are identity experts'
  int act; float limit;     // MODE_GATE_UP: the activation
  int weigh_input;          // the weight is on an expert's input: MODE_GATE_UP multiplies both sums by it, MODE_DOWN leaves it out
};

// A workgroup takes the TM items of a tile by BN weight rows of its expert, eight waves of 32 weight rows by 64 items each and
// two workgroups to a CU: K is short (700 to 2,000), so that a tile's first loads and its epilogue are a fifth of its
// time, and want another tile's products beside them.  (256 weight rows to a workgroup, one to a CU, read a third less but
// took 718 us where these take 644; waves of 64 x 64 653; W from global memory into registers, in place of LDS, 624 to 714
// by the shape.)  22,800 items of 64 experts (2,048 wide, 1,408 inner, 356 items each): 532 + 328 us for the two products
// before, with the pieces through registers into LDS and rows of 64 k-values padded, now 362 + 241 (730 TFLOP/s with the tiles
// that are not full).  Experts of few items are bound by their weights' way from memory instead: tiles of 64 items, waves of
// 32 x 32, leave room for a third stage of loads on their way (64 experts of 6 to a row, 150 rows 215 -> 199 us for the whole mixture, 512 rows
// 234 -> 231; 32 experts, 4 to a row, 120 -> 106, 155 -> 145; 16 of 1,024 x 704, 2 to a row, 30 -> 23, 35 -> 27; with two stages 206, 108
// and 27 at 150 rows; tiles of 32 items in three or four 208, 116 and 23, but from 30 items to an expert on 1.1 times the tiles of 64 and more).
constexpr int TILE_BN = 128;
template <int MODE, bool TILED, int BM, int WM, int STAGES>
__global__ __launch_bounds__(512, 4) void experts_kernel(ExpertsArgs a) {
  typedef ProductTiles<TILE_BN, BM, 32, WM, TILED, STAGES> P;
  static_assert(P::THREADS == 512, "eight waves");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[P::LDS];
  const int tid = threadIdx.x;
  int tn, tm;
  if (!product_tile((a.NW + TILE_BN - 1) / TILE_BN, *a.n_tiles, 2, &tn, &tm)) return;
  const int e = a.tile_expert[tm], start = a.tile_start[tm], count = min(a.tile_count[tm], BM), n0 = tn * TILE_BN;
  const int* items = a.sorted + start;
  if (e >= a.n_real) {        // an identity expert's tile
    if (MODE == MODE_DOWN)
      for (int i = tid; i < count * TILE_BN; i += P::THREADS) {
        const int m = items[i / TILE_BN], n = n0 + i % TILE_BN;
        if (n < a.NW)
          ((float*)a.out)[((size_t)(m % a.top) * a.T + m / a.top) * a.NW + n] = a.weights[m] * (float)a.identity[(size_t)(m / a.top) * a.NW + n];
      }
    return;
  }
  const int rows = min(TILE_BN, a.NW - n0);
  const size_t row_values = TILED ? (size_t)((a.K + 63) / 64 * 64) : (size_t)a.K;
  const tile_uintx4 w = tile_buffer(a.w + ((size_t)e * a.NW + n0) * row_values, (unsigned)(rows * row_values) * 2u);
  const tile_uintx4 x = MODE == MODE_GATE_UP ? tile_buffer(a.x, (unsigned)a.T * (unsigned)a.K * 2u)
                                             : tile_buffer(a.x + (size_t)start * a.K, (unsigned)count * (unsigned)a.K * 2u);
  tile_floatx4 acc[P::FN][P::FM];
  P::run(lds, w, x, a.K, a.K, [&](int i) { return i >= count ? TILE_NO_ROW : (MODE == MODE_GATE_UP ? items[i] / a.top : i) * a.K * 2; }, acc);
  const int lane = tid % 64, g = lane / 16;
#pragma unroll
  for (int b = 0; b < P::FM; ++b) {
    const int i = P::wm() + 16 * b + lane % 16;
    if (i >= count) continue;
    const int m = items[i];
    if (MODE == MODE_GATE_UP) {
      // 16 weight rows of Wg, the same 16 of Wu in turn: acc[c][b] is the gate of what acc[c + 1][b] is the up of
      const int ff = a.NW / 2;
      bf16_t* act = (bf16_t*)a.out + (size_t)(start + i) * ff;
      const float wi = a.weigh_input ? a.weights[m] : 1.f;
#pragma unroll
      for (int c = 0; c < P::FN; c += 2) {
        const int f = (n0 + P::wn() + 16 * c) / 2 + 4 * g;
        if (f >= ff) continue;
        bf16x4 y;
#pragma unroll
        for (int r = 0; r < 4; ++r) y[r] = (__bf16)gated_act(wi * acc[c][b][r], wi * acc[c + 1][b][r], a.act, a.limit);
        *(bf16x4*)(act + f) = y;
      }
    } else {
      const float wgt = a.weigh_input ? 1.f : a.weights[m];
      float* out = (float*)a.out + ((size_t)(m % a.top) * a.T + m / a.top) * a.NW;
#pragma unroll
      for (int c = 0; c < P::FN; ++c) {
        const int n = n0 + P::wn() + 16 * c + 4 * g;
        if (a.NW % 4 == 0) {
          if (n < a.NW) *(floatx4*)(out + n) = floatx4{wgt * acc[c][b][0], wgt * acc[c][b][1], wgt * acc[c][b][2], wgt * acc[c][b][3]};
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n + r < a.NW) out[n + r] = wgt * acc[c][b][r];
        }
      }
    }
  }
}

// The same products by four large waves, one workgroup to a CU that takes one tile of 192 items by 256 weight rows after the other
// (wave_tiles.h; weights in tiles, whose lines are touched ahead by each workgroup for itself).  The next tile's place in the lists and its
// items are asked for before a tile's steps, its first steps before the results go out.  What is left of the matrix rate is the tiles that are
// not full and the last round of the chip: 20,400 items of 32 experts (2,048 wide, 1,408 inner) both products and the order of the items
// 537 -> 477 us (740 TFLOP/s), 65,536 items 1,414 -> 1,219 (930).  Tiles of 128 items (three slots) were
// 1.0 to 1.2 x the eight waves' time; with tiles of 256 the sums, the fragments and the rows' addresses fill the registers, and the compiler
// moves sums about between the products in assembly, whose results it does not wait for: wrong sums.  A test looks for
// such moves (a sum read within 14 wait states of the product that writes it) in the built kernels, along every path.
template <int MODE, int FN, int FM>
struct ExpertWaves {
  typedef WaveTiles<FN, FM, true> P;
  static constexpr int PITCH = 16 * FN + 16, WAVE_BYTES = MODE == MODE_GATE_UP ? 16 * PITCH : 0, LDS = P::LDS + 4 * WAVE_BYTES;
};

// 16 rows of a wave's activations at a time, turned in LDS so that they go out in whole lines; stores beyond the rows and columns are dropped
template <int FN, int FM, int ACT>
__device__ __forceinline__ void waves_gate_up_out(const WaveTiles<FN, FM, true>& p, const ExpertsArgs& a, unsigned char* lds, tile_floatx4 (&acc)[FN][FM],
                                                  const float (&weight)[FM], int start, int count, int n0) {
  typedef ExpertWaves<MODE_GATE_UP, FN, FM> O;
  const int ff = a.NW / 2, m = p.wm(), rows = count - m, first = (n0 + p.wn()) / 2;
  const unsigned long long at0 = (unsigned long long)a.out + (size_t)(start + m) * ff * 2;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)at0), hi = __builtin_amdgcn_readfirstlane((unsigned)(at0 >> 32));
  const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc((void*)((unsigned long long)hi << 32 | lo), 0,
                                                                        __builtin_amdgcn_readfirstlane(max(0, min(16 * FM, rows)) * ff * 2), 0x00020000);
  unsigned char* st = lds + WaveTiles<FN, FM, true>::LDS + p.wid * O::WAVE_BYTES;
#pragma unroll
  for (int b = 0; b < FM; ++b) {
    const float w = weight[b];
#pragma unroll
    for (int c = 0; c < FN; c += 2) {
      asm volatile("" : "+a"(acc[c][b]), "+a"(acc[c + 1][b]));          // (not before: the registers beside the sums are taken)
      const tile_floatx4 gt = acc[c][b], up = acc[c + 1][b];
      bf16x4 y;
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = (__bf16)tile_gated<ACT>(w * gt[r], w * up[r], a.limit);
      *(bf16x4*)(st + p.col * O::PITCH + c * 16 + p.g * 8) = y;
    }
    constexpr int PIECES = FN;          // of 16 bytes to a row
#pragma unroll
    for (int j0 = 0; j0 < 16 * PIECES; j0 += 64) {
      const int j = j0 + p.lane, r = j / PIECES, at = 8 * (j % PIECES);
      const bool in = r < rows - 16 * b && first + at < ff;
      const tile_uintx4 v = *(const tile_uintx4*)(st + r * O::PITCH + 2 * at);
      __builtin_amdgcn_raw_buffer_store_b128(v, out, in ? ((16 * b + r) * ff + first + at) * 2 : TILE_NO_ROW, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <int MODE, int FN, int FM>
__global__ __launch_bounds__(256, 1) void experts_waves_kernel(ExpertsArgs a) {
  typedef ExpertWaves<MODE, FN, FM> O;
  typedef typename O::P P;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[O::LDS];
  static_assert(O::LDS <= 160 * 1024 && FN % 4 == 0, "LDS");
  const int nt = (a.NW + P::BN - 1) / P::BN, mt = a.n_tiles[1], total = nt * mt;
  if (MODE == MODE_DOWN) {          // identity experts' items, a wave to an item (NW is the rows' width then, a multiple of 8)
    const int places = (a.n_tiles[0] - mt) * WAVE_ITEMS;
    for (int p = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + threadIdx.x / 64); p < places; p += gridDim.x * 4) {
      const int tm = mt + p / WAVE_ITEMS, i = p % WAVE_ITEMS;
      if (i >= a.tile_count[tm]) continue;
      const int m = a.sorted[a.tile_start[tm] + i], t = m / a.top;
      const float w = a.weights[m];
      const bf16_t* x = a.identity + (size_t)t * a.NW;
      float* out = (float*)a.out + ((size_t)(m - t * a.top) * a.T + t) * a.NW;
      for (int n = threadIdx.x % 64 * 8; n < a.NW; n += 512) {
        const bf16x8 v = *(const bf16x8*)(x + n);
        *(floatx4*)(out + n) = floatx4{w * (float)v[0], w * (float)v[1], w * (float)v[2], w * (float)v[3]};
        *(floatx4*)(out + n + 4) = floatx4{w * (float)v[4], w * (float)v[5], w * (float)v[6], w * (float)v[7]};
      }
    }
  }
  const int per = (total + 7) / 8, end = min(total, (int)(blockIdx.x % 8 + 1) * per), stride = gridDim.x / 8;
  int id = blockIdx.x % 8 * per + blockIdx.x / 8;
  if (id >= end) return;
  const size_t row_values = (size_t)((a.K + 63) / 64 * 64);
  P p;
  p.init(lds);
  int e, start, count, n0, rows[FM];          // the tile, and where this lane's rows of x start
  auto scalar = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  auto find = [&](int t) {          // groups of EXPERTS_GROUP tiles of x by all of W's
    const int turn = scalar(t / (EXPERTS_GROUP * nt)), in = t - turn * EXPERTS_GROUP * nt, gm = min(EXPERTS_GROUP, mt - turn * EXPERTS_GROUP);
    const int tn = scalar(in / gm), tm = turn * EXPERTS_GROUP + in - tn * gm;
    e = scalar(a.tile_expert[tm]), start = scalar(a.tile_start[tm]), count = scalar(a.tile_count[tm]), n0 = tn * P::BN;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int row = (p.wid * FM + i) * 8 + p.lane / 8;
      rows[i] = row >= count ? -1 : MODE == MODE_GATE_UP ? a.sorted[start + row] : row;
    }
  };
  auto rows_of_w = [&]() {
    return tile_buffer(a.w + ((size_t)e * a.NW + n0) * row_values, (unsigned)(min(P::BN, a.NW - n0) * row_values) * 2u);
  };
  auto begin = [&]() {
    const tile_uintx4 x = MODE == MODE_GATE_UP ? tile_buffer(a.x, (unsigned)a.T * (unsigned)a.K * 2u)
                                               : tile_buffer(a.x + (size_t)start * a.K, (unsigned)count * (unsigned)a.K * 2u);
    p.begin(rows_of_w(), x, a.K, 0, [&](int, int i) { return rows[i] < 0 ? TILE_NO_ROW : (MODE == MODE_GATE_UP ? rows[i] / a.top : rows[i]) * a.K * 2; });
    p.touch_tiles(a.K);
  };
  find(id);
  begin();
  while (true) {
    const int this_start = start, this_count = count, this_n0 = n0;
    int item[FM];
    float weight[FM];
#pragma unroll
    for (int b = 0; b < FM; ++b) {
      const int i = p.wm() + 16 * b + p.col;
      item[b] = i < count && (MODE == MODE_DOWN || a.weigh_input) ? a.sorted[start + i] : -1;
    }
#pragma unroll
    for (int b = 0; b < FM; ++b) weight[b] = item[b] >= 0 && (MODE == MODE_GATE_UP || !a.weigh_input) ? a.weights[item[b]] : 1.f;
    id += stride;
    const bool more = id < end;
    if (more) find(id);
    p.next = rows_of_w(), p.next_steps = more ? (a.K + 63) / 64 : 0;
    if (!more) p.next[2] = 0;          // (nothing to touch)
    tile_floatx4 acc[FN][FM];
    p.run(lds, a.K, acc);
    if (more) begin();
    if constexpr (MODE == MODE_GATE_UP) {
      switch (a.act) {
        case ACT_GELU_TANH: waves_gate_up_out<FN, FM, ACT_GELU_TANH>(p, a, lds, acc, weight, this_start, this_count, this_n0); break;
        case ACT_SILU: waves_gate_up_out<FN, FM, ACT_SILU>(p, a, lds, acc, weight, this_start, this_count, this_n0); break;
        default: waves_gate_up_out<FN, FM, ACT_CLAMPED_SWISH>(p, a, lds, acc, weight, this_start, this_count, this_n0); break;
      }
    } else {
#pragma unroll
      for (int b = 0; b < FM; ++b) {
        const int t = item[b] / a.top;
        float* out = (float*)a.out + ((size_t)(item[b] - t * a.top) * a.T + t) * a.NW;
#pragma unroll
        for (int c = 0; c < FN; ++c) {
          asm volatile("" : "+a"(acc[c][b]));
          const int n = this_n0 + p.wn() + 16 * c + 4 * p.g;
          const tile_floatx4 v = acc[c][b];
          if (item[b] >= 0 && n < a.NW) *(floatx4*)(out + n) = floatx4{weight[b] * v[0], weight[b] * v[1], weight[b] * v[2], weight[b] * v[3]};
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (!more) break;
  }
}

template <int MODE>
static void launch_experts(const ExpertsArgs& a, int max_tiles, int tiled, int items, hipStream_t s) {
  const dim3 blocks((max_tiles * ((a.NW + TILE_BN - 1) / TILE_BN) + 7) / 8 * 8), threads(512);
  if (items == FEW_ITEMS) hipLaunchKernelGGL((experts_kernel<MODE, true, FEW_ITEMS, 32, 3>), blocks, threads, 0, s, a);
  else if (tiled) hipLaunchKernelGGL((experts_kernel<MODE, true, TM, 64, 2>), blocks, threads, 0, s, a);
  else hipLaunchKernelGGL((experts_kernel<MODE, false, TM, 64, 2>), blocks, threads, 0, s, a);
}

template <int MODE>
static void launch_experts_waves(const ExpertsArgs& a, int max_tiles, hipStream_t s) {
  const long long most = (long long)max_tiles * ((a.NW + 255) / 256);
  const dim3 blocks(most < 256 ? (int)(most + 7) / 8 * 8 : 256);
  hipLaunchKernelGGL((experts_waves_kernel<MODE, 8, WAVE_ITEMS / 32>), blocks, dim3(256), 0, s, a);
}

// ---------------------------------------------------------------------------------------
struct HeadsArgs {
  const bf16_t* x;          // row t of head h reads K values from x + t * x_row + h * x_head
  const bf16_t* w;          // [heads][N][K]
  bf16_t* out;              // [T][heads][out_head]
  int T, n_heads, K, N, x_row, x_head, out_head;
  ColumnGate gate;          // columns col + head * N + n of row t (rows null: none)
};

#define TN 128
#define TK 64
#define LDP (TK + 8)
// A workgroup of four waves takes 64 MT rows of a head and TN = 128 weight rows; steps of 64 k-values of both are staged in
// LDS (16-byte pieces, rows padded by 16 bytes against bank conflicts, the next step's pieces on their way into registers
// meanwhile).  The waves stand two by two: each multiplies 32 x MT rows with two tiles of 32 weight rows on the 32x32x16
// matrix instruction, C[weight row][row], so a lane ends up with runs of four consecutive output columns of one row.
template <int MT>
__global__ __launch_bounds__(256, 2) void heads_kernel(HeadsArgs a) {
  constexpr int BM = 64 * MT;
  __shared__ __attribute__((aligned(16))) bf16_t ws[TN][LDP];
  __shared__ __attribute__((aligned(16))) bf16_t xs[BM][LDP];
  const int tid = threadIdx.x;
  const int per = (a.T + BM - 1) / BM, head = blockIdx.x / per, start = (blockIdx.x % per) * BM, count = min(BM, a.T - start);
  const int n0 = blockIdx.y * TN;
  const int wave = tid / WAVE, lane = tid % WAVE, l32 = lane & 31, hi = lane >> 5;
  const int wm = wave & 1, wn = wave >> 1;          // this wave's rows: 32 MT wm ..., its weight rows: 64 wn ...
  floatx16 acc[MT][2];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mt][nt][i] = 0.f;
  const bf16_t* wbase = a.w + (size_t)head * a.N * a.K;
  const bf16_t* xbase = a.x + (size_t)head * a.x_head;
  bf16x8 zero;
#pragma unroll
  for (int i = 0; i < 8; ++i) zero[i] = (__bf16)0.f;
  // A step's pieces are asked for one step ahead: while the matrix cores work on step s from LDS, the loads of step
  // s + 1 are on their way into registers.  Pieces of 8 k-values: 8 to a row; TN rows of W and BM rows of x.
  constexpr int WP = TN * 8 / 256, XP = BM * 8 / 256;
  bf16x8 wv[WP], xv[XP];
  const bf16_t* wp[WP];
  const bf16_t* xp[XP];
  const int kc = 8 * (tid % 8);
#pragma unroll
  for (int p = 0; p < WP; ++p) {
    const int wrow = n0 + (tid + 256 * p) / 8;
    wp[p] = wrow < a.N ? wbase + (size_t)wrow * a.K + kc : nullptr;
  }
#pragma unroll
  for (int p = 0; p < XP; ++p) {
    const int i = (tid + 256 * p) / 8;
    xp[p] = i < count ? xbase + (size_t)(start + i) * a.x_row + kc : nullptr;
  }
  auto fetch = [&](int k0) {
    const bool in = k0 + kc < a.K;
#pragma unroll
    for (int p = 0; p < WP; ++p) wv[p] = (wp[p] && in) ? *(const bf16x8*)(wp[p] + k0) : zero;
#pragma unroll
    for (int p = 0; p < XP; ++p) xv[p] = (xp[p] && in) ? *(const bf16x8*)(xp[p] + k0) : zero;
  };
  fetch(0);
  for (int k0 = 0; k0 < a.K; k0 += TK) {
    __syncthreads();          // everyone is done with the last step's tiles
#pragma unroll
    for (int p = 0; p < WP; ++p) *(bf16x8*)&ws[(tid + 256 * p) / 8][kc] = wv[p];
#pragma unroll
    for (int p = 0; p < XP; ++p) *(bf16x8*)&xs[(tid + 256 * p) / 8][kc] = xv[p];
    __syncthreads();
    if (k0 + TK < a.K) fetch(k0 + TK);
#pragma unroll
    for (int ks = 0; ks < TK / 16; ++ks) {
      bf16x8 aop[2], bop[MT];
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) aop[nt] = *(const bf16x8*)&ws[64 * wn + 32 * nt + l32][16 * ks + 8 * hi];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) bop[mt] = *(const bf16x8*)&xs[32 * MT * wm + 32 * mt + l32][16 * ks + 8 * hi];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(aop[nt], bop[mt], acc[mt][nt], 0, 0, 0);
    }
  }
  // acc[mt][nt][i]: weight row n0 + 64 wn + 32 nt + 8 (i / 4) + 4 hi + i % 4 of row 32 MT wm + 32 mt + l32
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int i0 = 32 * MT * wm + 32 * mt + l32, m = start + i0;
    if (i0 >= count) continue;
    bf16_t* ob = a.out + ((size_t)m * a.n_heads + head) * a.out_head;
    if (a.gate.rows && a.N % 4 == 0 && a.gate.in_fours()) {
      int c[8];             // (columns beyond the head's read its last four again; nothing of them is stored)
      float f[8][4];
#pragma unroll
      for (int i = 0; i < 8; ++i) c[i] = head * a.N + min(n0 + 64 * wn + 32 * (i / 4) + 8 * (i % 4) + 4 * hi, a.N - 4);
      a.gate.at4<bf16_t>(m, c, f);
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[mt][i / 4][4 * (i % 4) + r] *= f[i][r];
    } else if (a.gate.rows) {
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int n = n0 + 64 * wn + 32 * nt + 8 * (i / 4) + 4 * hi + i % 4;
          if (n < a.N) acc[mt][nt][i] *= a.gate.at<bf16_t>(m, head * a.N + n);
        }
    }
    const bool whole4 = a.N % 4 == 0 && a.out_head % 4 == 0;      // runs of four columns, stored at once
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = n0 + 64 * wn + 32 * nt + 8 * q + 4 * hi;
        if (n >= a.N) continue;
        if (whole4) {
          bf16x4 y;
#pragma unroll
          for (int r = 0; r < 4; ++r) y[r] = (__bf16)acc[mt][nt][4 * q + r];
          *(bf16x4*)(ob + n) = y;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n + r < a.N) ob[n + r] = (bf16_t)acc[mt][nt][4 * q + r];
        }
      }
  }
}

// act [n_items][ff] (bfloat16, in the items' order) from x [T][K] and the paired weights w [n_real][2 ff][K]; item i is row i / top.
extern "C" int ifx_moe_gate_up_grouped(const void* x, const void* w, void* act, const int* sorted, const int* tile_expert,
                                       const int* tile_start, const int* tile_count, const int* n_tiles, int max_tiles,
                                       int T, int K, int ff, int top, int n_real, int act_kind, float limit, const float* in_weights,
                                       int tiled, int wave_items, void* stream) {
  IFX_REQUIRE(K > 0 && K % 8 == 0 && ff > 0 && ff % 16 == 0 && top > 0 && T >= 0, "moe_gate_up_grouped: K=%d must be a multiple of 8, ff=%d of 16", K, ff);
  IFX_REQUIRE((long long)T * K < (1ll << 30) - 4096, "moe_gate_up_grouped: %d rows of %d values are 2 GB or more", T, K);
  if (max_tiles <= 0 || T == 0) return 0;
  const ExpertsArgs a{(const bf16_t*)x, (const bf16_t*)w, act, sorted, tile_expert, tile_start, tile_count, n_tiles, in_weights,
                      nullptr, T, top, K, 2 * ff, n_real, act_kind, limit, in_weights ? 1 : 0};
  IFX_REQUIRE(wave_items == 0 || (tiled && (wave_items == WAVE_ITEMS || wave_items == FEW_ITEMS)), "moe_gate_up_grouped: tiles of %d items", wave_items);
  if (wave_items == WAVE_ITEMS) launch_experts_waves<MODE_GATE_UP>(a, max_tiles, (hipStream_t)stream);
  else launch_experts<MODE_GATE_UP>(a, max_tiles, tiled, wave_items, (hipStream_t)stream);
  IFX_LAUNCH_CHECK();
}

// parts [top][T][N] (float) = weights[item] * (Wd[e] act[place]), w [n_real][N][ff]
extern "C" int ifx_moe_down_grouped(const void* act, const void* w, float* parts, const float* weights, const int* sorted,
                                    const int* tile_expert, const int* tile_start, const int* tile_count, const int* n_tiles,
                                    int max_tiles, int T, int N, int ff, int top, int n_real, const void* identity,
                                    int weigh_input, int tiled, int wave_items, void* stream) {
  IFX_REQUIRE(!tiled || N % 16 == 0, "moe_down_grouped: tiled weights need N=%d to be a multiple of 16", N);
  IFX_REQUIRE(ff > 0 && ff % 8 == 0 && N > 0 && top > 0 && T >= 0, "moe_down_grouped: ff=%d must be a multiple of 8", ff);
  if (max_tiles <= 0 || T == 0) return 0;
  const ExpertsArgs a{(const bf16_t*)act, (const bf16_t*)w, parts, sorted, tile_expert, tile_start, tile_count, n_tiles, weights,
                      (const bf16_t*)identity, T, top, ff, N, n_real, 0, 0.f, weigh_input};
  IFX_REQUIRE(wave_items == 0 || (tiled && (wave_items == WAVE_ITEMS || wave_items == FEW_ITEMS)), "moe_down_grouped: tiles of %d items", wave_items);
  if (wave_items == WAVE_ITEMS) launch_experts_waves<MODE_DOWN>(a, max_tiles, (hipStream_t)stream);
  else launch_experts<MODE_DOWN>(a, max_tiles, tiled, wave_items, (hipStream_t)stream);
  IFX_LAUNCH_CHECK();
}

// out [T][H][out_head] (bfloat16): the first N elements of every head, W [H][N][K], head h of row t reads x + t * x_row + h * x_head
extern "C" int ifx_headwise_grouped(const void* x, const void* w, void* out, int T, int H, int K, int N, int x_row, int x_head,
                                    int out_head, const void* gate, int gate_ld, int gate_col, int gate_slices, long long gate_stride,
                                    void* stream) {
  IFX_REQUIRE(!gate || (gate_col >= 0 && gate_col + H * N <= gate_ld && gate_slices >= 0), "headwise_grouped: %d gates from column %d on do not fit rows of %d", H * N, gate_col, gate_ld);
  IFX_REQUIRE(K > 0 && K % 8 == 0 && x_row % 8 == 0 && x_head % 8 == 0 && N > 0 && H > 0 && out_head >= N, "headwise_grouped: K=%d, the rows of x (%d) and its heads (%d) must be multiples of 8", K, x_row, x_head);
  if (T <= 0) return 0;
  const HeadsArgs a{(const bf16_t*)x, (const bf16_t*)w, (bf16_t*)out, T, H, K, N, x_row, x_head, out_head,
                    ColumnGate{gate, gate_ld, gate_col, gate_slices, (size_t)gate_stride}};
  if (T > 64) hipLaunchKernelGGL((heads_kernel<2>), dim3(((T + 127) / 128) * H, (N + TN - 1) / TN), dim3(256), 0, (hipStream_t)stream, a);
  else hipLaunchKernelGGL((heads_kernel<1>), dim3(((T + 63) / 64) * H, (N + TN - 1) / TN), dim3(256), 0, (hipStream_t)stream, a);
  IFX_LAUNCH_CHECK();
}
