// Attention of prompts in 32 bits on the matrix cores: tiles of consecutive rows of a request over the paged cache, every
// score and every weighted value by v_mfma_f32_16x16x4_f32, whose four multiply-adds run one after the other in ascending
// order.  The operations and their order are those of the plain kernel (attn_plain.hip), so a row has the same bits by
// either: a score is the ascending sum over the key's elements times the scale; a tile of 64 keys gives its maximum, its
// weights' sum (halves of the tile first, neighbours last) and the ascending sum of its weighted values; every fourth tile is
// a part, and the parts are joined in order.  Formulas, limits and parameters stand there.
//
// A workgroup has 64 columns, (row, query head) pairs of a kv head's group counted row by row, 16 to a wave, and walks the
// keys that any of them sees in tiles of 64, staged once in LDS for all of its waves while the next tile is on its way to
// registers.  Scores are computed transposed, keys by columns, with the keys of a block of 16 in the order that leaves each
// weight in the lane and register where the product with the values wants it: nothing is exchanged between the two products,
// and a column's maximum and sum need two exchanges each.
//
// Few workgroups with long walks are four each, a part to a workgroup, and a second launch joins the parts; so do two maps,
// which are workgroups of their own over the same values.
//
// What bounds it: the matrix instruction (2,048 operations in 32 cycles: 157 TFLOP/s), beside it the exponentials (half as
// long) and the walk of the longest tile.  us by the plain kernel / here: two prompts of 2,000 rows, 14 heads of 64 on two 2,470 /
// 208 (70 TFLOP/s), 8 heads of 128 on two 2,770 / 246, two maps of 64 with values of 128 2,850 / 380; eight of 500 658 / 69, 727 / 96,
// 768 / 143; 512 rows behind 1,500 keys 561 / 65, 614 / 104, 717 / 90.
#include "common.h"

IFX_DEFINE_LAST_ERROR()

#define TILE_KEYS 64
#define PARTS 4
#define COLS 16                   // columns of a wave
#define PAD 4                     // floats between rows in LDS: 16 rows then lie on different banks

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f4;

struct F32Args {
  const float* q;
  const float* k_cache;
  const float* v_cache;
  float* out;
  const int* tiles;               // [n_tiles][2]: request, first column
  const int* q_start;
  const int* q_len;
  const int* kv_len;
  const int* block_table;
  int max_blocks, nH, nKV, page_size, window, maps;
  float scale;
  int keep_first, has_sink;
  float sink_score;
  const float* gate;
  const float* sinks;
  int chunk;
  float lambda, out_scale, norm_eps;
  float* part_o;                  // [row][head][map][PARTS or 1][dv] and, maximum and sum, [2]; null: the launch's results go to out
  float* part_ml;
  int n_tiles;
};

// what a column's position sees: keys [0, keep) and [lo, pos]
__device__ __forceinline__ int first_key(const F32Args& a, int pos) {
  int lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  if (a.chunk > 0) lo = max(lo, pos - pos % a.chunk);
  return lo;
}

// Keys of DK elements (one of ``maps`` vectors of a row, a workgroup each), values of DV.  SPLIT: a workgroup for each part.
template <int DK, int DV, int WAVES, bool SPLIT>
__global__ __launch_bounds__(WAVE * WAVES, 2) void attn_f32_kernel(F32Args a) {
#pragma clang fp contract(off)
  constexpr int KS = DK + PAD, VS = TILE_KEYS + PAD, THREADS = WAVE * WAVES, VC = DV / 16;
  constexpr int K_LOADS = TILE_KEYS * DK / 4 / THREADS, V_LOADS = TILE_KEYS * DV / 4 / THREADS;
  constexpr bool ALL_IN_LDS = !SPLIT && DV > 64;        // (128 elements: registers for the joined parts are not left)
  static_assert(TILE_KEYS * DK / 4 % THREADS == 0 && TILE_KEYS * DV / 4 % THREADS == 0, "whole rounds of loads");
  __shared__ __attribute__((aligned(16))) float k_s[TILE_KEYS * KS];
  __shared__ __attribute__((aligned(16))) float v_s[DV * VS];
  __shared__ f4 all_s[ALL_IN_LDS ? VC * THREADS : 1];
  __shared__ int odd_value;       // a staged tile that some columns see in part holds values that are not finite
  const int wid = threadIdx.x / WAVE, lane = threadIdx.x % WAVE, i16 = lane % 16, grp = lane / 16;
  const int G = a.nH / a.nKV, P = a.page_size, KD = a.maps * DK;
  // a tile's kv heads, maps and parts follow one another
  int item = blockIdx.x;
  const int only = SPLIT ? item % PARTS : 0;
  if (SPLIT) item /= PARTS;
  const int map = item % a.maps, kvh = item / a.maps % a.nKV, tile = item / a.maps / a.nKV;
  const int req = a.tiles[2 * tile], c0 = a.tiles[2 * tile + 1];
  const int q_len = a.q_len[req], row0 = a.q_start[req], past = a.kv_len[req] - q_len, cols = q_len * G;
  const int* table = a.block_table + (size_t)req * a.max_blocks;
  const int col = c0 + wid * COLS + i16;
  const bool real = col < cols;
  const int row = real ? col / G : 0, head = kvh * G + (real ? col % G : 0);
  const int pos = real ? past + row : -1;
  const int lo = real ? first_key(a, pos) : 0, keep = lo > 0 ? min(a.keep_first, lo) : 0;
  const int t_first = keep > 0 ? 0 : lo / TILE_KEYS * TILE_KEYS;
  // ... and what the workgroup's columns see between them (lo only grows with the position)
  const int pos_lo = past + c0 / G, pos_hi = past + min(c0 + WAVES * COLS - 1, cols - 1) / G;
  const int lo_min = first_key(a, pos_lo), lo_max = first_key(a, pos_hi), keep_max = lo_max > 0 ? min(a.keep_first, lo_max) : 0;
  const int last_tile = pos_hi / TILE_KEYS, lo_tile = lo_min / TILE_KEYS, kept_tiles = min((keep_max + TILE_KEYS - 1) / TILE_KEYS, lo_tile);
  const bool has_sink = a.has_sink || a.sinks;
  const float sink_score = a.sinks ? a.sinks[head] : a.sink_score;

  // query elements 4 s + grp of column i16, the matrix instruction's second operand (a column that is not there has the first
  // row's, and sees nothing)
  float q[DK / 4];
  {
    const float* qrow = a.q + ((size_t)(row0 + row) * a.nH + head) * KD + map * DK + grp;
#pragma unroll
    for (int s = 0; s < DK / 4; ++s) q[s] = qrow[4 * s];
  }

  // the first tile at or behind t of t's part that is not between the kept first keys and the window
  auto at_or_after = [&](int t) { return t >= kept_tiles && t < lo_tile ? t + (lo_tile - t + PARTS - 1) / PARTS * PARTS : t; };
  auto page_of = [&](int t) {     // of key t 64 + lane, asked for only where a column sees it
    const int j = t * TILE_KEYS + lane;
    return (j >= lo_min || j < keep_max) && j <= pos_hi ? table[j / P] : -1;
  };
  // (asked for with page 0 in place of one that no column sees, and such keys made zero when they come: nothing waits here)
  f4 k_next[K_LOADS], v_next[V_LOADS];
  unsigned k_seen = 0, v_seen = 0;
  bool partly = false;            // some column does not see all of the tile's keys
  auto load = [&](int t, int page) {
    const int off = (t * TILE_KEYS + lane) % P;
    k_seen = 0;
#pragma unroll
    for (int n = 0; n < K_LOADS; ++n) {
      const int u = threadIdx.x + n * THREADS, key = u / (DK / 4), e = u % (DK / 4) * 4;
      const int pg = __shfl(page, key, WAVE), of = __shfl(off, key, WAVE);
      k_seen |= (pg >= 0 ? 1u : 0u) << n;
      k_next[n] = *(const f4*)(a.k_cache + (((size_t)max(pg, 0) * a.nKV + kvh) * P + of) * KD + map * DK + e);
    }
    // (four keys of a value's row lie in one page; those of them that are seen know it)
    const int quad = threadIdx.x % (TILE_KEYS / 4), of = __shfl(off, 4 * quad, WAVE);
    int some = 0;
    v_seen = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int pg = __shfl(page, 4 * quad + i, WAVE);
      v_seen |= (pg >= 0 ? 1u : 0u) << i;
      some = max(some, pg);
    }
    partly = t * TILE_KEYS + TILE_KEYS - 1 > pos_lo || t * TILE_KEYS < lo_max;
#pragma unroll
    for (int n = 0; n < V_LOADS; ++n) {
      const int e = (threadIdx.x + n * THREADS) / (TILE_KEYS / 4);
      v_next[n] = *(const f4*)(a.v_cache + (((size_t)some * a.nKV + kvh) * DV + e) * P + of);
    }
  };

  f4 acc[VC], all[SPLIT || ALL_IN_LDS ? 1 : VC];
  float m, l, all_m = -INFINITY, all_l = 0.f;
  struct Place { int part, t; };
  auto here_or_on = [&](Place at) {          // past the last tile: on to the next parts
    while (at.part < PARTS && at.t > last_tile) {
      at.part = SPLIT ? PARTS : at.part + 1;
      at.t = at_or_after(at.part);
    }
    return at;
  };
  auto begin_part = [&](int n) {
    m = has_sink && n == 0 ? sink_score : -INFINITY;
    l = has_sink && n == 0 ? 1.f : 0.f;
#pragma unroll
    for (int c = 0; c < VC; ++c) acc[c] = f4{0.f, 0.f, 0.f, 0.f};
  };
  auto end_part = [&](int n) {
    if (SPLIT) return;
    const bool first = n == 0, some = !(l == 0.f);
    const float most = fmaxf(all_m, m);
    const float fa = all_l > 0.f ? expf(all_m - most) : 0.f, fb = l > 0.f ? expf(m - most) : 0.f;
    all_l = first ? l : some ? fmaf(l, fb, all_l * fa) : all_l;
    all_m = first ? m : some ? most : all_m;
#pragma unroll
    for (int c = 0; c < VC; ++c) {
      f4 to = first ? acc[c] : ALL_IN_LDS ? all_s[c * THREADS + threadIdx.x] : all[ALL_IN_LDS ? 0 : c];
#pragma unroll
      for (int r = 0; r < 4; ++r) to[r] = !first && some ? fmaf(acc[c][r], fb, to[r] * fa) : to[r];
      if (ALL_IN_LDS) all_s[c * THREADS + threadIdx.x] = to;
      else all[SPLIT || ALL_IN_LDS ? 0 : c] = to;
    }
  };
  begin_part(only);
  Place at = here_or_on({only, at_or_after(only)}), next = at;
  int page = -1;
  if (at.part < PARTS) {                     // (otherwise SPLIT, and a part without tiles)
    load(at.t, page_of(at.t));
    next = here_or_on({at.part, at_or_after(at.t + PARTS)});
    if (next.part < PARTS) page = page_of(next.t);
  }
  if (!SPLIT && at.part > 0) {               // (parts without tiles but the first, which holds the sink, change nothing)
    end_part(0);
    begin_part(at.part);
  }
  if (threadIdx.x == 0) odd_value = 0;

  while (at.part < PARTS) {
    __syncthreads();              // the last tile is done with
    if (partly) {
      bool odd = false;
#pragma unroll
      for (int n = 0; n < K_LOADS; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) k_next[n][i] = k_seen >> n & 1 ? k_next[n][i] : 0.f;
#pragma unroll
      for (int n = 0; n < V_LOADS; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v_next[n][i] = v_seen >> i & 1 ? v_next[n][i] : 0.f;
          odd = odd || !(fabsf(v_next[n][i]) < INFINITY);
        }
      if (odd) odd_value = 1;
    }
#pragma unroll
    for (int n = 0; n < K_LOADS; ++n) {
      const int u = threadIdx.x + n * THREADS;
      *(f4*)(k_s + u / (DK / 4) * KS + u % (DK / 4) * 4) = k_next[n];
    }
#pragma unroll
    for (int n = 0; n < V_LOADS; ++n) {
      const int u = threadIdx.x + n * THREADS;
      *(f4*)(v_s + u / (TILE_KEYS / 4) * VS + u % (TILE_KEYS / 4) * 4) = v_next[n];
    }
    __syncthreads();
    // (the next tile's keys and values, and the pages of the one behind it, are asked for here)
    Place behind = next;
    if (next.part < PARTS) {
      load(next.t, page);
      behind = here_or_on({next.part, at_or_after(next.t + PARTS)});
      if (behind.part < PARTS) page = page_of(behind.t);
    }
    const int t0 = at.t * TILE_KEYS;
    const bool takes = t0 >= t_first && t0 <= pos && !(t0 >= keep && t0 + TILE_KEYS <= lo);
    if (__any(takes)) {           // (uniform over the wave)
      const bool whole = __all(takes && t0 + TILE_KEYS - 1 <= pos && t0 >= lo);
      unsigned sees = 0xffff;     // this lane's keys that its column sees
      if (!whole) {
        sees = 0;
#pragma unroll
        for (int x = 0; x < 16; ++x) {
          const int j = t0 + 4 * x + grp;
          sees |= ((j >= lo || j < keep) && j <= pos ? 1u : 0u) << x;
        }
      }
      // key 16 b + 4 r + grp of the tile in lane group grp, register r of block b
      f4 s[4];
      const float* kr = k_s + (4 * (i16 % 4) + i16 / 4) * KS + grp;
#pragma unroll
      for (int b = 0; b < 4; ++b) s[b] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < DK / 4; ++e)
#pragma unroll
        for (int b = 0; b < 4; ++b) s[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[16 * b * KS + 4 * e], q[e], s[b], 0, 0, 0);
      float most = -INFINITY;
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[b][r] = sees >> (4 * b + r) & 1 ? s[b][r] * a.scale : -INFINITY;
          most = fmaxf(most, s[b][r]);
        }
      most = fmaxf(most, __shfl_xor(most, 16, WAVE));
      most = fmaxf(most, __shfl_xor(most, 32, WAVE));
      const float m_new = fmaxf(m, most);
      // (as in the plain kernel: a tile of scores of minus infinity counts for nothing beside a sink or behind the first tile)
      const float from = m_new == -INFINITY && (t0 != t_first || (has_sink && sink_score > -INFINITY)) ? 0.f : m_new;
      const float alpha = takes ? expf(m - from) : 1.f;
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float p = expf(s[b][r] - from);
          s[b][r] = sees >> (4 * b + r) & 1 ? p : 0.f;
        }
      float sum[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) sum[r] = (s[0][r] + s[2][r]) + (s[1][r] + s[3][r]);
      float total = (sum[0] + sum[2]) + (sum[1] + sum[3]);
      total += __shfl_xor(total, 32, WAVE);
      total += __shfl_xor(total, 16, WAVE);
      l = fmaf(l, alpha, total);
      m = takes ? m_new : m;
#pragma unroll
      for (int c = 0; c < VC; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[c][r] *= alpha;
      const float* vr = v_s + i16 * VS + grp;
      if (!whole && odd_value) {
        // values that are not finite, and columns that do not see their keys: element by element, only what is seen
        // (key 4 x + g of column i16: register x of lane 16 g + i16)
#pragma unroll 1
        for (int x = 0; x < 16; ++x) {
#pragma unroll 1
          for (int g = 0; g < 4; ++g) {
            const int key = 4 * x + g, j = t0 + key;
            const float p = __shfl(s[0][0], 16 * g + i16, WAVE);
            if ((j >= lo || j < keep) && j <= pos) {
#pragma unroll
              for (int c = 0; c < VC; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[c][r] = fmaf(p, v_s[(16 * c + 4 * grp + r) * VS + key], acc[c][r]);
            }
          }
#pragma unroll
          for (int b = 0; b < 4; ++b)             // the next weight to the front
            s[b] = f4{s[b][1], s[b][2], s[b][3], b < 3 ? s[b < 3 ? b + 1 : 3][0] : 0.f};
        }
      } else {
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int c = 0; c < VC; ++c)
              acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[16 * c * VS + 16 * b + 4 * r], s[b][r], acc[c], 0, 0, 0);
      }
    }
    if (next.part != at.part) {
      end_part(at.part);
      if (!SPLIT) begin_part(next.part);
    }
    at = next;
    next = behind;
  }
  if (!real) return;
  const size_t at_row = (size_t)(row0 + row) * a.nH + head;
  if (a.part_o) {
    const size_t place = (at_row * a.maps + map) * (SPLIT ? PARTS : 1) + only;
    float* to = a.part_o + place * DV + 4 * grp;
    const float pl = SPLIT ? l : all_l;
    if (!(pl == 0.f)) {
#pragma unroll
      for (int c = 0; c < VC; ++c) *(f4*)(to + 16 * c) = SPLIT ? acc[c] : ALL_IN_LDS ? all_s[c * THREADS + threadIdx.x] : all[SPLIT || ALL_IN_LDS ? 0 : c];
    }
    if (grp == 0) { a.part_ml[2 * place] = SPLIT ? m : all_m; a.part_ml[2 * place + 1] = pl; }
    return;
  }
  float* to = a.out + at_row * DV + 4 * grp;
  const float inv = (all_l > 0.f ? 1.f / all_l : 0.f) * (a.gate ? a.gate[at_row] : 1.f);
#pragma unroll
  for (int c = 0; c < VC; ++c) {
    f4 o = ALL_IN_LDS ? all_s[c * THREADS + threadIdx.x] : all[SPLIT || ALL_IN_LDS ? 0 : c];
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] *= inv;
    *(f4*)(to + 16 * c) = o;
  }
}

// A wave joins the parts of a (row, head) that workgroups of their own left, and takes the second map from the first.
template <int DC, int MAPS>
__global__ __launch_bounds__(256) void attn_f32_join_kernel(F32Args a, int dv, int cols, int parts) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x % WAVE, G = a.nH / a.nKV;
  // tile by tile as the first launch had them, its columns of every kv head
  const long long item = (long long)blockIdx.x * 4 + threadIdx.x / WAVE;
  const int kvh = (int)(item / cols % a.nKV), tile = (int)(item / cols / a.nKV);
  if (tile >= a.n_tiles) return;
  const int req = a.tiles[2 * tile], col = a.tiles[2 * tile + 1] + (int)(item % cols);
  if (col >= a.q_len[req] * G) return;
  const size_t at_row = (size_t)(a.q_start[req] + col / G) * a.nH + kvh * G + col % G;
  float acc[MAPS][DC], l[MAPS];
#pragma unroll
  for (int w = 0; w < MAPS; ++w) {
    const float* o = a.part_o + (at_row * MAPS + w) * parts * dv + lane;
    const float* ml = a.part_ml + (at_row * MAPS + w) * parts * 2;
    float m = ml[0];
    l[w] = ml[1];
#pragma unroll
    for (int c = 0; c < DC; ++c) acc[w][c] = l[w] == 0.f || lane + c * WAVE >= dv ? 0.f : o[c * WAVE];
    for (int n = 1; n < parts; ++n) {
      const float mn = ml[2 * n], ln = ml[2 * n + 1];
      if (ln == 0.f) continue;
      const float most = fmaxf(m, mn);
      const float fa = l[w] > 0.f ? expf(m - most) : 0.f, fb = ln > 0.f ? expf(mn - most) : 0.f;
      l[w] = fmaf(ln, fb, l[w] * fa);
#pragma unroll
      for (int c = 0; c < DC; ++c)
        if (lane + c * WAVE < dv) acc[w][c] = fmaf(o[(size_t)n * dv + c * WAVE], fb, acc[w][c] * fa);
      m = most;
    }
  }
  float* to = a.out + at_row * dv;
  const float inv = (l[0] > 0.f ? 1.f / l[0] : 0.f) * (a.gate ? a.gate[at_row] : 1.f);
  if (MAPS == 1) {
#pragma unroll
    for (int c = 0; c < DC; ++c)
      if (lane + c * WAVE < dv) to[lane + c * WAVE] = acc[0][c] * inv;
    return;
  }
  const float inv2 = (l[MAPS - 1] > 0.f ? 1.f / l[MAPS - 1] : 0.f) * a.lambda;
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < DC; ++c) {
    acc[0][c] = lane + c * WAVE < dv ? fmaf(acc[0][c], inv, -(acc[MAPS - 1][c] * inv2)) : 0.f;
    ss = fmaf(acc[0][c], acc[0][c], ss);
  }
  const float f = a.out_scale / sqrtf(wave_sum(ss) / (float)dv + a.norm_eps);
#pragma unroll
  for (int c = 0; c < DC; ++c)
    if (lane + c * WAVE < dv) to[lane + c * WAVE] = acc[0][c] * f;
}

#define FOR_SHAPES(X) X(64, 64, 4) X(64, 128, 4) X(96, 96, 4) X(128, 96, 4) X(128, 128, 8)

// The columns of a workgroup for these sizes; 0: there is no kernel for them (pages of multiples of four keys: a value's entries of four keys are one load).
extern "C" int ifx_attn_f32_cols(int d, int dv, int maps, int page_size) {
  if (maps < 1 || maps > 2 || page_size <= 0 || page_size % 4) return 0;
#define TAKES(DK_, DV_, WAVES_) if (d == DK_ && dv == DV_) return WAVES_ * COLS;
  FOR_SHAPES(TAKES)
#undef TAKES
  return 0;
}

// part_o [T, nH, maps, split ? 4 : 1, dv] and part_ml [.., 2]: needed with two maps or split.
extern "C" int ifx_attn_f32(const float* q, const float* k_cache, const float* v_cache, float* out, const int* tiles, int n_tiles,
                            const int* q_start, const int* q_len, const int* kv_len, const int* block_table, int max_blocks,
                            int nH, int nKV, int d, int dv, int page_size, int window, float scale, int keep_first, int has_sink,
                            float sink_score, const float* gate, const float* sinks, int chunk, int maps, float lambda,
                            float out_scale, float norm_eps, int split, float* part_o, float* part_ml, void* stream) {
  IFX_REQUIRE(nH > 0 && nKV > 0 && nH % nKV == 0, "attn_f32: bad head counts nH=%d nKV=%d", nH, nKV);
  IFX_REQUIRE(keep_first >= 0 && chunk >= 0 && window >= 0 && max_blocks > 0, "attn_f32: bad limits");
  const int cols = ifx_attn_f32_cols(d, dv, maps, page_size);
  IFX_REQUIRE(cols, "attn_f32: no kernel for keys of %d x %d, values of %d, pages of %d", maps, d, dv, page_size);
  IFX_REQUIRE(!(split || maps > 1) || (part_o && part_ml), "attn_f32: parts of their own and two maps need room for their results");
  const long long groups = (long long)n_tiles * nKV * maps * (split ? PARTS : 1), joins = (long long)n_tiles * nKV * cols / 4;
  IFX_REQUIRE(n_tiles >= 0 && groups < (1LL << 22) && joins < (1LL << 24), "attn_f32: %d tiles", n_tiles);
  if (n_tiles == 0) return 0;
  F32Args a{q, k_cache, v_cache, out, tiles, q_start, q_len, kv_len, block_table, max_blocks, nH, nKV, page_size, window, maps, scale, keep_first, has_sink, sink_score, gate, sinks, chunk, lambda, out_scale, norm_eps, part_o, part_ml, n_tiles};
  if (!split && maps == 1) a.part_o = a.part_ml = nullptr;
  hipStream_t s = (hipStream_t)stream;
#define GO(DK_, DV_, WAVES_)                                                                                                             \
  if (d == DK_ && dv == DV_) {                                                                                                           \
    if (split) hipLaunchKernelGGL((attn_f32_kernel<DK_, DV_, WAVES_, true>), dim3((unsigned)groups), dim3(WAVE * WAVES_), 0, s, a);      \
    else hipLaunchKernelGGL((attn_f32_kernel<DK_, DV_, WAVES_, false>), dim3((unsigned)groups), dim3(WAVE * WAVES_), 0, s, a);           \
  }
  FOR_SHAPES(GO)
#undef GO
  if (a.part_o) {
    if (maps == 1) hipLaunchKernelGGL((attn_f32_join_kernel<2, 1>), dim3((unsigned)joins), dim3(256), 0, s, a, dv, cols, split ? PARTS : 1);
    else hipLaunchKernelGGL((attn_f32_join_kernel<2, 2>), dim3((unsigned)joins), dim3(256), 0, s, a, dv, cols, split ? PARTS : 1);
  }
  IFX_LAUNCH_CHECK();
}
