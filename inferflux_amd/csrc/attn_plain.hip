// Plain attention over the paged cache: any head size up to 640, float or bf16 storage, float
// math.  The keys of a (query row, query head) come in tiles of 64, aligned to absolute key positions, and the tiles in four
// parts, every fourth tile each: a wave's lanes score one key of a tile each, the wave takes the tile's maximum and sum, then
// every lane accumulates its output elements over the tile's keys in ascending order.  The parts' running maxima, sums and
// outputs are joined in the parts' order.  So the sequence of operations for a (position, head) is the same however the request was
// cut into steps and whatever is beside it: results are bit-equal across cuttings.  This is the attention of the 32-bit
// path, whose prompts a kernel on the matrix cores gives the same bits, and the reference beside the bfloat16 kernels.
//
// What bounds a step of few rows is the chain of a tile's trips to memory, shuffles and dependent additions, about 4 us, so
// four waves take a part each (four rows of 14 heads and 150 keys 9 us, 2,000 keys 57, where one wave takes 19 and 190).  Steps
// of many rows fill the chip with a wave to a row and head, which takes its parts one after the other and leaves out those
// without tiles: neighbouring waves are heads that read the same keys, and no wave waits for others or holds a slot idle
// (64 prompts of 40 tokens, 14 heads of 64 67 us where four waves take 180, 8 of 500 660 and 765; 80 elements in bfloat16 56 and
// 190, 470 and 680).
//
// Formula (runtime/backends/cuda/kernels/flash_attention.cu:71-72 GQA map, 86 causal limit, 144
// scale after the dot product, 152-173 online softmax): head h reads kv head h / (nH / nKV);
// the query at position p sees keys j with max(0, p - window + 1) <= j <= p; s_j = (q . k_j) *
// scale; o = sum_j softmax(s)_j v_j.
//
// Three further parameters, each off when zero: ``keep_first``, the first positions of a request that a windowed
// query still sees beside its window (j <= p and (p - j < window or j < keep_first)), at their true positions;
// ``has_sink``, a key without value whose score is ``sink_score`` and which only takes part in the softmax's
// denominator (with score 0: p_j = exp(s_j) / (1 + sum exp(s_j))); ``gate`` [T, nH], a factor on each head's output.
//
// ``sinks`` [nH] (or null) gives every head a sink score of its own.  ``chunk`` > 0 cuts the sequence into blocks of that
// many positions counted from its start, and a query sees only the keys of its own block (j <= p and j / chunk ==
// p / chunk; together with a window, both limits hold).
//
// Differential attention (``maps`` = 2): a head's query and a kv head's key are two vectors of d elements each, laid out
// one after the other; each pair gives a softmax map of its own over the same values, and the head's output is
// o = a_1 - lambda a_2, divided by its root mean square over the dv elements (norm_eps inside the root), times out_scale.
//
// Cache layouts: K [page][kv head][offset][maps d], V [page][kv head][dv][offset].  Values may have another width
// than keys (dv != d): the output row of a head then has dv elements.
#include "common.h"

IFX_DEFINE_LAST_ERROR()

#define MAX_D 640
#define WAVES_PER_BLOCK 4
#define PARTS 4          // of a row's tiles, every fourth each

// eight consecutive elements as floats: one 16-byte load of bfloat16, two of float
__device__ __forceinline__ void load8(const bf16_t* p, float* v) {
  typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
  const bf16x8 t = *(const bf16x8*)p;
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = (float)t[i];
}
__device__ __forceinline__ void load8(const float* p, float* v) {
  const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

struct AttnArgs {
  const void* q;
  const void* k_cache;
  const void* v_cache;
  void* out;
  const int* row_req;
  const int* positions;
  const int* block_table;
  int max_blocks;
  int T, nH, nKV, d, dv, page_size, window;
  float scale;
  int keep_first;
  int has_sink;
  float sink_score;
  const float* gate;
  const float* sinks;
  int chunk;
  float lambda, out_scale, norm_eps;
  const int* rows;          // the rows to do (null: all)
  int row0, n_rows;         // the launch's, of them
};

// One map's running maximum, sum of weights and weighted values (element e of the values in lane e % 64).
template <int DC>
struct Part {
  float m, l, acc[DC];
};

// ``next`` added to ``all``: the parts of a row in their order.  A part without keys (a sum of 0) changes nothing.
template <int DC>
__device__ __forceinline__ void join(Part<DC>& all, float m, float l, const float* acc) {
  if (l == 0.f) return;
  const float most = fmaxf(all.m, m);
  const float fa = all.l > 0.f ? expf(all.m - most) : 0.f, fb = l > 0.f ? expf(m - most) : 0.f;
  all.l = fmaf(l, fb, all.l * fa);
#pragma unroll
  for (int c = 0; c < DC; ++c) all.acc[c] = fmaf(acc[c], fb, all.acc[c] * fa);
  all.m = most;
}

// ROW_WAVES 4: a workgroup per (row, head), a part of its tiles to a wave; 1: a wave per (row, head), one part after the other.
// DC: sixty-fourths of the values' elements there is room for.  AT_ONCE (keys of up to 64 elements in eights, values of up to 64 DC, pages of multiples of
// eight keys; ROW_WAVES 4): a tile's keys are asked for at once and its values before their weights are known, one trip to memory each
// instead of one after the other for eight elements and eight keys (the same operations in the same order): 4 rows of 14 heads of 64 and 150
// keys 8.3 -> 6.7 us, 600 keys 18.7 -> 14.7, 16 rows and 250 keys 10.1 -> 8.7; in bfloat16 7.8 -> 6.9, 17.3 -> 16.1, 8.6 -> 7.8.
template <typename T, int MAPS, int ROW_WAVES, int DC, bool AT_ONCE>
__global__ __launch_bounds__(WAVE * WAVES_PER_BLOCK) void attn_plain_kernel(AttnArgs a) {
  __shared__ float q_s[ROW_WAVES == 1 ? WAVES_PER_BLOCK : 1][MAX_D];
  __shared__ float joined[ROW_WAVES == 1 ? 1 : MAPS][ROW_WAVES == 1 ? 1 : WAVES_PER_BLOCK][ROW_WAVES == 1 ? 1 : MAX_D + 2];   // each wave's outputs, maximum and sum
  const int wid = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const long long item = ROW_WAVES == 1 ? (long long)blockIdx.x * WAVES_PER_BLOCK + wid : (long long)blockIdx.x;
  // (ROW_WAVES 1: all lanes of a wave leave together, and no barrier of the workgroup follows)
  if (ROW_WAVES == 1 && item >= (long long)a.n_rows * a.nH) return;
  const int nth = a.row0 + (int)(item / a.nH), head = (int)(item % a.nH), row = a.rows ? a.rows[nth] : nth;
  const int d = a.d, dv = a.dv, P = a.page_size;
  const int kvh = head / (a.nH / a.nKV);
  const int pos = a.positions[row];
  const int* table = a.block_table + (size_t)a.row_req[row] * a.max_blocks;
  int lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  if (a.chunk > 0) lo = max(lo, pos - pos % a.chunk);
  const int keep = lo > 0 ? min(a.keep_first, lo) : 0;      // keys [0, keep) and [lo, pos] are seen

  const int kd = MAPS * d;      // elements of a query's and a key's row
  const T* qrow = (const T*)a.q + ((size_t)row * a.nH + head) * kd;
  float* qs = q_s[ROW_WAVES == 1 ? wid : 0];
  if (ROW_WAVES == 1) {
    for (int e = lane; e < kd; e += WAVE) qs[e] = to_f(qrow[e]);
    // qs is written and read by this wave only.
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_s_waitcnt(0);
  } else {
    for (int e = threadIdx.x; e < kd; e += WAVE * WAVES_PER_BLOCK) qs[e] = to_f(qrow[e]);
    __syncthreads();
  }

  // (the sink is a key of score sink_score whose value is zero: it starts the first part's running maximum and sum)
  const bool has_sink = a.has_sink || a.sinks;
  const float sink_score = a.sinks ? a.sinks[head] : a.sink_score;
  const T* Kc = (const T*)a.k_cache;
  const T* Vc = (const T*)a.v_cache;
  const int t_first = keep > 0 ? 0 : (lo / WAVE) * WAVE;
  Part<DC> all[MAPS], part[MAPS];
  // (parts without tiles are left out; the first holds the sink)
  const int tile0 = t_first / WAVE, tiles = pos / WAVE - tile0 + 1;
  bool begun = false;
#pragma unroll 1
  for (int i = 0; i < (ROW_WAVES > 1 ? 1 : PARTS); ++i) {
    const int n = ROW_WAVES > 1 ? wid : i;
    if (ROW_WAVES == 1 && (n - tile0 & (PARTS - 1)) >= tiles && !(has_sink && n == 0)) continue;
#pragma unroll
    for (int w = 0; w < MAPS; ++w) {
      part[w].m = has_sink && n == 0 ? sink_score : -INFINITY;
      part[w].l = has_sink && n == 0 ? 1.f : 0.f;
#pragma unroll
      for (int c = 0; c < DC; ++c) part[w].acc[c] = 0.f;
    }
    for (int t0 = t_first; t0 <= pos; t0 += WAVE) {
      if (t0 >= keep && t0 + WAVE <= lo) {     // between the kept first keys and the window: on to the window's first tile
        t0 = (lo / WAVE) * WAVE - WAVE;
        continue;
      }
      if (t0 / WAVE % PARTS != n) continue;
      const int j = t0 + lane;
      const bool valid = (j >= lo || j < keep) && j <= pos;
      int page = 0, off = 0;
      float s[MAPS], p[MAPS];
      float vv_all[AT_ONCE ? WAVE / 8 : 1][AT_ONCE ? DC : 1][8];
      if constexpr (AT_ONCE) {
        if (valid) page = table[j / P];
#pragma unroll
        for (int g = 0; g < WAVE; g += 8) {
          const int j0 = t0 + g;
          if (j0 > pos || (j0 + 7 < lo && j0 >= keep)) continue;  // uniform over the wave
          // (the eight keys are one page's; the first of them that is seen knows it)
          const int pg = __builtin_amdgcn_readlane(page, j0 < keep || j0 >= lo ? g : g + lo - j0);
          const T* vb = Vc + ((size_t)pg * a.nKV + kvh) * dv * P + j0 % P;
#pragma unroll
          for (int c = 0; c < DC; ++c)
            if (lane + c * WAVE < dv) load8(vb + (size_t)(lane + c * WAVE) * P, vv_all[g / 8][c]);
        }
      }
#pragma unroll
      for (int w = 0; w < MAPS; ++w) s[w] = -INFINITY;
      if (valid) {
        if (!AT_ONCE) page = table[j / P];
        off = j % P;
#pragma unroll
        for (int w = 0; w < MAPS; ++w) {
          const T* kr = Kc + (((size_t)page * a.nKV + kvh) * P + off) * kd + w * d;
          const float* qv = qs + w * d;
          float dot = 0.f;
          auto piece = [&](int e) {
            float kv[8];
            load8(kr + e, kv);
#pragma unroll
            for (int i = 0; i < 8; ++i) dot = fmaf(qv[e + i], kv[i], dot);
          };
          if constexpr (AT_ONCE) {
            float kv[8][8];
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (8 * e < d) load8(kr + 8 * e, kv[e]);
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (8 * e < d) {
#pragma unroll
                for (int i = 0; i < 8; ++i) dot = fmaf(qv[8 * e + i], kv[e][i], dot);
              }
          } else if (d % 8 == 0 && ROW_WAVES == 1) {        // the key's row in 16-byte pieces; the same additions in the same order
#pragma unroll 2
            for (int e = 0; e < d; e += 8) piece(e);
          } else if (d % 8 == 0) {
            for (int e = 0; e < d; e += 8) piece(e);
          } else {
            for (int e = 0; e < d; ++e) dot = fmaf(qv[e], to_f(kr[e]), dot);
          }
          s[w] = dot * a.scale;
        }
      }
#pragma unroll
      for (int w = 0; w < MAPS; ++w) {
        const float m_new = fmaxf(part[w].m, wave_max(s[w]));  // finite unless every score overflows: the tile holds a visible key
        // (a tile of scores of minus infinity counts for nothing beside a sink or behind the row's first tile, whichever wave
        // meets it first)
        const float from = m_new == -INFINITY && (t0 != t_first || (has_sink && sink_score > -INFINITY)) ? 0.f : m_new;
        p[w] = valid ? expf(s[w] - from) : 0.f;
        const float alpha = expf(part[w].m - from);  // 0 on the first tile (m = -inf)
        part[w].l = part[w].l * alpha + wave_sum(p[w]);
#pragma unroll
        for (int c = 0; c < DC; ++c) part[w].acc[c] *= alpha;
        part[w].m = m_new;
      }
      if (P % 8 == 0) {
        // Eight keys at a time: they lie in one page, where a value element's eight entries are 16 consecutive bytes.
        // Keys outside the range have weight 0 and their entries (stale or zero, never written with anything that is
        // not finite) add nothing; an element's sum still runs over the keys in ascending order.
#pragma unroll
        for (int g = 0; g < WAVE; g += 8) {
          const int j0 = t0 + g;
          if (j0 > pos || (j0 + 7 < lo && j0 >= keep)) continue;  // uniform over the wave
          float pj[MAPS][8];
#pragma unroll
          for (int w = 0; w < MAPS; ++w)
#pragma unroll
            for (int i = 0; i < 8; ++i)
              pj[w][i] = AT_ONCE ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p[w]), g + i)) : __shfl(p[w], g + i, WAVE);
          if constexpr (AT_ONCE) {
#pragma unroll
            for (int c = 0; c < DC; ++c)
              if (lane + c * WAVE < dv) {
#pragma unroll
                for (int w = 0; w < MAPS; ++w)
#pragma unroll
                  for (int i = 0; i < 8; ++i) part[w].acc[c] = fmaf(pj[w][i], vv_all[g / 8][c][i], part[w].acc[c]);
              }
            continue;
          }
          const T* vb = Vc + ((size_t)table[j0 / P] * a.nKV + kvh) * dv * P + j0 % P;
#pragma unroll
          for (int c = 0; c < DC; ++c) {
            const int e = lane + c * WAVE;
            if (e < dv) {
              float vv[8];
              load8(vb + (size_t)e * P, vv);
#pragma unroll
              for (int w = 0; w < MAPS; ++w)
#pragma unroll
                for (int i = 0; i < 8; ++i) part[w].acc[c] = fmaf(pj[w][i], vv[i], part[w].acc[c]);
            }
          }
        }
      } else
      for (int jj = 0; jj < WAVE; ++jj) {
        float pj[MAPS];
        bool none = true;
#pragma unroll
        for (int w = 0; w < MAPS; ++w) {
          pj[w] = __shfl(p[w], jj, WAVE);
          none = none && pj[w] == 0.f;
        }
        const int pg = __shfl(page, jj, WAVE), of = __shfl(off, jj, WAVE);
        if (none) continue;  // uniform over the wave; keys outside the range are never read
        const T* vb = Vc + ((size_t)pg * a.nKV + kvh) * dv * P + of;
#pragma unroll
        for (int c = 0; c < DC; ++c) {
          const int e = lane + c * WAVE;
          if (e < dv) {
            const float vv = to_f(vb[(size_t)e * P]);
#pragma unroll
            for (int w = 0; w < MAPS; ++w) part[w].acc[c] = fmaf(pj[w], vv, part[w].acc[c]);
          }
        }
      }
    }
    if (ROW_WAVES == 1) {
#pragma unroll
      for (int w = 0; w < MAPS; ++w) {
        if (!begun) all[w] = part[w];
        else join(all[w], part[w].m, part[w].l, part[w].acc);
      }
      begun = true;
    }
  }
  if (ROW_WAVES > 1) {      // every element by one lane of the first wave
#pragma unroll
    for (int w = 0; w < MAPS; ++w) {
      all[w] = part[w];
#pragma unroll
      for (int c = 0; c < DC; ++c)
        if (lane + c * WAVE < dv) joined[w][wid][lane + c * WAVE] = part[w].acc[c];
      if (lane == 0) { joined[w][wid][MAX_D] = part[w].m; joined[w][wid][MAX_D + 1] = part[w].l; }
    }
    __syncthreads();
    if (wid > 0) return;
#pragma unroll
    for (int w = 0; w < MAPS; ++w)
#pragma unroll
      for (int k = 1; k < PARTS; ++k) {
        float acc[DC];
#pragma unroll
        for (int c = 0; c < DC; ++c) acc[c] = lane + c * WAVE < dv ? joined[w][k][lane + c * WAVE] : 0.f;
        join(all[w], joined[w][k][MAX_D], joined[w][k][MAX_D + 1], acc);
      }
  }
  T* orow = (T*)a.out + ((size_t)row * a.nH + head) * dv;
  const float inv = (all[0].l > 0.f ? 1.f / all[0].l : 0.f) * (a.gate ? a.gate[(size_t)row * a.nH + head] : 1.f);
  if (MAPS == 1) {
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      const int e = lane + c * WAVE;
      if (e < dv) orow[e] = from_f<T>(all[0].acc[c] * inv);
    }
    return;
  }
  // the second map subtracted, the head's root mean square over dv, the constant factor
  const float inv2 = (all[MAPS - 1].l > 0.f ? 1.f / all[MAPS - 1].l : 0.f) * a.lambda;
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < DC; ++c) {
    const int e = lane + c * WAVE;
    all[0].acc[c] = e < dv ? all[0].acc[c] * inv - all[MAPS - 1].acc[c] * inv2 : 0.f;
    ss = fmaf(all[0].acc[c], all[0].acc[c], ss);
  }
  const float f = a.out_scale / sqrtf(wave_sum(ss) / (float)dv + a.norm_eps);
#pragma unroll
  for (int c = 0; c < DC; ++c) {
    const int e = lane + c * WAVE;
    if (e < dv) orow[e] = from_f<T>(all[0].acc[c] * f);
  }
}

// Waves to a (row, head): four where the launch leaves most of the chip's waves free by a wave each.  us by one : by four waves of
// 512 items and 60 / 250 keys 9 : 9, 28 : 16 (64 elements), 12 : 13, 44 : 24 (128), 42 : 34, 149 : 71 (576); of 900 items 9 : 10, 32 : 24 and,
// 1,000 keys, 115 : 74 (64), 137 : 63 (80, bfloat16), but 12 : 17, 44 : 49 and 158 : 179 (128), 40 : 42, 140 : 157 and 700 : 686 (576); of 2,800
// items and 250 keys 48 : 58 (64), 49 : 55 (80).
static int choose_row_waves(long long items, long long keys, int width) {
  return items <= 512 || (items <= 1024 && keys > 128 && width <= 96) ? 4 : 1;
}

extern "C" int ifx_attn_plain(const void* q, const void* k_cache, const void* v_cache, void* out, int dtype,
                              const int* row_req, const int* positions, const int* block_table,
                              int max_blocks, int T, int nH, int nKV, int d, int dv, int page_size, int window,
                              float scale, int keep_first, int has_sink, float sink_score, const float* gate, const float* sinks,
                              int chunk, int maps, float lambda, float out_scale, float norm_eps, int row_waves, const int* rows_of, void* stream) {
  IFX_REQUIRE(keep_first >= 0, "attn_plain: keep_first %d", keep_first);
  IFX_REQUIRE(T >= 0 && nH > 0 && nKV > 0 && nH % nKV == 0, "attn_plain: bad head counts nH=%d nKV=%d", nH, nKV);
  IFX_REQUIRE(maps == 1 || maps == 2, "attn_plain: %d maps (1 or 2)", maps);
  IFX_REQUIRE(chunk >= 0, "attn_plain: chunk %d", chunk);
  IFX_REQUIRE(d > 0 && maps * d <= MAX_D, "attn_plain: head_dim %d x %d outside 1..%d", maps, d, MAX_D);
  IFX_REQUIRE(dv > 0 && dv <= MAX_D, "attn_plain: value head_dim %d outside 1..%d", dv, MAX_D);
  IFX_REQUIRE(page_size > 0 && max_blocks > 0 && window >= 0, "attn_plain: bad page_size/max_blocks/window");
  if (T == 0) return 0;
  IFX_REQUIRE(dtype == DT_F32 || dtype == DT_BF16, "attn_plain: unknown dtype %d", dtype);
  IFX_REQUIRE(row_waves == 0 || row_waves == 1 || row_waves == 4, "attn_plain: %d waves to a row and head (0, 1 or 4)", row_waves);
  if (row_waves == 0) row_waves = choose_row_waves((long long)T * nH, (long long)max_blocks * page_size, maps * d);
  AttnArgs a{q, k_cache, v_cache, out, row_req, positions, block_table, max_blocks, T, nH, nKV, d, dv, page_size, window, scale, keep_first, has_sink, sink_score, gate, sinks, chunk, lambda, out_scale, norm_eps, rows_of, 0, 0};
  hipStream_t s = (hipStream_t)stream;
  // (a tile's values take registers: two waves to a SIMD of up to 64 elements, one of up to 128, so the items that are there at once)
  const bool at_once = d % 8 == 0 && d <= 64 && dv <= 128 && page_size % 8 == 0 && (long long)T * nH <= (dv <= 64 ? 512 : 256);
  const int rows = max(1, (1 << 23) / nH);          // rows of a launch: a grid holds fewer than 2^32 threads
  for (; a.row0 < T; a.row0 += a.n_rows) {
    a.n_rows = min(rows, T - a.row0);
    const unsigned items = (unsigned)a.n_rows * (unsigned)nH;
    const dim3 blocks(row_waves == 1 ? (items + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK : items), threads(WAVE * WAVES_PER_BLOCK);
#define GO(T_, MAPS_)                                                                                        \
  do {                                                                                                       \
    if (row_waves == 1) hipLaunchKernelGGL((attn_plain_kernel<T_, MAPS_, 1, MAX_D / WAVE, false>), blocks, threads, 0, s, a);     \
    else if (at_once && dv <= 64) hipLaunchKernelGGL((attn_plain_kernel<T_, MAPS_, 4, 1, true>), blocks, threads, 0, s, a); \
    else if (at_once) hipLaunchKernelGGL((attn_plain_kernel<T_, MAPS_, 4, 2, true>), blocks, threads, 0, s, a); \
    else hipLaunchKernelGGL((attn_plain_kernel<T_, MAPS_, 4, MAX_D / WAVE, false>), blocks, threads, 0, s, a); \
  } while (0)
    if (dtype == DT_F32 && maps == 1) GO(float, 1);
    else if (dtype == DT_BF16 && maps == 1) GO(bf16_t, 1);
    else if (dtype == DT_F32) GO(float, 2);
    else GO(bf16_t, 2);
#undef GO
  }
  IFX_LAUNCH_CHECK();
}
