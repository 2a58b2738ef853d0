// Products of many rows with the activation as their epilogue, on the matrix cores (bfloat16 in and out, float sums), from the sums
// as they are:
//   OUT_PAIRS   out[M][N / 2] = act(x Wg^T) * (x Wu^T), W [N][K] with the rows of Wg and Wu in turn: a lane holds a gate and its up
//   OUT_ACT     out[M][N] = act(x W^T)
// The library's product followed by a launch for the activation writes the N columns and reads them back (2,048 rows of
// 37,888 columns: 233 MB, 40 us of 552) and rounds them to bfloat16 in between.
//
// The inner loop is wave_tiles.h, and for small tiles, of which up to three workgroups to a CU hide each other's ends, product_tiles.h.
// What is chosen here is the tile.  A large tile reads less of LDS and of the caches for its products, but there are few of
// them, and the last of the rounds that they take on 256 CUs may be nearly empty (600 rows of 22,016 x 2,048: 258 tiles of
// 256 x 256 take 89 us, 232 of 384 x 160 49 us).  So choose_tile() takes the tile whose rounds are estimated to take least, from
// what rounds of each were measured to take (see `kinds`: gate/up of 1,337 sizes with cold weights, off by 10 % in the mean square; the choice
// is 0.3 to 0.7 % off the best tile in the mean, by coefficients fitted to one half 0.4 to 1 % at the other; 384 x 128, 256 x 160 and 128 x 256
// were the best of all by 1 % in the mean, and left out).
// 2,048 rows of 37,888 x 3,584: 425 us (1,310 TFLOP/s; tiles of 256 x 256 by eight waves took 481, the library and the
// activation 552); 600 of 22,016 x 2,048 51 (93; 72); 4,500 of 17,920 x 1,536 200 (255; 239).  Which sizes come here is a rule
// of ops.py (many_tiles_take, pairs_tiles_take), with both sides measured.
//
// The plain product of deep weights, too, for callers that add partial sums (down):
//   OUT_SUMS    parts[slice][M][N] = x W^T over a slice of K, in float
// The library's has no kernel that fits some of these sizes (6,144 rows of 3,584 x 18,944, where 336 tiles of 256 x 256 are 1.3 rounds:
// 1,061 us, 786 TFLOP/s) and its batched product over slices none that fits others (520 rows 115 us, 1,034 of 2,048 x 11,008 62).
// Slices of tiles fill the rounds: 650, 69 and 45 us.  Which sizes, tiles and slices: ifx_gemm_tiles_sums_plan.
#include "product_tiles.h"
#include "wave_tiles.h"
#include "tile_acts.h"

IFX_DEFINE_LAST_ERROR()

typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;

enum { OUT_PAIRS = 0, OUT_ACT = 1, OUT_SUMS = 2 };

struct TilesArgs {
  const bf16_t* x;          // [M][K]
  const bf16_t* w;          // [N][K]
  void* out;                // OUT_PAIRS: bf16 [M][N / 2]; OUT_ACT: bf16 [M][N]; OUT_SUMS: float [slices][M][N]
  int M, N, K, act;
  float limit;
  int slices, slice_k;      // K in so many slices of slice_k values (a multiple of 64; the last what is left)
};

#define GROUP 4          // tiles of x that meet a tile of W one after the other

template <int FN, int FM, int OUT>
struct TilesOut {
  static constexpr bool TURNED = OUT != OUT_SUMS;          // (a lane's four sums in float are a whole store)
  static constexpr int CHUNK = OUT == OUT_ACT && (FN > 8 || WaveTiles<FN, FM>::SLOTS > 2) ? FN / 2 : FN;          // fragments that are turned in LDS at a time
  static constexpr int ROW = 16 * CHUNK * (OUT == OUT_PAIRS ? 1 : 2);      // bytes of a row of them
  static constexpr int PITCH = ROW + 16, WAVE_BYTES = TURNED ? 16 * PITCH : 0;
  static constexpr int LDS = WaveTiles<FN, FM>::LDS + 4 * WAVE_BYTES;
};

template <int FN, int FM, int OUT, int ACT>
__device__ __forceinline__ void tiles_out(const WaveTiles<FN, FM>& p, const TilesArgs& a, unsigned char* lds, tile_floatx4 (&acc)[FN][FM], int m, int n) {
  typedef TilesOut<FN, FM, OUT> O;
  // this wave's results: a buffer from its first row on; stores beyond it, or with TILE_NO_ROW for an offset, are dropped
  const int columns = OUT == OUT_PAIRS ? a.N / 2 : a.N, first = OUT == OUT_PAIRS ? n / 2 : n;
  const int rows = a.M - m;
  const unsigned long long at0 = (unsigned long long)a.out + (size_t)m * columns * 2;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)at0), hi = __builtin_amdgcn_readfirstlane((unsigned)(at0 >> 32));
  const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc((void*)((unsigned long long)hi << 32 | lo), 0,
                                                                        __builtin_amdgcn_readfirstlane(max(0, min(16 * FM, rows)) * columns * 2), 0x00020000);
  // 16 rows of the wave's results at a time, turned in LDS so that they go out in whole lines
  unsigned char* st = lds + WaveTiles<FN, FM>::LDS + p.wid * O::WAVE_BYTES;
  const bool whole = columns % 8 == 0;
#pragma unroll
  for (int b = 0; b < FM; ++b)
#pragma unroll
    for (int c0 = 0; c0 < FN; c0 += O::CHUNK) {
#pragma unroll
      for (int c = 0; c < O::CHUNK; ++c) {
        asm volatile("" : "+a"(acc[c0 + c][b]));          // (not before: the registers beside the sums are taken)
        const tile_floatx4 v = acc[c0 + c][b];
        if (OUT == OUT_PAIRS) {
          bf16x2 y;
          y[0] = (__bf16)tile_gated<ACT>(v[0], v[1], a.limit);
          y[1] = (__bf16)tile_gated<ACT>(v[2], v[3], a.limit);
          *(bf16x2*)(st + p.col * O::PITCH + c * 16 + p.g * 4) = y;
        } else {
          bf16x4 y;
#pragma unroll
          for (int r = 0; r < 4; ++r) y[r] = (__bf16)tile_act<ACT>(v[r]);
          *(bf16x4*)(st + p.col * O::PITCH + c * 32 + p.g * 8) = y;
        }
      }
      constexpr int PIECES = O::ROW / 16;
      const int from = first + c0 * (OUT == OUT_PAIRS ? 8 : 16), step = 16 * b * columns * 2;
      if (whole) {
#pragma unroll
        for (int j0 = 0; j0 < 16 * PIECES; j0 += 64) {
          const int j = j0 + p.lane, r = j / PIECES, at = 8 * (j % PIECES);
          const bool in = j < 16 * PIECES && r < rows - 16 * b && from + at < columns;
          const tile_uintx4 v = *(const tile_uintx4*)(st + min(r, 15) * O::PITCH + 2 * at);
          __builtin_amdgcn_raw_buffer_store_b128(v, out, in ? (r * columns + from + at) * 2 : TILE_NO_ROW, step, 0);
        }
      } else {            // (an even number of columns)
#pragma unroll 1
        for (int j = p.lane; j < 64 * PIECES; j += 64) {
          const int r = j / (4 * PIECES), at = 2 * (j % (4 * PIECES));
          const bool in = r < rows - 16 * b && from + at < columns;
          const unsigned v = *(const unsigned*)(st + r * O::PITCH + 2 * at);
          __builtin_amdgcn_raw_buffer_store_b32(v, out, in ? (r * columns + from + at) * 2 : TILE_NO_ROW, step, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
}

// The sums of a slice of K as they are; stores beyond the rows and columns are dropped.
template <int FN, int FM>
__device__ __forceinline__ void tiles_sums(const WaveTiles<FN, FM>& p, const TilesArgs& a, tile_floatx4 (&acc)[FN][FM], int slice, int m, int n) {
  const int rows = a.M - m;
  const unsigned long long at0 = (unsigned long long)a.out + ((size_t)slice * a.M + min(m, a.M)) * a.N * 4;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)at0), hi = __builtin_amdgcn_readfirstlane((unsigned)(at0 >> 32));
  const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc((void*)((unsigned long long)hi << 32 | lo), 0,
                                                                        __builtin_amdgcn_readfirstlane(max(0, min(16 * FM, rows)) * a.N * 4), 0x00020000);
#pragma unroll
  for (int b = 0; b < FM; ++b) {
#pragma unroll
    for (int c = 0; c < FN; ++c) {
      asm volatile("" : "+a"(acc[c][b]));
      const int at = n + 16 * c + 4 * p.g;
      const bool in = p.col < rows - 16 * b && at < a.N;
      const tile_floatx4 v = acc[c][b];
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(tile_uintx4, v), out, in ? (p.col * a.N + at) * 4 : TILE_NO_ROW, 16 * b * a.N * 4, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// One workgroup to a CU, one tile after the other.  Workgroup b runs on XCD b % 8, which takes a contiguous range of the tiles.
template <int FN, int FM, int OUT>
__global__ __launch_bounds__(256, 1) void tiles_kernel(TilesArgs a) {
  typedef WaveTiles<FN, FM> P;
  typedef TilesOut<FN, FM, OUT> O;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[O::LDS];
  static_assert(O::LDS <= 160 * 1024, "LDS");
  const int nt = (a.N + P::BN - 1) / P::BN, mt = (a.M + P::BM - 1) / P::BM, total = nt * mt * a.slices;
  const int per = (total + 7) / 8, end = min(total, (int)(blockIdx.x % 8 + 1) * per), stride = gridDim.x / 8;
  int id = blockIdx.x % 8 * per + blockIdx.x / 8;
  if (id >= end) return;
  P p;
  p.init(lds);
  int n0, m0, share, sharers, slice = 0, K = a.K;
  auto find = [&](int t) {          // groups of GROUP tiles of x by all of W's
    auto div = [](int v, int by) { return __builtin_amdgcn_readfirstlane(v / by); };        // (by vector instructions: back to scalars)
    if (OUT == OUT_SUMS) {
      slice = div(t, nt * mt), t -= slice * nt * mt;
      K = min(a.slice_k, a.K - slice * a.slice_k);
    }
    const int turn = div(t, GROUP * nt), in = t - turn * GROUP * nt;
    sharers = min(GROUP, mt - turn * GROUP);
    const int tn = div(in, sharers);
    share = in - tn * sharers;
    m0 = (turn * GROUP + share) * P::BM, n0 = tn * P::BN;
  };
  auto rows_of_w = [&]() {
    const int k0 = slice * a.slice_k;
    return tile_buffer(a.w + (size_t)n0 * a.K + k0, ((unsigned)min(P::BN, a.N - n0) * (unsigned)a.K - (unsigned)k0) * 2u);
  };
  auto begin = [&]() {
    const int count = min(P::BM, a.M - m0);
    const int k0 = slice * a.slice_k;
    const tile_uintx4 x = tile_buffer(a.x + (size_t)m0 * a.K + k0, ((unsigned)count * (unsigned)a.K - (unsigned)k0) * 2u);
    p.begin(rows_of_w(), x, K, a.K * 2, [&](int m, int) { return m < count ? m * a.K * 2 : TILE_NO_ROW; });
    p.touch_rows(share, sharers, a.K * 2);
  };
  find(id);
  begin();
  while (true) {
    const int n = n0 + p.wn(), m = m0 + p.wm(), this_slice = slice, this_k = K;
    id += stride;
    const bool more = id < end;
    if (more) find(id);
    p.next = rows_of_w(), p.next_steps = more ? (K + 63) / 64 : 0;
    if (!more) p.next[2] = 0;          // (nothing to touch)
    tile_floatx4 acc[FN][FM];
    p.run(lds, this_k, acc);
    if (more) begin();
    if constexpr (OUT == OUT_SUMS) tiles_sums<FN, FM>(p, a, acc, this_slice, m, n);
    else switch (a.act) {
      case ACT_GELU_TANH: tiles_out<FN, FM, OUT, ACT_GELU_TANH>(p, a, lds, acc, m, n); break;
      case ACT_SILU: tiles_out<FN, FM, OUT, ACT_SILU>(p, a, lds, acc, m, n); break;
      case ACT_NONE: if constexpr (OUT == OUT_ACT) tiles_out<FN, FM, OUT, ACT_NONE>(p, a, lds, acc, m, n); break;
      default: tiles_out<FN, FM, OUT, OUT == OUT_PAIRS ? ACT_CLAMPED_SWISH : ACT_RELU_SQUARED>(p, a, lds, acc, m, n); break;
    }
    if (!more) break;
  }
}

// Tiles by small waves on product_tiles.h, a tile to a workgroup: for products of some hundred rows, whose tiles of 256 x 256 are few.
// They are bound by the trips to memory of a short walk (three stages of loads stand between a request and its use) and, large ones,
// by the caches: tiles of 64 x 64 by four waves, three workgroups to a CU, of 128 x 64 by eight, two, of 128 x 128 by eight, one.  us of
// sums, cold weights, by large tiles (slices and what they cost the reader included) / the library / here: 150 rows of 896 x 896
// 10.7 / 7.7 / 5.6, of 896 x 4,864 16.3 / 11.3 / 8.5, 300 of 1,536 x 8,960 29.4 / 30.2 / 22.8, 512 of 2,048 x 2,048 19.0 / 11.3 / 11.2; 100 rows by
// the product that shares x through LDS / here of 2,048 x 2,048 12.2 / 7.4, of 2,048 x 11,008 27.8 / 19.3; gate/up of 150 and 300 rows of 9,728 x 896 17.2 / 16.2 / 11.1 and 17.3 / 19.3 / 14.0.
// Four stages of 64 x 64 and 64 rows by 128 items were within 2 % of these; the two tiles of two stages that were here before (192 x 128,
// 128 x 128) nowhere better.
template <int BN, int BM, int WN, int WM, int OUT, int ACT>
__device__ __forceinline__ void small_out(const TilesArgs& a, tile_floatx4 (&acc)[WN / 16][WM / 16], int slice, int m0, int n0) {
  const int lane = threadIdx.x % 64, g = lane / 16;
#pragma unroll
  for (int b = 0; b < WM / 16; ++b) {
    const int m = m0 + 16 * b + lane % 16;
    if (m >= a.M) continue;
#pragma unroll
    for (int c = 0; c < WN / 16; ++c) {
      const int n = n0 + 16 * c + 4 * g;
      if (n >= a.N) continue;
      const tile_floatx4 v = acc[c][b];
      if constexpr (OUT == OUT_PAIRS) {
        bf16x2 y;
        y[0] = (__bf16)tile_gated<ACT>(v[0], v[1], a.limit);
        y[1] = (__bf16)tile_gated<ACT>(v[2], v[3], a.limit);
        *(bf16x2*)((bf16_t*)a.out + (size_t)m * (a.N / 2) + n / 2) = y;
      } else if constexpr (OUT == OUT_SUMS) {
        *(tile_floatx4*)((float*)a.out + ((size_t)slice * a.M + m) * a.N + n) = v;
      } else {
        bf16_t* out = (bf16_t*)a.out + (size_t)m * a.N + n;
        bf16x4 y;
#pragma unroll
        for (int r = 0; r < 4; ++r) y[r] = (__bf16)tile_act<ACT>(v[r]);
        if (a.N % 4 == 0) *(bf16x4*)out = y;
        else {          // (N is even)
          *(bf16x2*)out = bf16x2{y[0], y[1]};
          if (n + 2 < a.N) *(bf16x2*)(out + 2) = bf16x2{y[2], y[3]};
        }
      }
    }
  }
}

template <int BN, int BM, int WN, int WM, int PER_CU, int OUT>
__global__ __launch_bounds__(64 * (BN / WN) * (BM / WM), PER_CU * (BN / WN) * (BM / WM) / 4) void small_kernel(TilesArgs a) {
  typedef ProductTiles<BN, BM, WN, WM, false, 3> P;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[P::LDS];
  static_assert(PER_CU * P::LDS <= 160 * 1024, "LDS");
  const int mt = (a.M + BM - 1) / BM;
  int tn, tm;
  if (!product_tile((a.N + BN - 1) / BN, mt * a.slices, min(mt, GROUP), &tn, &tm)) return;
  const int slice = tm / mt, k0 = slice * a.slice_k, K = min(a.slice_k, a.K - k0), m0 = (tm - slice * mt) * BM, n0 = tn * BN;
  const int rows = min(BN, a.N - n0), count = min(BM, a.M - m0);
  const tile_uintx4 w = tile_buffer(a.w + (size_t)n0 * a.K + k0, ((unsigned)rows * (unsigned)a.K - (unsigned)k0) * 2u);
  const tile_uintx4 x = tile_buffer(a.x + (size_t)m0 * a.K + k0, ((unsigned)count * (unsigned)a.K - (unsigned)k0) * 2u);
  tile_floatx4 acc[P::FN][P::FM];
  P::run(lds, w, x, K, a.K, [&](int i) { return i < count ? i * a.K * 2 : TILE_NO_ROW; }, acc);
  const int m = m0 + P::wm(), n = n0 + P::wn();
  if constexpr (OUT == OUT_SUMS) small_out<BN, BM, WN, WM, OUT, ACT_NONE>(a, acc, slice, m, n);
  else switch (a.act) {
    case ACT_GELU_TANH: small_out<BN, BM, WN, WM, OUT, ACT_GELU_TANH>(a, acc, 0, m, n); break;
    case ACT_SILU: small_out<BN, BM, WN, WM, OUT, ACT_SILU>(a, acc, 0, m, n); break;
    case ACT_NONE: if constexpr (OUT == OUT_ACT) small_out<BN, BM, WN, WM, OUT, ACT_NONE>(a, acc, 0, m, n); break;
    default: small_out<BN, BM, WN, WM, OUT, OUT == OUT_PAIRS ? ACT_CLAMPED_SWISH : ACT_RELU_SQUARED>(a, acc, 0, m, n); break;
  }
}

enum { TILE_256_256, TILE_320_192, TILE_128_64, TILE_128_128, TILE_384_160, TILE_256_192, TILE_192_256, TILE_256_128, TILE_64_64, TILE_KINDS };

// A tile's size and the workgroups of it to a CU.
static const struct { int bn, bm, per_cu; } kinds[TILE_KINDS] = {
    {256, 256, 1}, {320, 192, 1}, {128, 64, 2}, {128, 128, 1}, {384, 160, 1}, {256, 192, 1}, {192, 256, 1}, {256, 128, 1}, {64, 64, 3}};

// us of a launch with tiles of a kind: a launch, a full round of the chip (and each 1,000 k-values of it), the last round by the workgroups on its
// fullest CU (and each 1,000 k-values, and those times the share of CUs that have the last of them: fewer of them find memory faster, and
// the chip's power goes further).
struct TileCost { double launch, base, per_k, last[3][3]; };

// ... of gate/up.  Tiles by small waves: fitted to 5,534 sizes of 65 to 1,200 rows, 1,024 to 38,000 weight rows, 128 to 4,096 k-values, off by 9 to 10 %
// in the mean square.
static const TileCost pairs_cost[TILE_KINDS] = {
    {3.07, 9.00, 22.71, {{8.66, 15.99, 5.92}}}, {2.39, 9.30, 21.06, {{8.14, 14.48, 4.28}}},
    {2.92, 2.70, 15.15, {{1.44, 5.26, 3.15}, {1.97, 13.46, 3.98}}}, {1.96, 4.47, 11.42, {{4.08, 7.21, 4.81}}},
    {3.16, 8.88, 22.56, {{7.07, 14.47, 5.78}}}, {2.32, 7.33, 17.34, {{6.39, 12.35, 4.09}}},
    {2.81, 7.66, 16.78, {{5.97, 11.85, 4.51}}}, {2.82, 5.06, 14.36, {{4.16, 9.91, 4.28}}},
    {3.64, 2.14, 13.25, {{0.67, 3.48, 1.61}, {0.96, 7.60, 2.26}, {1.19, 12.75, 2.54}}}};

// ... of the partial sums of a slice (380 sizes of 896 to 20,000 k-values in 1 to 8 slices: off by 5 to 7 % in the mean square; 160 more of cold
// weights: 6 to 7.5 %, tiles of 256 x 128, which have got three slots since, 9.7 %, of which 4 % too long; the choice is 1.0 % off the best in the mean,
// 0.7 % with those fitted again).  Tiles by small waves: 51,415 products of 8,424 sizes of 65 to 1,200 rows, 256 to 8,192 weight rows, 256 to 19,000
// k-values in 1 to 16 slices, 11 to 12 %.
static const TileCost sums_cost[TILE_KINDS] = {
    {1.71, 9.86, 22.96, {{10.23, 15.63, 6.15}}}, {3.43, 8.36, 21.49, {{8.44, 15.09, 4.84}}}, {}, {1.87, 4.35, 11.28, {{2.98, 7.07, 5.83}}},
    {2.80, 7.93, 22.05, {{9.30, 15.29, 4.32}}}, {2.78, 6.62, 18.46, {{7.16, 11.93, 5.03}}}, {1.58, 6.75, 18.74, {{7.87, 11.78, 5.63}}},
    {1.86, 4.34, 15.21, {{5.42, 10.92, 3.72}}}, {3.05, 2.46, 13.31, {{0.21, 3.68, 1.72}, {1.07, 7.25, 2.71}, {1.90, 12.21, 2.60}}}};

static double tile_us(int kind, const TileCost* costs, int M, int N, int slices, int slice_k) {
  const auto& k = kinds[kind];
  const TileCost& c = costs[kind];
  const long long tiles = (long long)((N + k.bn - 1) / k.bn) * ((M + k.bm - 1) / k.bm) * slices, per = (tiles + 7) / 8, round = 32 * k.per_cu;      // (of an XCD)
  const int rest = (int)(per % round), fullest = (rest + 31) / 32;
  const double kk = slice_k / 1000.0;
  double us = c.launch + (double)(per / round) * (c.base + c.per_k * kk);
  if (rest > 0) {
    const double* last = c.last[fullest - 1];
    us += last[0] + kk * (last[1] + last[2] * (rest - 32 * (fullest - 1)) / 32.0);
  }
  return us;
}

static bool small_waves(int kind) { return kind == TILE_128_64 || kind == TILE_128_128 || kind == TILE_64_64; }

static int choose_tile(int M, int N, int K, int out) {
  int best = 0;
  for (int i = 1; i < TILE_KINDS; ++i)
    if (!(out == OUT_ACT && i == TILE_128_64) && tile_us(i, pairs_cost, M, N, 1, K) < tile_us(best, pairs_cost, M, N, 1, K)) best = i;
  return best;
}

// ... and what the reader of the sums pays for every slice after the first
static double sums_us(int kind, int M, int N, int slices, int slice_k) {
  return tile_us(kind, sums_cost, M, N, slices, slice_k) + (slices > 1 ? 0.5 + 1.2e-6 * (double)M * (double)N * (slices - 1) : 0.0);
}

#define SUMS_MIN_ROWS 257
#define SUMS_MIN_N 896          // (lower weights were not measured)
#define SUMS_MIN_K 8192
#define SMALL_MIN_ROWS 129
#define SMALL_MIN_K 896
#define SMALL_MOST 4.0e9        // M N K
#define CAPTURED_MIN_K 3000
#define CAPTURED_LEAST 2.5e9
#define SUMS_MAX_SLICES 8
#define SUMS_MAX_BYTES (512ll << 20)      // of partial sums

// Whether the product of M rows with a weight [N, K], whose reader adds partial sums, is faster here than by the library, by which
// tile and in how many slices: slices << 8 | tile (1 slice: the plain product in bfloat16), 0: it is not.  The library's time over
// this one's, with the norm that adds the sums (100 sizes drawn over 129 to 8,192 rows, 896 to 8,192 weight rows, 8,192 to 20,000
// k-values and 40 of four models' down; geometric mean and worst), by the number of tiles of 256 x 256:
//   up to 128 tiles (the library takes slices of K): 257 to 600 rows 1.30 and 0.88, more 1.20 and 0.90, up to 256 rows 1.14 and 0.68; where
//   the library's slices fill a round to 85 % or more 1.1 and, as 2,048 rows of 3,584 x 18,944 behind other products, 0.96.  (And the batched
//   product costs the host 15 us more: 24 arriving requests at the 3B shape 244.8 -> 234.8 ms from 257 rows on, 239.8 from 800.)
//   129 to 256 tiles, which are one round of the library's: 0.94     more, whose last round is at most 85 % full on the whole: 1.22 and
//   0.81, fuller ones 0.97            weights of 4,096 to 8,192 k-values, of multiples of 512 rows: 0.94
// Small products come here for the host's sake: the library's choice of a kernel and launch take it 26 us a call (the batched product
// 40), this one's 8, and steps that mix portions with decoding are run launch by launch.  On the GPU they take longer here, 1.1 to 1.7 x with the
// norm (150 rows of 1,536 x 1,536 9.3 there and 15.4 here, 692 of 1,920 x 1,024 14.5 and 21.8, 520 of 2,560 x 2,048 19.1 and 23.5; from about
// M N K = 2.5e9 about as long), so a step gains where the host is its longer side and loses where the GPU is, which no size of one product
// tells.  Whole steps of one prompt, 160 to 1,200 tokens by sixteen models, the library's time over this one's: 1.074 in the mean (24 layers of
// 896 1.17 to 1.41; 28 of 1,536 1.44 at 160 tokens, 1.17 at 520, 0.98 from 900 on; 36 of 2,048 1.32 at 160, 1.08 at 420, 0.98 at 520 and 600;
// eight layers of 1,024 or 2,048 with recurrences or experts 0.98 to 1.24), seven of 128 below 0.99, the worst 0.977.  A line at 2e9 for fewer than
// 3,000 k-values spares three of them and loses up to 8 % at eight layers of 1,024 and 2,048: 1.068 in the mean.
// `captured`: a step that is being captured costs the host nothing when it is replayed, and the library's product is not cut there.  Small
// ones then come here only where the GPU gains: 15 of 16 sizes from CAPTURED_MIN_K and CAPTURED_LEAST on (1.16 in the mean; 150 rows of
// 2,048 x 11,008 33.2 there and 28.6 here, 252 of 2,320 x 4,416 28.0 and 20.7), 22 of 99 shallower or smaller ones (0.83).  A decode step of 160
// requests at the layers of 896, 1,536 and 2,048 above: 1.93, 2.96 and 4.41 ms where all come here, 4.63 at 2,048 where none do, now 1.87, 2.86
// and 4.35.
// `library_slices`: the slices that the library would take.
extern "C" int ifx_gemm_tiles_sums_plan(int M, int N, int K, int library_slices, int captured) {
  if (N < SUMS_MIN_N || K > 1 << 20 || N > 1 << 20 || N % 8 || K % 8) return 0;
  const double size = (double)M * N * K;
  const bool small = size <= SMALL_MOST && M >= SMALL_MIN_ROWS && (captured ? K >= CAPTURED_MIN_K && size >= CAPTURED_LEAST : K >= SMALL_MIN_K);
  if (!small) {
    if (M < SUMS_MIN_ROWS || K < SUMS_MIN_K) return 0;
    const long long tiles = (long long)((N + 255) / 256) * ((M + 255) / 256), library = tiles * library_slices;
    if ((tiles > 128 && tiles <= 256) || library >= 0.85 * 256 * ((library + 255) / 256)) return 0;
  }
  int best = 0;
  double least = 0;
  for (int s = 1; s <= SUMS_MAX_SLICES; ++s) {
    const int slice_k = ((K + s - 1) / s + 63) / 64 * 64;
    if ((K + slice_k - 1) / slice_k != s || (s > 1 && (long long)s * M * N * 4 > SUMS_MAX_BYTES)) continue;
    for (int kind = 0; kind < TILE_KINDS; ++kind) {
      if (small_waves(kind)) continue;
      const double us = sums_us(kind, M, N, s, slice_k);
      if (best == 0 || us < least) best = s << 8 | kind, least = us;
    }
  }
  return best;
}

// The same for a model's weights and 65 to 2,048 rows (few_tiles_plan in ops.py has the limits and the lines), with tiles by small waves, too: slices (1 without `keep`: the
// plain product) << 8 | tile.
#define FEW_MAX_SLICES 16
extern "C" int ifx_gemm_tiles_few_plan(int M, int N, int K, int keep) {
  int best = 0;
  double least = 0;
  for (int s = 1; s <= (keep ? FEW_MAX_SLICES : 1); ++s) {
    const int slice_k = ((K + s - 1) / s + 63) / 64 * 64;
    if ((K + slice_k - 1) / slice_k != s || (s > 1 && (slice_k < 128 || (long long)s * M * N * 4 > SUMS_MAX_BYTES))) continue;
    for (int kind = 0; kind < TILE_KINDS; ++kind) {
      if (kind == TILE_128_64) continue;
      const double us = sums_us(kind, M, N, s, slice_k);
      if (best == 0 || us < least) best = s << 8 | kind, least = us;
    }
  }
  return best;
}

template <int FN, int FM>
static void launch_waves(const TilesArgs& a, int out, hipStream_t s) {
  typedef WaveTiles<FN, FM> P;
  const int tiles = ((a.N + P::BN - 1) / P::BN) * ((a.M + P::BM - 1) / P::BM) * a.slices, blocks = tiles < 256 ? (tiles + 7) / 8 * 8 : 256;
  if (out == OUT_PAIRS) hipLaunchKernelGGL((tiles_kernel<FN, FM, OUT_PAIRS>), dim3(blocks), dim3(256), 0, s, a);
  else if (out == OUT_ACT) hipLaunchKernelGGL((tiles_kernel<FN, FM, OUT_ACT>), dim3(blocks), dim3(256), 0, s, a);
  else hipLaunchKernelGGL((tiles_kernel<FN, FM, OUT_SUMS>), dim3(blocks), dim3(256), 0, s, a);
}

template <int BN, int BM, int WN, int WM, int PER_CU>
static void launch_small(const TilesArgs& a, int out, hipStream_t s) {
  const dim3 blocks(((a.N + BN - 1) / BN * ((a.M + BM - 1) / BM) * a.slices + 7) / 8 * 8), threads(64 * (BN / WN) * (BM / WM));
  if (out == OUT_PAIRS) hipLaunchKernelGGL((small_kernel<BN, BM, WN, WM, PER_CU, OUT_PAIRS>), blocks, threads, 0, s, a);
  if constexpr (BN == BM) {
    if (out == OUT_ACT) hipLaunchKernelGGL((small_kernel<BN, BM, WN, WM, PER_CU, OUT_ACT>), blocks, threads, 0, s, a);
    else if (out == OUT_SUMS) hipLaunchKernelGGL((small_kernel<BN, BM, WN, WM, PER_CU, OUT_SUMS>), blocks, threads, 0, s, a);
  }
}

static void launch_kind(const TilesArgs& a, int kind, int out, hipStream_t s) {
  switch (kind) {
    case TILE_256_256: launch_waves<8, 8>(a, out, s); break;
    case TILE_320_192: launch_waves<10, 6>(a, out, s); break;
    case TILE_128_64: launch_small<128, 64, 32, 32, 2>(a, out, s); break;
    case TILE_128_128: launch_small<128, 128, 64, 32, 1>(a, out, s); break;
    case TILE_64_64: launch_small<64, 64, 32, 32, 3>(a, out, s); break;
    case TILE_384_160: launch_waves<12, 5>(a, out, s); break;
    case TILE_256_192: launch_waves<8, 6>(a, out, s); break;
    case TILE_192_256: launch_waves<6, 8>(a, out, s); break;
    case TILE_256_128: launch_waves<8, 4>(a, out, s); break;
  }
}

// x, w, with OUT_ACT the result: on 16 bytes.  tile: one of the kinds above, or -1 for the one that choose_tile takes.
// OUT_ACT also takes ACT_NONE: the plain product.
extern "C" int ifx_gemm_tiles(const void* x, const void* w, void* result, int M, int N, int K, int out, int act, float limit, int tile, void* stream) {
  IFX_REQUIRE(out == OUT_PAIRS || out == OUT_ACT, "gemm_tiles: result %d", out);
  IFX_REQUIRE(M >= 0 && N > 0 && N % (out == OUT_PAIRS ? 4 : 2) == 0 && K > 0 && K % 8 == 0 && K <= 1 << 20 && N <= 1 << 22,
              "gemm_tiles: N=%d must be a multiple of %d, K=%d of 8", N, out == OUT_PAIRS ? 4 : 2, K);
  if (out == OUT_PAIRS)
    IFX_REQUIRE(act == ACT_SILU || act == ACT_GELU_TANH || (act == ACT_CLAMPED_SWISH && limit > 0.f), "gated activation: unknown kind %d (limit %g)", act, (double)limit);
  else
    IFX_REQUIRE(act == ACT_SILU || act == ACT_GELU_TANH || act == ACT_RELU_SQUARED || act == ACT_NONE, "activation: unknown kind %d", act);
  IFX_REQUIRE(((size_t)x | (size_t)w | (size_t)result) % 16 == 0, "gemm_tiles: x, the weight and the result must lie on 16 bytes");
  if (M == 0) return 0;
  const TilesArgs a{(const bf16_t*)x, (const bf16_t*)w, result, M, N, K, act, limit, 1, K};
  const int kind = tile < 0 ? choose_tile(M, N, K, out) : tile;
  IFX_REQUIRE(kind < TILE_KINDS && !(out == OUT_ACT && kind == TILE_128_64), "gemm_tiles: tile %d", tile);
  launch_kind(a, kind, out, (hipStream_t)stream);
  IFX_LAUNCH_CHECK();
}

// parts [slices][M][N] in float: x times w transposed over slices of slice_k values of K (a multiple of 64); x, w, parts on 16 bytes
extern "C" int ifx_gemm_tiles_sums(const void* x, const void* w, float* parts, int M, int N, int K, int slices, int slice_k, int tile, void* stream) {
  IFX_REQUIRE(M >= 0 && N > 0 && N % 4 == 0 && K > 0 && K % 8 == 0 && K <= 1 << 20 && N <= 1 << 20, "gemm_tiles_sums: N=%d must be a multiple of 4, K=%d of 8", N, K);
  IFX_REQUIRE(slices > 0 && slice_k > 0 && slice_k % 64 == 0 && (long long)slices * slice_k >= K && (long long)(slices - 1) * slice_k < K,
              "gemm_tiles_sums: %d slices of %d values of K=%d", slices, slice_k, K);
  IFX_REQUIRE(((size_t)x | (size_t)w | (size_t)parts) % 16 == 0, "gemm_tiles_sums: x, the weight and the result must lie on 16 bytes");
  IFX_REQUIRE(tile >= 0 && tile < TILE_KINDS && tile != TILE_128_64, "gemm_tiles_sums: tile %d", tile);
  if (M == 0) return 0;
  const TilesArgs a{(const bf16_t*)x, (const bf16_t*)w, parts, M, N, K, ACT_NONE, 0.f, slices, slice_k};
  launch_kind(a, tile, OUT_SUMS, (hipStream_t)stream);
  IFX_LAUNCH_CHECK();
}
