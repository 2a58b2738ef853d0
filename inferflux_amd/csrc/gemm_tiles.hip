// out[M][N / 2] = act(x Wg^T) * (x Wu^T) for many rows, on the matrix cores (bfloat16 in and out, float sums), W [N][K] with
// the rows of Wg and Wu in turn: a lane holds a gate and its up, and the activation is the product's epilogue, from the sums
// as they are.  The library's product followed by a launch for the activation writes the N columns and reads them back (2,048
// rows of 37,888 columns: 233 MB, 40 us of 545) and rounds them to bfloat16 in between.
//
// The inner loop is product_tiles.h; what is chosen here is the tile, and whether the library's product and the activation's
// launch would be faster.  Large tiles read less of LDS for their products but there are few of them, and the last of the
// rounds that they take on 256 CUs may be nearly empty; so choose_tile() takes the tile whose rounds are estimated to take least,
// from what a round of each was measured to take (see `kinds`; estimates are off by 7 % in the mean square, the choice is
// within 4 % of the best tile at nine sizes of ten).
// (256 x 192, 256 x 128 and 384 x 128 with one workgroup to a CU were never the fastest by more than 2 %; 256 x 256 by four
// waves of 128 x 128, which read a third less of LDS, took 700 us where eight waves take 475: one wave to a SIMD does not
// hide the loop's own latencies.)
//
// The library runs a round of its 256 x 256 tiles in 0.75 to 0.8 of the time of one here (K 1,536 to 8,192: 1,300 to 1,480 TFLOP/s
// where its rounds are full, 1,000 to 1,200 here), so what this product has to win is the activation's two trips to memory and
// the launch, which weigh less the deeper the weight.  By K (ten weights of 1,024 to 32,768 rows, 300 to 16,384 rows of x; a replayed
// graph, geometric mean and worst of library and activation / this): 64 1.66 x and 1.11; 256 1.52, 1.04; 512 1.40, 0.99; 640 1.21, 0.87;
// 768 1.15, 0.82; 1,024 1.10, 0.78; 1,280 1.01, 0.71; 1,792 to 8,192 0.97, 0.65.  Beyond about 1,500 k-values the library is faster by a
// fifth where the kernel it chooses fits the size and slower by as much where it does not (2,048 rows: N 20,480, K 3,584 354 : 283 us;
// 37,888 x 3,584 563 : 510; 35,840 x 3,072 406 : 430; 40,960 x 2,560 368 : 418; 49,152 x 3,584 563 : 655), and no property of the
// size tells which.  So the product is taken up to PAIRS_MAX_K k-values, where the estimate of the library's time (its rounds of
// 256 x 256, 256 x 128 or 128 x 128, whichever least, off by 10 % in the mean) is at least 1.2 times this one's.  Of 2,300 sizes of
// up to 1,536 k-values that rule takes 1,124: mean 1.41 x, worst 0.95 x, ten below 1; of other sizes, drawn at random, 768: mean
// 1.80 x, worst 0.88 x (at launches of 6 us, where the launch that it saves weighs more than the 0.7 us).
#include "product_tiles.h"

IFX_DEFINE_LAST_ERROR()

typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;

struct PairsArgs {
  const bf16_t* x;          // [M][K]
  const bf16_t* w;          // [N][K]
  bf16_t* out;              // [M][N / 2]
  int M, N, K, act;
  float limit;
};

template <int BN, int BM, int WN, int WM, int PER_CU>
__global__ __launch_bounds__(64 * (BN / WN) * (BM / WM), 2 * PER_CU) void pairs_kernel(PairsArgs a) {
  typedef ProductTiles<BN, BM, WN, WM, false> P;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[P::LDS];
  int tn, tm;
  if (!product_tile((a.N + BN - 1) / BN, (a.M + BM - 1) / BM, 4, &tn, &tm)) return;
  const int n0 = tn * BN, m0 = tm * BM, rows = min(BN, a.N - n0), count = min(BM, a.M - m0);
  const tile_uintx4 w = tile_buffer(a.w + (size_t)n0 * a.K, (unsigned)rows * (unsigned)a.K * 2u);
  const tile_uintx4 x = tile_buffer(a.x + (size_t)m0 * a.K, (unsigned)count * (unsigned)a.K * 2u);
  tile_floatx4 acc[P::FN][P::FM];
  P::run(lds, w, x, a.K, [&](int i) { return i * a.K * 2; }, acc);
  const int lane = threadIdx.x % 64, g = lane / 16;
#pragma unroll
  for (int b = 0; b < P::FM; ++b) {
    const int m = m0 + P::wm() + 16 * b + lane % 16;
    if (m >= a.M) continue;
    bf16_t* out = a.out + (size_t)m * (a.N / 2);
#pragma unroll
    for (int c = 0; c < P::FN; ++c) {
      const int n = n0 + P::wn() + 16 * c + 4 * g;
      if (n >= a.N) continue;
      bf16x2 y;
      y[0] = (__bf16)gated_act(acc[c][b][0], acc[c][b][1], a.act, a.limit);
      y[1] = (__bf16)gated_act(acc[c][b][2], acc[c][b][3], a.act, a.limit);
      *(bf16x2*)(out + n / 2) = y;
    }
  }
}

enum { TILE_256_256, TILE_320_192, TILE_192_128, TILE_128_128, TILE_KINDS };

template <int BN, int BM, int WN, int WM, int PER_CU>
static void launch_pairs(const PairsArgs& a, hipStream_t s) {
  const int blocks = ((a.N + BN - 1) / BN * ((a.M + BM - 1) / BM) + 7) / 8 * 8;
  hipLaunchKernelGGL((pairs_kernel<BN, BM, WN, WM, PER_CU>), dim3(blocks), dim3(64 * (BN / WN) * (BM / WM)), 0, s, a);
}

// us of a launch with tiles of a kind: full rounds of 256 CUs (with `per_cu` workgroups each) and the last one
static double tiles_us(int kind, int M, int N, int K) {
  static const struct { int bn, bm, per_cu; double base, per_k, one_base, one_per_k; } kinds[TILE_KINDS] = {
      {256, 256, 1, 13.7, 0.0206, 0, 0}, {320, 192, 1, 13.0, 0.0190, 0, 0},
      {192, 128, 2, 7.6, 0.0189, 5.6, 0.0112}, {128, 128, 2, 5.4, 0.0147, 3.7, 0.0089}};      // (one_: with one workgroup to a CU only)
  const auto& k = kinds[kind];
  const long long tiles = (long long)((N + k.bn - 1) / k.bn) * ((M + k.bm - 1) / k.bm), round = 256 * k.per_cu, rest = tiles % round;
  const double full = k.base + k.per_k * K;
  return 2.0 + (double)(tiles / round) * full + (rest == 0 ? 0.0 : k.per_cu == 2 && rest <= 256 ? k.one_base + k.one_per_k * K : full);
}

static int choose_tile(int M, int N, int K) {
  int best = 0;
  for (int i = 1; i < TILE_KINDS; ++i)
    if (tiles_us(i, M, N, K) < tiles_us(best, M, N, K)) best = i;
  return best;
}

// us of the library's product and the activation's launch
static double library_us(int M, int N, int K) {
  auto rounds = [&](int bn, int bm) { return (double)(((long long)((N + bn - 1) / bn) * ((M + bm - 1) / bm) + 255) / 256); };
  const double product = K * fmin(0.0151 * rounds(256, 256), fmin(0.00984 * rounds(256, 128), 0.0059 * rounds(128, 128)));
  return 7.5 + 1.24e-6 * (double)M * (double)N + product;
}

#define PAIRS_MAX_K 1536
#define PAIRS_MIN_ROWS 129      // fewer rows were not measured (up to 128 are mostly the streaming products')

// whether ifx_gemm_pairs is the faster way for M rows (see above)
extern "C" int ifx_gemm_pairs_wins(int M, int N, int K) {
  return M >= PAIRS_MIN_ROWS && K <= PAIRS_MAX_K && library_us(M, N, K) >= 1.2 * tiles_us(choose_tile(M, N, K), M, N, K);
}

// x, w: on 16 bytes.  tile: one of the kinds above, or -1 for the one that choose_tile takes
extern "C" int ifx_gemm_pairs(const void* x, const void* w, void* out, int M, int N, int K, int act, float limit, int tile, void* stream) {
  IFX_REQUIRE(M >= 0 && N > 0 && N % 4 == 0 && K > 0 && K % 8 == 0 && K <= 1 << 20, "gemm_pairs: N=%d must be a multiple of 4, K=%d of 8", N, K);
  IFX_REQUIRE(act == ACT_SILU || act == ACT_GELU_TANH || (act == ACT_CLAMPED_SWISH && limit > 0.f), "gated activation: unknown kind %d (limit %g)", act, (double)limit);
  IFX_REQUIRE(((size_t)x | (size_t)w) % 16 == 0, "gemm_pairs: x and the weight must lie on 16 bytes");
  if (M == 0) return 0;
  const PairsArgs a{(const bf16_t*)x, (const bf16_t*)w, (bf16_t*)out, M, N, K, act, limit};
  hipStream_t s = (hipStream_t)stream;
  switch (tile < 0 ? choose_tile(M, N, K) : tile) {
    case TILE_256_256: launch_pairs<256, 256, 128, 64, 1>(a, s); break;
    case TILE_320_192: launch_pairs<320, 192, 80, 96, 1>(a, s); break;
    case TILE_192_128: launch_pairs<192, 128, 48, 64, 2>(a, s); break;
    case TILE_128_128: launch_pairs<128, 128, 32, 64, 2>(a, s); break;
    default: IFX_FAIL("gemm_pairs: tile %d", tile);
  }
  IFX_LAUNCH_CHECK();
}
