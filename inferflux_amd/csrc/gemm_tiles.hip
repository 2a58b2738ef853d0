// out[M][N / 2] = act(x Wg^T) * (x Wu^T) for many rows, on the matrix cores (bfloat16 in and out, float sums), W [N][K] with
// the rows of Wg and Wu in turn: a lane holds a gate and its up, and the activation is the product's epilogue, from the sums
// as they are.  The library's product followed by a launch for the activation writes the N columns and reads them back (2,048
// rows of 37,888 columns: 233 MB, 40 us of 545) and rounds them to bfloat16 in between.
//
// The inner loop is product_tiles.h; what is chosen here is the tile.  Large tiles read less of LDS for their products but
// there are few of them, and the last of the rounds that they take on 256 CUs may be nearly empty; so launch() takes the tile
// whose rounds are estimated to take least, from what a round of each was measured to take:
//   256 x 256  one workgroup to a CU, waves of 128 x 64     12 + 0.0232 K us
//   320 x 192  one, 80 x 96                                 10.5 + 0.0215 K
//   192 x 128  two, 48 x 64                                 5.5 + 0.0200 K, 8.8 + 0.0112 K with one to a CU only
//   128 x 128  two, 32 x 64                                 10 + 0.0127 K, 7 + 0.0093 K
// (256 x 192, 256 x 128 and 384 x 128 with one workgroup to a CU were never the fastest by more than 2 %; 256 x 256 by four
// waves of 128 x 128, which read a third less of LDS, took 700 us where eight waves take 475: one wave to a SIMD does not
// hide the loop's own latencies.)
// Measured, library and activation : this, us (weights N x K; 512 / 1,024 / 2,048 / 8,192 rows):
//    9,728 x   896   24 : 19      37 : 29     68 : 53     190 : 167
//   17,920 x 1,536   41 : 39      77 : 63    136 : 118    454 : 461
//   22,016 x 2,048   58 : 55     105 : 102   196 : 178    718 : 674
//   11,264 x 2,048   37 : 33      60 : 51     96 : 98     405 : 362
//   37,888 x 3,584  145 : 188    319 : 288   551 : 481   1792 : 1906
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

// the tile whose rounds on 256 CUs should take least (see above)
static int choose_tile(int M, int N, int K) {
  static const struct { int bn, bm, per_cu; double base, per_k, one_base, one_per_k; } kinds[TILE_KINDS] = {
      {256, 256, 1, 12.0, 0.0232, 0, 0}, {320, 192, 1, 10.5, 0.0215, 0, 0},
      {192, 128, 2, 5.5, 0.0200, 8.8, 0.0112}, {128, 128, 2, 10.0, 0.0127, 7.0, 0.0093}};
  int best = 0;
  double least = 0;
  for (int i = 0; i < TILE_KINDS; ++i) {
    const auto& k = kinds[i];
    const long long tiles = (long long)((N + k.bn - 1) / k.bn) * ((M + k.bm - 1) / k.bm), round = 256 * k.per_cu, rest = tiles % round;
    const double full = k.base + k.per_k * K;
    const double t = (double)(tiles / round) * full + (rest == 0 ? 0.0 : k.per_cu == 2 && rest <= 256 ? k.one_base + k.one_per_k * K : full);
    if (i == 0 || t < least) { best = i; least = t; }
  }
  return best;
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
