// Weight-streaming matrix product for 9-64 rows from the tiled copy of W (layout: gemm_bf16.hip), bf16 in, float sums on the matrix
// cores, out bf16 or float:  out[M,N] = x[M,K] * W[N,K]^T.
//
// W is read once, and the rows of x once for every workgroup; what bounds such a product is how much of both a compute unit
// keeps on its way.  A workgroup of four waves owns NTW row tiles of W, all rows of x (MT tiles of 16) and a slice of K, and takes both in
// steps of 128 k-values through a ring of slots in LDS, filled by loads that go there directly: they cost no registers, so the
// ring is as deep as LDS allows (steps of (NTW + MT) 4 KB, 8 to 48; as many as 160 KB hold: three to five, of up to 16 rows eight), and a
// step costs one barrier.  (The product of gemm_wide.hip, whose loads come through registers, takes 16.9 us for the 12 steps of 17,920 x 1,536 at
// 64 rows and this 14.7, which is 55 MB of W at 3.7 TB/s and 44 MB of x from the L2; about 4 us of either are the launch's start and end.
// Which sizes come here: ops.ring_takes, ops.ring_takes_few and ops._ring_in_one_slice, with both sides measured; workgroups and slices:
// ops.ring_plan.)
//
// Rows of x lie in a slot as in product_tiles.h (two halves of 64 k-values, piece p of row r at p ^ (r & 7) ^ (r >> 3 & 1)), row tiles
// of W as they are stored (a k-tile is a wave's fragment in the order of its lanes; of tiles of fewer than 16 rows the lanes of the
// other rows load zeros).  With four tiles of x (33-64 rows) a wave multiplies one of them with all row tiles; with two (17-32
// rows) two waves share one, half of the step's k-tiles each, with one (9-16 rows) all four, a k-tile each, and add their sums through LDS.
//
// Two tiles of 8 rows (weights of up to 2,048 rows) are joined into one of 16 by the loads, half of whose lanes take the one and half the other: alone each would fill half a
// fragment, and half of its slot with zeros, so that the ring held half as much of W.  us at 16 / 32 / 64 rows, of K in slices, each alone / joined (and cut as
// ring_plan now does): 1,536 x 8,960 8.9, 9.2, 11.9 / 7.6, 8.0, 10.3, 1,536 x 1,536 4.6, 4.7, 6.0 / 4.2, 4.2, 5.1, 2,048 x 11,008 12.3, 13.7, 16.1 / 10.3, 11.0, 14.2,
// 1,024 x 4,224 5.5, 5.4, 7.3 / 4.3, 4.8, 6.3, 896 x 896 3.8, 4.0, 4.8 / 3.0, 3.4, 4.0.
//
// With more than one slice of K the slices write float partial sums, added in slice order by whoever reads them.
#include "product_tiles.h"

IFX_DEFINE_LAST_ERROR()

typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
typedef __attribute__((__vector_size__(2 * sizeof(float)))) float floatx2;

struct RingArgs {
  const bf16_t* x;          // [M][K]
  const bf16_t* w;          // the tiled copy
  void* out;                // [M][N] (epi 0) or [M][N / 2]
  float* part;              // [slices][M][N] where there are several
  int M, N, K, n_tiles, tile_rows, steps;      // steps: of 128 k-values, to a slice
  int joined;               // the copy's tiles hold 8 rows, two of which make one of 16 here (n_tiles and tile_rows are of those)
  const int* order;         // tile t of the copy holds the weight's rows 16 order[t] ...; null: in order
};

template <int NTW, int MT>
struct Ring {
  static constexpr int STAGE = (NTW + MT) * 4096, LOADS = NTW + MT;      // bytes of a step; direct loads of a wave and a step
  static constexpr int MOST = MT == 1 ? 8 : 5, SLOTS = 160 * 1024 / STAGE < MOST ? 160 * 1024 / STAGE : MOST;
  static_assert(SLOTS >= 3 && (SLOTS - 2) * LOADS < 64, "ring");
};

__device__ __forceinline__ void ring_load(const tile_uintx4& buffer, int offset, int step_bytes, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               : : "s"(lds_addr), "v"(offset), "s"(buffer), "s"(step_bytes) : "memory", "m0");
}
__device__ __forceinline__ void ring_load_streaming(const tile_uintx4& buffer, int offset, int step_bytes, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
               : : "s"(lds_addr), "v"(offset), "s"(buffer), "s"(step_bytes) : "memory", "m0");
}

__device__ __forceinline__ void store2(float* p, float a, float b) { *(floatx2*)p = floatx2{a, b}; }
__device__ __forceinline__ void store2(bf16_t* p, float a, float b) {
  bf16x2 w;
  w[0] = (__bf16)a; w[1] = (__bf16)b;
  *(bf16x2*)p = w;
}
__device__ __forceinline__ void store4(float* p, const tile_floatx4& v) { *(tile_floatx4*)p = v; }
__device__ __forceinline__ void store4(bf16_t* p, const tile_floatx4& v) {
  bf16x4 w;
#pragma unroll
  for (int r = 0; r < 4; ++r) w[r] = (__bf16)v[r];
  *(bf16x4*)p = w;
}

template <int NTW, int MT, typename TO, int EPI>
__global__ __launch_bounds__(256, 1) void ring_gemm_kernel(RingArgs a) {
  typedef Ring<NTW, MT> R;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[R::SLOTS * R::STAGE];
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, col = lane % 16, g = lane / 16;
  const unsigned base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)lds;
  auto place = [](int row) { return (row & 7) ^ ((row >> 3) & 1); };
  const int k_tiles = (a.K + 63) / 64 * 2, all_steps = (a.K + 127) / 128;
  const int first_tile = blockIdx.x * NTW, s0 = blockIdx.y * a.steps, steps = min(a.steps, all_steps - s0);
  const int k_tile_bytes = 64 * (a.joined ? 8 : a.tile_rows), tile_bytes = (a.joined ? 2 : 1) * k_tiles * k_tile_bytes;
  // (of joined tiles the last may have one half only: the buffer ends with the copy)
  const int held_tiles = a.joined ? min(2 * NTW, (a.N + 7) / 8 - 2 * first_tile) : min(NTW, a.n_tiles - first_tile);
  const tile_uintx4 wb = tile_buffer(a.w + (size_t)first_tile * (tile_bytes / 2), (unsigned)held_tiles * (unsigned)k_tiles * k_tile_bytes);
  const tile_uintx4 xb = tile_buffer(a.x, (unsigned)a.M * (unsigned)a.K * 2u);
  // this wave loads k-tile wid of every row tile's four, and MT runs of eight rows of x
  const int w_lane = a.joined ? col / 8 * (k_tiles * k_tile_bytes) + (8 * g + col % 8) * 16 : col < a.tile_rows ? (a.tile_rows * g + col) * 16 : TILE_NO_ROW;
  int xo[MT], xk[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int q = wid * MT + i, h = q / (2 * MT), row = q % (2 * MT) * 8 + lane / 8;
    xk[i] = 64 * h + 8 * (lane % 8 ^ place(row));
    xo[i] = row < a.M ? row * a.K * 2 + xk[i] * 2 : TILE_NO_ROW;
  }
  auto issue = [&](int s, int slot) {          // s: counted from the slice's first
    const unsigned to = base + slot * R::STAGE;
    const int at = s0 + s;
    tile_uintx4 w = wb, x = xb;
    if (s >= steps || at * 4 + wid >= k_tiles) w[2] = 0;      // (nothing, as zeros: the number of loads stays the same)
    if (s >= steps) x[2] = 0;
#pragma unroll
    for (int j = 0; j < NTW; ++j)
      ring_load_streaming(w, w_lane == TILE_NO_ROW ? TILE_NO_ROW : w_lane + j * tile_bytes, (at * 4 + wid) * k_tile_bytes, to + (j * 4 + wid) * 1024);
    const bool last = at * 128 + 128 > a.K;
#pragma unroll
    for (int i = 0; i < MT; ++i)
      ring_load(x, last && at * 128 + xk[i] >= a.K ? TILE_NO_ROW : xo[i], at * 256, to + NTW * 4096 + (wid * MT + i) * 1024);
  };
  constexpr int KT0_STEP = MT;          // k-tiles of a step to a wave
  const int m_tile = wid % MT, kt0 = wid / MT * MT;
  tile_floatx4 acc[NTW];
#pragma unroll
  for (int j = 0; j < NTW; ++j) acc[j] = tile_floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < R::SLOTS - 1; ++s) issue(s, s);
  int slot = 0;
  for (int s = 0; s < steps; ++s) {
    // step s is there; every wave has read step s - 1 (the wait for its LDS reads is in there: the products that take them are no memory
    // operations and could be moved behind the barrier)
    tile_meet<(R::SLOTS - 2) * R::LOADS>();
    issue(s + R::SLOTS - 1, slot == 0 ? R::SLOTS - 1 : slot - 1);
    const unsigned char* st = lds + slot * R::STAGE;
    tile_bf16x8 wf[KT0_STEP][NTW], xf[KT0_STEP];
#pragma unroll
    for (int i = 0; i < KT0_STEP; ++i) {
      const int kt = kt0 + i;
      xf[i] = *(const tile_bf16x8*)(st + NTW * 4096 + kt / 2 * (MT * 2048) + (16 * m_tile + col) * 128 + ((kt % 2 * 4 + g) ^ place(col)) * 16);
#pragma unroll
      for (int j = 0; j < NTW; ++j) wf[i][j] = *(const tile_bf16x8*)(st + (j * 4 + kt) * 1024 + lane * 16);
    }
    __builtin_amdgcn_sched_barrier(0);          // (all of a step's reads are on their way before its first product)
#pragma unroll
    for (int i = 0; i < KT0_STEP; ++i)
#pragma unroll
      for (int j = 0; j < NTW; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i][j], xf[i], acc[j], 0, 0, 0);
    slot = slot == R::SLOTS - 1 ? 0 : slot + 1;
  }
  tile_meet<0>();          // (the loads beyond the end; all have read the last step)
  if (MT < 4) {
    tile_floatx4* shares = (tile_floatx4*)lds;
    if (wid >= MT)
#pragma unroll
      for (int j = 0; j < NTW; ++j) shares[((wid - MT) * NTW + j) * 64 + lane] = acc[j];
    __syncthreads();
    if (wid >= MT) return;
#pragma unroll
    for (int k = 0; k < 4 / MT - 1; ++k)
#pragma unroll
      for (int j = 0; j < NTW; ++j) acc[j] += shares[((k * MT + wid) * NTW + j) * 64 + lane];
  }
  // acc[j][r] = out[m = 16 m_tile + col][n = tile_rows (row tile of the weight) + 4 g + r], for 4 g + r < tile_rows
  const int m = 16 * m_tile + col, held = min(4, a.tile_rows - 4 * g);      // (held: even, may be <= 0)
  if (m >= a.M) return;
#pragma unroll
  for (int j = 0; j < NTW; ++j) {
    const int tile = first_tile + j;
    if (tile >= a.n_tiles) continue;
    const int n0 = a.tile_rows * (a.order ? a.order[tile] : tile) + 4 * g;
    const bool whole = held == 4 && n0 + 3 < a.N && ((a.N | n0) & 3) == 0;
    if (gridDim.y > 1) {
      float* dst = a.part + ((size_t)blockIdx.y * a.M + m) * a.N + n0;
      if (whole) {
        store4(dst, acc[j]);
      } else if (((a.N | n0) & 1) == 0) {
#pragma unroll
        for (int r = 0; r < 4; r += 2)
          if (r < held && n0 + r < a.N) store2(dst + r, acc[j][r], acc[j][r + 1]);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (r < held && n0 + r < a.N) dst[r] = acc[j][r];
      }
    } else if (EPI == 0 || EPI >= 4) {
      if (EPI >= 4)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[j][r] = plain_act(acc[j][r], EPI == 4 ? ACT_RELU_SQUARED : ACT_GELU_TANH);
      TO* dst = (TO*)a.out + (size_t)m * a.N + n0;
      if (whole) {
        store4(dst, acc[j]);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (r < held && n0 + r < a.N) dst[r] = from_f<TO>(acc[j][r]);
      }
    } else {
      TO* dst = (TO*)a.out + (size_t)m * (a.N / 2) + n0 / 2;
      const float v0 = gated_epilogue<EPI>(acc[j][0], acc[j][1]), v1 = gated_epilogue<EPI>(acc[j][2], acc[j][3]);
      if (whole) {
        store2(dst, v0, v1);
      } else {
        if (held > 0 && n0 + 1 < a.N) dst[0] = from_f<TO>(v0);
        if (held > 2 && n0 + 3 < a.N) dst[1] = from_f<TO>(v1);
      }
    }
  }
}

template <int NTW, int MT>
static int launch_ring(const RingArgs& a, int out_dtype, int slices, int epi, hipStream_t s) {
  const dim3 grid((a.n_tiles + NTW - 1) / NTW, slices);
#define GO(TO_, EPI_) hipLaunchKernelGGL((ring_gemm_kernel<NTW, MT, TO_, EPI_>), grid, dim3(256), 0, s, a)
  if (epi == 1) GO(bf16_t, 1);
  else if (epi == 3) GO(bf16_t, 3);
  else if (epi == 4 && MT == 1) GO(bf16_t, (MT == 1 ? 4 : 0));
  else if (epi == 5 && MT == 1) GO(bf16_t, (MT == 1 ? 5 : 0));
  else if (out_dtype == DT_BF16) GO(bf16_t, 0);
  else GO(float, 0);
#undef GO
  IFX_LAUNCH_CHECK();
}

// x [M <= 64, K] times the tiled copy w of W [N, K], transposed, by workgroups of row_tiles (1 to 8) row tiles and `slices` slices of
// `steps` steps of 128 k-values.  epi 1 (3): gate/up rows in turn, out = silu(gate) * up (the tanh form of gelu), bfloat16, one slice.
// With several slices the partial sums are left in part [slices][M][N].
extern "C" int ifx_ring_gemm(const void* x, const void* w, void* out, int out_dtype, float* part, int M, int N, int K, int row_tiles,
                             int slices, int steps, int epi, const int* order, int tile_rows, void* stream) {
  IFX_REQUIRE(M >= 0 && M <= 64 && N > 0 && K > 0 && K % 8 == 0, "ring_gemm: M=%d must be at most 64, K=%d a multiple of 8 (N=%d)", M, K, N);
  IFX_REQUIRE(tile_rows >= 8 && tile_rows <= 16 && tile_rows % 2 == 0 && (tile_rows == 16 || !order), "ring_gemm: %d rows to a tile", tile_rows);
  IFX_REQUIRE(row_tiles >= 1 && row_tiles <= 8 && slices >= 1 && steps >= 1, "ring_gemm: %d row tiles, %d slices of %d steps", row_tiles, slices, steps);
  const int all = (K + 127) / 128;
  IFX_REQUIRE((all + steps - 1) / steps == slices, "ring_gemm: %d steps do not cut into %d slices of %d", all, slices, steps);
  IFX_REQUIRE(epi == 0 || ((epi == 4 || epi == 5) && M <= 16 && !order && slices == 1 && out_dtype == DT_BF16) || ((epi == 1 || epi == 3) && N % 2 == 0 && !order && slices == 1 && out_dtype == DT_BF16), "ring_gemm: epilogue %d with N=%d, %d slices", epi, N, slices);
  IFX_REQUIRE(slices == 1 ? out != nullptr : part != nullptr, "ring_gemm: no result");
  IFX_REQUIRE(out_dtype == DT_BF16 || out_dtype == DT_F32, "ring_gemm: unknown out dtype %d", out_dtype);
  IFX_REQUIRE((size_t)x % 16 == 0, "ring_gemm: x must lie on 16 bytes");
  IFX_REQUIRE((long long)row_tiles * ((K + 63) / 64 * 64) * tile_rows * 2 < (1ll << 31) - 4096 && (long long)M * K * 2 < (1ll << 31) - 4096, "ring_gemm: K=%d is too deep", K);
  if (M == 0) return 0;
  const int joined = tile_rows == 8 && slices > 1 && row_tiles % 2 == 0, rows = joined ? 16 : tile_rows;
  if (joined) row_tiles /= 2;
  const RingArgs a{(const bf16_t*)x, (const bf16_t*)w, out, part, M, N, K, (N + rows - 1) / rows, rows, steps, joined, order};
  hipStream_t s = (hipStream_t)stream;
#define CASE(NTW_) case NTW_: return M <= 16 ? launch_ring<NTW_, 1>(a, out_dtype, slices, epi, s) : M <= 32 ? launch_ring<NTW_, 2>(a, out_dtype, slices, epi, s) : launch_ring<NTW_, 4>(a, out_dtype, slices, epi, s)
  switch (row_tiles) {
    CASE(1); CASE(2); CASE(3); CASE(4); CASE(5); CASE(6); CASE(7); CASE(8);
  }
#undef CASE
  IFX_FAIL("ring_gemm: %d row tiles", row_tiles);
}
