// The inner loop of a product of many rows on the matrix cores (bfloat16 in, float sums): C[n][m] = sum_k W[n][k] X[m][k] for a
// tile of BN weight rows and BM rows of x, by (BN / WN) (BM / WM) waves that hold WN x WM sums each.
//
// Steps of 64 k-values of both operands are staged in LDS by loads that go there directly (no registers, no instructions to
// store them; rows beyond the operands' ends arrive as zeros), STAGES stages in turn.  What bounds it is LDS: a step's
// matrix instructions take 2 BN BM 64 / 4,096 cycles of a CU, its reads from LDS (WN + WM) 128 bytes a wave at 128 bytes a
// cycle, and the direct loads' writes (BN + BM) 128 bytes besides.  So the loop is software-pipelined by half steps: the
// fragments of the second half are read while the first half is multiplied; then the step's slot is free, the loads of
// the step after next (STAGES steps on) go out to it, and the next step's first half is read while the second half is multiplied.  Fetch
// and wait thus stand a whole step apart, and the only wait of a step is the barrier in its middle.
//
// A row of x is 128 bytes in LDS, 8 pieces of 16; piece p of row r lies at p ^ (r & 7) ^ (r >> 3 & 1), so that the 16 rows a
// fragment takes a piece of meet every bank evenly.  Rows of W lie likewise, or, with TILED, as the tiles of
// ifx_tile_weights (16 rows x 32 k-values, 1 KB), which are a wave's fragments in the order of its lanes.
//
// Sums run over k in ascending order, 32 k-values to an instruction, whatever the tile: an element of C does not depend on
// BN, BM or what shares its tile.
#pragma once
#include "common.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 tile_bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float tile_floatx4;
typedef unsigned int tile_uintx4 __attribute__((ext_vector_type(4)));

// a buffer of `bytes` (< 2^31 - 64) from base on, the same in all lanes: loads beyond its end give zeros
__device__ __forceinline__ tile_uintx4 tile_buffer(const void* base, unsigned bytes) {
  const unsigned long long b = (unsigned long long)base;
  tile_uintx4 r;
  r[0] = __builtin_amdgcn_readfirstlane((unsigned)b);
  r[1] = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32) & 0xffffu);
  r[2] = __builtin_amdgcn_readfirstlane(bytes);
  r[3] = 0x00020000u;                       // raw 32-bit data format of gfx9
  return r;
}

#define TILE_NO_ROW 0x7fffffff              // an offset beyond every buffer

__device__ __forceinline__ void tile_direct_load(const tile_uintx4& buffer, int offset, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" : : "s"(lds_addr), "v"(offset), "s"(buffer) : "memory", "m0");
}

// the last N direct loads may still be on their way; everything this wave read from LDS has arrived; all waves meet
template <int N>
__device__ __forceinline__ void tile_meet() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N) : "memory");
}

template <int BN, int BM, int WN, int WM, bool TILED, int STAGES = 2>
struct ProductTiles {
  static constexpr int ROW = 128, WAVES = (BN / WN) * (BM / WM), THREADS = 64 * WAVES;
  static constexpr int W_BYTES = BN * ROW, STAGE = (BN + BM) * ROW, LDS = STAGES * STAGE;
  static constexpr int FN = WN / 16, FM = WM / 16;      // this wave's fragments
  static constexpr int LW = BN / 8 / WAVES, LX = BM / 8 / WAVES;      // direct loads of a wave and a step (1 KB each)
  static_assert(BN % (8 * WAVES) == 0 && BM % (8 * WAVES) == 0 && BN % WN == 0 && BM % WM == 0, "tiles");

  // where in C this wave's sums stand: acc[a][b][r] is weight row wn() + 16 a + 4 (lane / 16) + r, row wm() + 16 b + lane % 16
  static __device__ __forceinline__ int wave() { return __builtin_amdgcn_readfirstlane(threadIdx.x / 64); }
  static __device__ __forceinline__ int wn() { return wave() % (BN / WN) * WN; }
  static __device__ __forceinline__ int wm() { return wave() / (BN / WN) * WM; }

  // w: the tile's BN weight rows of K values each (TILED: from the tile's first row tile on, k_tiles tiles of 32 k-values to
  // a row tile, an even number); x: row m of the tile starts at byte x_offset(m) (TILE_NO_ROW: zeros).  K a multiple of 8; rows of
  // W (not TILED) w_pitch values apart.
  template <class XOffset>
  static __device__ __forceinline__ void run(unsigned char* lds, const tile_uintx4& w, const tile_uintx4& x, int K, int w_pitch, XOffset x_offset,
                                             tile_floatx4 (&acc)[FN][FM]) {
    const int wid = wave(), lane = threadIdx.x % 64, col = lane % 16, g = lane / 16;
    const unsigned base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)lds;
    auto place = [](int row) { return (row & 7) ^ ((row >> 3) & 1); };
    const int steps = (K + 63) / 64;
    int wo[LW], wk[LW], xo[LX], xk[LX];
#pragma unroll
    for (int i = 0; i < LW; ++i) {
      const int j = wid * LW + i, row = 8 * j + lane / 8;
      wk[i] = TILED ? 0 : 8 * (lane % 8 ^ place(row));
      wo[i] = TILED ? (j / 2) * steps * 2048 + j % 2 * 1024 + lane * 16 : row * w_pitch * 2 + wk[i] * 2;
    }
#pragma unroll
    for (int i = 0; i < LX; ++i) {
      const int row = (wid * LX + i) * 8 + lane / 8, at = x_offset(row);
      xk[i] = at == TILE_NO_ROW ? K : 8 * (lane % 8 ^ place(row));          // (K: at no step within the row)
      xo[i] = at == TILE_NO_ROW ? 0 : at + xk[i] * 2;
    }
    auto issue = [&](int s, int slot) {
      const int k0 = 64 * s;
      const unsigned to = base + slot * STAGE;
#pragma unroll
      for (int i = 0; i < LW; ++i)
        tile_direct_load(w, k0 + wk[i] < K ? wo[i] + s * (TILED ? 2048 : 128) : TILE_NO_ROW, to + (wid * LW + i) * 1024);
#pragma unroll
      for (int i = 0; i < LX; ++i)
        tile_direct_load(x, k0 + xk[i] < K ? xo[i] + s * 128 : TILE_NO_ROW, to + W_BYTES + (wid * LX + i) * 1024);
    };
    int wr[2], xr[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int at = col * ROW + (((4 * h + g) ^ place(col)) * 16);
      wr[h] = TILED ? wn() * ROW + h * 1024 + lane * 16 : wn() * ROW + at;
      xr[h] = W_BYTES + wm() * ROW + at;
    }
    tile_bf16x8 wf[2][FN], xf[2][FM];
    auto read = [&](int slot, int h) {
      const unsigned char* st = lds + slot * STAGE;
#pragma unroll
      for (int b = 0; b < FM; ++b) xf[h][b] = *(const tile_bf16x8*)(st + xr[h] + b * 16 * ROW);
#pragma unroll
      for (int a = 0; a < FN; ++a) wf[h][a] = *(const tile_bf16x8*)(st + wr[h] + a * 16 * ROW);
    };
    auto multiply = [&](int h) {
#pragma unroll
      for (int a = 0; a < FN; ++a)
#pragma unroll
        for (int b = 0; b < FM; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h][a], xf[h][b], acc[a][b], 0, 0, 0);
      // the next half's reads spread among this half's products
      constexpr int R = FN + FM, PER = FN * FM / R, REST = FN * FM - R * PER;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, PER, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, REST > 0 ? REST : 1, 0);
    };
#pragma unroll
    for (int a = 0; a < FN; ++a)
#pragma unroll
      for (int b = 0; b < FM; ++b) acc[a][b] = tile_floatx4{0.f, 0.f, 0.f, 0.f};
    __builtin_amdgcn_s_waitcnt(0);
#pragma unroll
    for (int s = 0; s < STAGES; ++s) issue(s, s);
    tile_meet<(STAGES - 1) * (LW + LX)>();
    read(0, 0);
    int slot = 0;
    for (int s = 0; s < steps; ++s) {
      const int next = STAGES == 2 ? slot ^ 1 : slot == STAGES - 1 ? 0 : slot + 1;
      read(slot, 1);
      multiply(0);
      tile_meet<(STAGES - 2) * (LW + LX)>();
      issue(s + STAGES, slot);
      read(next, 0);
      multiply(1);
      slot = next;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
};

// The tile of a workgroup when `total` tiles stand in groups of `group` tiles of x by all nt tiles of W, the tile of x running
// fastest within a group: workgroup b runs on XCD b % 8, whose L2 so sees a contiguous range of them, a group's tiles of x
// against one tile of W after the other.  False: this workgroup has none.
__device__ __forceinline__ bool product_tile(int nt, int mt, int group, int* tn, int* tm) {
  const int total = nt * mt, per = (total + 7) / 8, id = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if ((int)(blockIdx.x / 8) >= per || id >= total) return false;
  const int first = id / (group * nt) * group, gm = min(group, mt - first), in = id % (group * nt);
  *tm = first + in % gm;
  *tn = in / gm;
  return true;
}
