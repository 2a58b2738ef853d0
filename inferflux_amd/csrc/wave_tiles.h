// The inner loop of a product of many rows by four large waves (bfloat16 in, float sums): C[n][m] = sum_k W[n][k] X[m][k] for
// a tile of 32 FN weight rows and 32 FM rows of x; each of the workgroup's four waves, one to a SIMD, holds a quarter of the sums.
//
// Steps of 64 k-values of both operands are staged in LDS by loads that go there directly, two slots in turn (three of tiles of 256 x 128), and each step
// is taken in two halves: while one half's fragments are multiplied, the next half's are read.  A step of 256 x 256 is 2,048
// cycles of matrix instructions to a SIMD, and the rest has to stay out of their way:
//   LDS   a wave of 128 x 128 reads 32 KB a step, a third less than two of 128 x 64 (which fill LDS as long as the matrix
//         cores).  Instruction for instruction the loop takes 2,165 cycles a step without its loads, at 1.95 GHz.
//   order with one wave to a SIMD nothing hides a bad order of instructions, so the matrix instructions are volatile assembly
//         and everything between them stays where it is written: reads and loads one by one between them, the step's only
//         barrier in its middle.  (Left to the compiler the same loop took 1.5 times as long.)
//   loads those of a step go out one step (about 1 us) ahead, as far as LDS reaches, which is shorter than a trip to memory
//         under load: 3,050 cycles a step where W comes from memory (2,048 rows x 37,888 x 3,584).  So W's lines are touched two
//         more steps ahead by loads whose values nobody reads, which brings them as far as the L2: 2,480 cycles.  The workgroups that
//         meet the same rows of W share the touches; the last steps touch the next tile's first ones.  x comes from the caches;
//         touching it too costs more than it gives (1.05 x).
//   ends  a workgroup takes one tile after the other and asks for a tile's first steps before it writes the one before
//         it out (12 us a tile without that and with division and expf() in the activation, now 7).
// Tiles of 256 x 128 are half the arithmetic for three quarters of the bytes and wait for loads one step ahead; their three slots reach two
// (260 rows of 37,888 x 3,584 125 -> 107 us, 530 of 2,048 x 11,008 in six slices 34.3 -> 32.3, 300 of 17,920 x 1,536 24.1 -> 22.9).
// Rows of 32 k-values in five slots, which reach twice as far ahead, took 1.05 x the time: half lines cost more requests.
//
// A row is 128 bytes in LDS, 8 pieces of 16; piece p of row r lies at p ^ (r & 7) ^ (r >> 3 & 1), so that the 16 rows a
// fragment takes a piece of meet every bank evenly.  With TILED W comes as the tiles of ifx_tile_weights (16 rows x 32 k-values, 1 KB), which
// lie in LDS as they are: a fragment each, in the order of a wave's lanes.
//
// Sums run over k in ascending order, 32 k-values to an instruction, whatever the tile: an element of C does not depend on
// the tile's size or what shares it.
#pragma once
#include "product_tiles.h"

template <int FN, int FM, bool TILED = false>
struct WaveTiles {
  static constexpr int BN = 32 * FN, BM = 32 * FM, WN = 16 * FN, WM = 16 * FM, THREADS = 256;
  static constexpr int ROW = 128, W_STEP = TILED ? 2048 : ROW, W_BYTES = BN * ROW, STAGE = (BN + BM) * ROW;
  static constexpr int SLOTS = 3 * STAGE + 1024 <= 148 * 1024 ? 3 : 2;
  static constexpr int TOUCHED = SLOTS * STAGE, LDS = SLOTS * STAGE + 1024;      // (the touches' values: 256 bytes a wave)
  static constexpr int READS = FN + FM, LOADS = FN + FM, PRODUCTS = FN * FM, AHEAD = 2;
  static_assert(FN * FM <= 64, "a wave's sums are 256 registers at most");

  int wid, lane, col, g;        // this wave, lane, and the lane's column and k-group in a fragment
  unsigned base;                // the workgroup's LDS
  int wo[FN], xo[FM], touch;      // byte offsets of what this lane loads; its row of W to touch
  tile_uintx4 w, x, next;       // buffers of this tile's rows, and of the next one's W
  int next_steps;               // ... and its steps, 0: there is no next tile
  bool touches;                 // whether this wave touches rows of W

  static __device__ __forceinline__ int place(int row) { return (row & 7) ^ ((row >> 3) & 1); }
  static __device__ __forceinline__ void multiply(tile_floatx4& c, const tile_bf16x8& a, const tile_bf16x8& b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ void load(const tile_uintx4& buffer, int offset, int step_bytes, unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 : : "s"(lds_addr), "v"(offset), "s"(buffer), "s"(step_bytes) : "memory", "m0");
  }
  static __device__ __forceinline__ void load_one(const tile_uintx4& buffer, int offset, int step_bytes, unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
                 : : "s"(lds_addr), "v"(offset), "s"(buffer), "s"(step_bytes) : "memory", "m0");
  }

  // where in C this wave's sums stand: acc[a][b][r] is weight row wn() + 16 a + 4 g + r, row wm() + 16 b + col
  __device__ __forceinline__ int wn() const { return wid % 2 * WN; }
  __device__ __forceinline__ int wm() const { return wid / 2 * WM; }

  __device__ __forceinline__ void init(unsigned char* lds) {
    wid = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    lane = threadIdx.x % 64, col = lane % 16, g = lane / 16;
    base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)lds;
  }

  // Asks for a tile's first steps, a slot each (K a multiple of 8).  wb, xb: buffers that start at the tile's first row of W and
  // x, at the first of the K values; row m of x starts at byte x_offset(m, i), where i is the
  // number of m among the rows that this lane loads, row n of W at n * w_row.
  template <class XOffset>
  __device__ __forceinline__ void begin(const tile_uintx4& wb, const tile_uintx4& xb, int K, int w_row, XOffset x_offset) {
    w = wb, x = xb;
#pragma unroll
    for (int i = 0; i < FN; ++i) {
      const int row = (wid * FN + i) * 8 + lane / 8;
      wo[i] = TILED ? tiles_at(wid * FN + i, K) + 16 * lane : row * w_row + 16 * (lane % 8 ^ place(row));
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int row = (wid * FM + i) * 8 + lane / 8, at = x_offset(row, i);
      xo[i] = at == TILE_NO_ROW ? at : at + 16 * (lane % 8 ^ place(row));
    }
    const int steps = (K + 63) / 64;
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
      if (s == steps - 1 && K % 64 != 0) cut(K);
      if (s < steps) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) issue(i, s, s);
      }
    }
  }
  // rows of W to touch: of a group of `sharers` workgroups that meet the same tile of W this one is `share`
  __device__ __forceinline__ void touch_rows(int share, int sharers, int w_row) {
    const int set = share + sharers * wid;        // of 64 rows
    touches = set < (BN + 63) / 64;
    touch = set * 64 + lane < BN ? (set * 64 + lane) * w_row : TILE_NO_ROW;
  }
  // ... of tiles, all of them by this workgroup: a step's lines of 8 rows, 128 bytes each, lie one after the other
  __device__ __forceinline__ void touch_tiles(int K) {
    const int line = 64 * wid + lane;
    touches = 64 * wid < BN;
    touch = line < BN ? tiles_at(line / 8, K) + 128 * (line % 8) : TILE_NO_ROW;
  }

  // acc = the tile's sums.  All of the workgroup's waves are done with the slots when it returns.
  __device__ __forceinline__ void run(const unsigned char* lds, int K, tile_floatx4 (&acc)[FN][FM]) {
    const int steps = (K + 63) / 64;
    const bool uneven = K % 64 != 0;
    int wr[2], xr[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int at = col * ROW + ((4 * h + g) ^ place(col)) * 16;
      wr[h] = wn() * ROW + (TILED ? 1024 * h + 16 * lane : at);
      xr[h] = W_BYTES + wm() * ROW + at;
    }
    tile_bf16x8 wf[2][FN], xf[2][FM];
    auto read = [&](int i, int slot, int h) {
      const unsigned char* st = lds + slot * STAGE;
      if (i < FM) xf[h][i] = *(const tile_bf16x8*)(st + xr[h] + i * 16 * ROW);
      else wf[h][i - FM] = *(const tile_bf16x8*)(st + wr[h] + (i - FM) * 16 * ROW);
    };
    // the products of half h; between them the other half is read from `from`, and with LOAD step s goes out to slot `to`
    auto half = [&](int h, int from, bool LOAD, int s, int to) {
      int r = 0, l = 0;
#pragma unroll
      for (int p = 0; p < PRODUCTS; ++p) {
        const int a = p / FM, b = (a & 1) ? FM - 1 - p % FM : p % FM;
        multiply(acc[a][b], wf[h][a], xf[h][b]);
        if (r < READS && r * (PRODUCTS - 12) <= (p + 1) * READS) read(r++, from, h ^ 1);
        else if (LOAD && l < LOADS && p % 2 == 1) issue(l++, s, to);
      }
#pragma unroll
      for (; r < READS; ++r) read(r, from, h ^ 1);
      if (LOAD) {
#pragma unroll
        for (; l < LOADS; ++l) issue(l, s, to);
        if (touches) {
          const int t = s + AHEAD;
          if (t < steps) load_one(w, touch, t * W_STEP, base + TOUCHED + wid * 256);
          else load_one(next, touch, max(0, min(t - steps, next_steps - 1)) * W_STEP, base + TOUCHED + wid * 256);      // (within the next one's K, which may be a step long)
        }
      }
    };
    // step s + 1 is there (this wave's touch, the last of what it asked for, may still be on its way), and step s has been read
    auto meet = [&](bool touched) {
      __builtin_amdgcn_s_waitcnt(0xc07f);        // lgkmcnt(0)
      if (touched && touches) asm volatile("s_waitcnt vmcnt(1)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      asm volatile("s_barrier" ::: "memory");
    };
#pragma unroll
    for (int a = 0; a < FN; ++a)
#pragma unroll
      for (int b = 0; b < FM; ++b) acc[a][b] = tile_floatx4{0.f, 0.f, 0.f, 0.f};
    if (steps >= SLOTS) tile_meet<(SLOTS - 1) * LOADS>();          // (whatever was issued after begin() leaves the first step's loads the oldest)
    else tile_meet<0>();
#pragma unroll
    for (int i = 0; i < READS; ++i) read(i, 0, 0);
    int s = 0;
    if constexpr (SLOTS == 3) {
      // step s lies in slot s % 3; the loads of step s + 2, and a touch behind them, may still be on their way where step s + 1 is met
      auto meet3 = [&](int newer) {
        __builtin_amdgcn_s_waitcnt(0xc07f);        // lgkmcnt(0)
        if (newer == 2 && touches) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(LOADS + 1) : "memory");
        else if (newer >= 1) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        asm volatile("s_barrier" ::: "memory");
      };
      int at = 0;
      for (; s + 3 < steps; ++s) {
        const int then = at == 2 ? 0 : at + 1;
        half(0, at, false, 0, 0);
        meet3(s > 0 ? 2 : 1);
        if (uneven && s + 3 == steps - 1) cut(K);
        half(1, then, true, s + 3, at);
        at = then;
      }
      for (; s < steps; ++s) {
        const int then = at == 2 ? 0 : at + 1;
        half(0, at, false, 0, 0);
        meet3(0);
        half(1, then, false, 0, 0);
        at = then;
      }
    } else {
      for (; s + 2 < steps; s += 2) {
        half(0, 0, false, 0, 0);
        meet(s > 0);
        if (uneven && s + 2 == steps - 1) cut(K);
        half(1, 1, true, s + 2, 0);
        half(0, 1, false, 0, 0);
        meet(true);
        if (uneven && s + 3 == steps - 1) cut(K);
        half(1, 0, true, min(s + 3, steps - 1), 1);        // (beyond the end: the last step again, into a slot that nothing reads)
      }
      for (; s < steps; ++s) {
        half(0, s & 1, false, 0, 0);
        meet(false);
        half(1, s & 1 ^ 1, false, 0, 0);
      }
    }
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");          // (the last products' sums are there)
    meet(false);
  }

 private:
  // where the j-th 1 KB of a step of tiles lies: tile j % 2 along k of row tile j / 2
  static __device__ __forceinline__ int tiles_at(int j, int K) { return j / 2 * ((K + 63) / 64 * 2048) + j % 2 * 1024; }
  __device__ __forceinline__ void issue(int i, int s, int slot) {
    const unsigned to = base + slot * STAGE;
    if (i < FN) load(w, wo[i], s * W_STEP, to + (wid * FN + i) * 1024);
    else load(x, xo[i - FN], s * ROW, to + W_BYTES + (wid * FM + i - FN) * 1024);
  }
  // pieces beyond K in the last step arrive as zeros
  __device__ __forceinline__ void cut(int K) {
    const int k0 = (K - 1) / 64 * 64;
    if (!TILED)          // (tiles are padded with zeros)
#pragma unroll
      for (int i = 0; i < FN; ++i)
        if (k0 + 8 * (lane % 8 ^ place((wid * FN + i) * 8 + lane / 8)) >= K) wo[i] = TILE_NO_ROW;
#pragma unroll
    for (int i = 0; i < FM; ++i)
      if (k0 + 8 * (lane % 8 ^ place((wid * FM + i) * 8 + lane / 8)) >= K) xo[i] = TILE_NO_ROW;
  }
};
