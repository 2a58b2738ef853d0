// Attention of single rows whose splits of the keys have not been merged: partial results as the row kernel writes them
// (attn_mfma.hip), joined by the kernel that reads them instead of by a launch between the two (5 us a layer, of
// which a reader saves all but 0.1 to 0.3).
#pragma once
#include "common.h"

// The sink joins a finished (maximum M, sum L, unnormalised output) once, where the output is written: returns the
// factor on the output, 1 / (L + 2^(sink - M)) (times the head's gate), with care for a maximum below the sink's score.
// ``at`` is row * nH + head; with ``sinks`` the head's own score is taken.
__device__ __forceinline__ float finish_factor(float M, float L, int has_sink, float sink_l2, const float* gate, size_t gate_at,
                                               const float* sinks = nullptr, int nH = 1) {
  float f = 1.f;
  if (sinks) {
    has_sink = 1;
    sink_l2 = sinks[gate_at % (size_t)nH] * 1.4426950408889634f;
  }
  if (has_sink) {
    const float Ms = fmaxf(M, sink_l2);
    f = M == -INFINITY ? 0.f : exp2f(M - Ms);
    L = L * f + exp2f(sink_l2 - Ms);
  }
  const float inv = L > 0.f ? f / L : 0.f;
  return gate ? inv * gate[gate_at] : inv;
}

struct SplitRows {
  const float* o;          // [T][H][splits][D], unnormalised
  const float* ml;         // [T][H][splits][2]: maximum (times log2 e; -infinity: the split saw no key, and its o may hold anything), sum
  const float* sinks;      // [H] a score per head that joins the softmax's denominator, or null
  int splits, D;
};
constexpr int SPLITS_MAX = 32;            // splits a reader takes: all of them are on their way at once
constexpr int SPLITS_MAX_WIDTH = 128;     // elements of a head: the row kernel's largest

// One (row, head)'s merge by WAVES waves, wave ``w`` taking splits w, w + WAVES, ...; every lane asks for all it needs before it uses
// any of it.  ``ask`` loads, ``weigh`` forms the splits' weights and the factor on the output, ``sums`` adds this wave's splits in
// rising order, for each of the head's first ``width`` elements (zeros behind them), still to be added over the waves and multiplied by the factor.
template <int WAVES>
struct SplitMerge {
  static constexpr int PER = SPLITS_MAX / WAVES, C = SPLITS_MAX_WIDTH / WAVE;
  float2 ml;
  float part[PER][C];
  float weight;      // lane s: split s's

  __device__ __forceinline__ void ask(const SplitRows& p, size_t at, int width, int w, int lane) {
    const float* o = p.o + at * p.splits * p.D;
    ml = lane < p.splits ? *(const float2*)(p.ml + (at * p.splits + lane) * 2) : float2{-INFINITY, 0.f};
#pragma unroll
    for (int i = 0; i < PER; ++i)
#pragma unroll
      for (int c = 0; c < C; ++c)
        part[i][c] = (w + i * WAVES < p.splits && lane + WAVE * c < width) ? o[(size_t)(w + i * WAVES) * p.D + lane + WAVE * c] : 0.f;
  }
  __device__ __forceinline__ float weigh(const SplitRows& p, size_t at, int H) {
    const float M = wave_max(ml.x);
    weight = ml.x == -INFINITY ? 0.f : exp2f(ml.x - M);
    return finish_factor(M, wave_sum(weight * ml.y), 0, 0.f, nullptr, at, p.sinks, H);
  }
  __device__ __forceinline__ void sums(int w, float* out, int lane) {
    float acc[C];
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const float f = __shfl(weight, w + i * WAVES, WAVE);
#pragma unroll
      for (int c = 0; c < C; ++c) acc[c] = fmaf(f, f != 0.f ? part[i][c] : 0.f, acc[c]);
    }
#pragma unroll
    for (int c = 0; c < C; ++c) out[lane + WAVE * c] = acc[c];
  }
};
