// The activations that the products of many rows have as their epilogue (gemm_tiles.hip, grouped_gemm.hip).
#pragma once
#include "common.h"

// act(g) up and act(v) for the epilogues, where a lane has up to 256 of them and the matrix cores wait: a / (1 + exp(-z)) in 32-bit
// arithmetic, without what expf() and the division spend on ranges.  The exponential is the hardware's exp2 of at most a half, reduced by the
// product with log2(e) in two parts (Cody and Waite); the quotient is the hardware's reciprocal with one correction (Markstein), in quarters, so
// that no reciprocal is a denormal number.  REST: the rounding of 1 + exp(-z) is corrected, too.  Errors against 64 bits, of 2^-24 of the result,
// largest and mean square, expf() or tanhf() and a division : this : hardware's exp2 and reciprocal alone
//   silu          |g| < 4 2.49, 0.663 : 2.44, 0.664 : 5.8, 1.08     |g| < 20 3.06, 0.645 : 3.06, 0.647 : 17, 3.8
//   gated clamp   |g| < 4 6.8, 1.43 : 6.8, 1.43 : 11, 1.84
//   gelu (REST)   |v| < 1 6.1, 0.85 : 3.9, 0.64 : 5.0, 0.91         |v| < 4 14,091, 933 : 22, 2.7 : 24, 2.9 (of all values together 3.3e-8 : 2.3e-8 : 4.4e-8)
// Gelu's tanh form is v / (1 + exp(-2 u)), which keeps the tail where 1 + tanh(u) cancels; without REST its 4.1e-8 at positive v are more than tanhf's.
// us a launch of gate/up (silu) in the same order: 2,048 rows of 37,888 x 3,584 453 : 425 : 415, 4,500 of 17,920 x 1,536 224 : 200 : 191, 2,048 of
// 9,728 x 896 44.8 : 40.2 : 37.0.
template <bool REST>
__device__ __forceinline__ float over_one_plus_exp(float a, float z) {
  const float y = __builtin_amdgcn_fmed3f(-z, -126.f, 126.f);          // (beyond, exp() is 0 or infinite anyway)
  const float whole = rintf(y * 1.44269504f);
  const float e = ldexpf(__builtin_amdgcn_exp2f(fmaf(y, 1.92596299e-8f, fmaf(y, 1.44269504f, -whole))), (int)whole);
  const float d = fmaf(e, 0.25f, 0.25f), n = 0.25f * a, r = __builtin_amdgcn_rcpf(d), q = n * r;
  float left = fmaf(-d, q, n);
  if (REST) left = fmaf(-fmaf(e, 0.25f, 0.25f - d), q, left);
  return __builtin_amdgcn_div_fixupf(fmaf(left, r, q), d, n);          // (infinities)
}
__device__ __forceinline__ float tile_gelu(float v) { return over_one_plus_exp<true>(v, 1.5957691216057308f * (v + 0.044715f * v * v * v)); }
template <int ACT> __device__ __forceinline__ float tile_gated(float g, float up, float limit) {
  if (ACT == ACT_GELU_TANH) return tile_gelu(g) * up;
  if (ACT == ACT_SILU) return over_one_plus_exp<false>(g, g) * up;
  g = fminf(g, limit), up = fminf(fmaxf(up, -limit), limit);
  return over_one_plus_exp<false>(g, 1.702f * g) * (up + 1.0f);
}
template <int ACT> __device__ __forceinline__ float tile_act(float v) {
  if (ACT == ACT_NONE) return v;
  if (ACT == ACT_RELU_SQUARED) { const float r = fmaxf(v, 0.f); return r * r; }
  return ACT == ACT_GELU_TANH ? tile_gelu(v) : over_one_plus_exp<false>(v, v);
}
