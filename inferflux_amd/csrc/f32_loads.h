// What the true 32-bit products share (gemm_f32.hip, moe_f32.hip): the loads of four k-values of a row.
#pragma once
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Four consecutive elements k .. k + 3 of a row of K, zeros behind its end.  VEC: the row starts on 16 bytes (8 for bf16)
// and K is a multiple of 4, so four elements are all there or all not.
template <bool VEC, typename T>
__device__ __forceinline__ f32x4 load4(const T* __restrict__ row, int k, int K) {
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if constexpr (VEC && sizeof(T) == 4) {
    if (k < K) v = *(const f32x4*)(row + k);
  } else if constexpr (VEC) {
    typedef bf16_t bf16x4 __attribute__((ext_vector_type(4)));
    if (k < K) {
      const bf16x4 b = *(const bf16x4*)(row + k);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = (float)b[j];
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (k + j < K) v[j] = to_f(row[k + j]);
  }
  return v;
}
