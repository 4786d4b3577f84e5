// Sums of split products: part [splits, rows, columns] fp32, added in order.
#pragma once
#include "common.h"

namespace arks {

using f32x4 = __attribute__((ext_vector_type(4))) float;

// 4 columns of all splits, `stride` floats apart; 8 loads in flight
__device__ __forceinline__ f32x4 sum_parts4(const float* p,
                                            const int64_t stride,
                                            const int splits) {
  f32x4 s{0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < splits; s0 += 8) {
    f32x4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v[j] = *reinterpret_cast<const f32x4*>(
          p + (int64_t)min(s0 + j, splits - 1) * stride);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (s0 + j < splits) s += v[j];
  }
  return s;
}

__device__ __forceinline__ float2 sum_parts2(const float* p,
                                             const int64_t stride,
                                             const int splits) {
  float2 s{0.f, 0.f};
  for (int s0 = 0; s0 < splits; s0 += 8) {
    float2 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v[j] = *reinterpret_cast<const float2*>(
          p + (int64_t)min(s0 + j, splits - 1) * stride);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (s0 + j < splits) {
        s.x += v[j].x;
        s.y += v[j].y;
      }
  }
  return s;
}

}  // namespace arks
