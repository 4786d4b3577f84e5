// Sums of split products: part [splits, rows, columns] fp32, added in order.
#pragma once
#include "common.h"

namespace arks {

using f32x2 = __attribute__((ext_vector_type(2))) float;
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

// The same at two places, 16 loads in flight (1 x 3584, 8 splits and their
// norm 4.6 us; one place after the other 5.4).
template <typename T>
__device__ __forceinline__ void sum_parts_pair(const float* p, const float* q,
                                               const int64_t stride,
                                               const int splits, T& a, T& b) {
  a = b = T{};
  for (int s0 = 0; s0 < splits; s0 += 8) {
    T v[8], w[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int64_t at = (int64_t)min(s0 + j, splits - 1) * stride;
      v[j] = *reinterpret_cast<const T*>(p + at);
      w[j] = *reinterpret_cast<const T*>(q + at);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (s0 + j < splits) {
        a += v[j];
        b += w[j];
      }
  }
}

}  // namespace arks
