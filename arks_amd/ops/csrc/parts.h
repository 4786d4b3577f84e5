// What a product leaves to its consumer to add: sums of split products, part
// [splits, rows, columns] fp32, added in order, and the rows of a token's experts.
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

// The weighted mix of a token's k rows of y: 8 columns from h on, in the rows'
// order, 8 rows' loads in flight. start(j), weight(j) for j up to the next multiple
// of 8: where row j begins in y, and its weight, 0 from k on; rows of weight 0 count
// as nothing (they may hold anything).
template <typename Start, typename Weight>
__device__ __forceinline__ ushort8 mix_rows8(const bf16* y, const int k, const int h,
                                             Start start, Weight weight) {
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int j0 = 0; j0 < k; j0 += 8) {
    ushort8 u[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      u[j] = *reinterpret_cast<const ushort8*>(y + start(j0 + j) + h);
    __builtin_amdgcn_sched_barrier(0);  // all 8 are asked for first
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float w = weight(j0 + j);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        acc[e] += w == 0.f ? 0.f : w * bf16_bits_to_float(u[j][e]);
    }
  }
  ushort8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = float_to_bf16_bits(acc[e]);
  return o;
}

}  // namespace arks
