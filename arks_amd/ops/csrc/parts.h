// What a product leaves to its consumer to add: sums of split products, part
// [splits, rows, columns] fp32, added in order, and the rows of a token's experts.
#pragma once
#include "common.h"

namespace arks {

using f32x2 = __attribute__((ext_vector_type(2))) float;
using f32x4 = __attribute__((ext_vector_type(4))) float;

// How many splits' loads are asked for at once (U below). Loads of splits that are not
// there repeat the last one and take as long as others: us, always 8 -> so, 64 rows of
// 3584 and their norm, 2 splits 3.43 -> 2.78, 4 splits 3.44 -> 2.99; 4608 columns to
// be rotated, 3 splits 4.43 -> 3.90; 200 rows, 3 splits 5.23 -> 4.41.
inline int parts_flight(const int splits) {
  return splits <= 2 ? 2 : splits <= 4 ? 4 : 8;
}

// 4 columns of all splits, `stride` floats apart; U loads in flight
template <int U>
__device__ __forceinline__ f32x4 sum_parts4(const float* p,
                                            const int64_t stride,
                                            const int splits) {
  f32x4 s{0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < splits; s0 += U) {
    f32x4 v[U];
#pragma unroll
    for (int j = 0; j < U; ++j)
      v[j] = *reinterpret_cast<const f32x4*>(
          p + (int64_t)min(s0 + j, splits - 1) * stride);
#pragma unroll
    for (int j = 0; j < U; ++j)
      if (s0 + j < splits) s += v[j];
  }
  return s;
}

// The same at two places, 2 * U loads in flight (1 x 3584, 8 splits and their
// norm 4.6 us; one place after the other 5.4).
template <int U, typename T>
__device__ __forceinline__ void sum_parts_pair(const float* p, const float* q,
                                               const int64_t stride,
                                               const int splits, T& a, T& b) {
  a = b = T{};
  for (int s0 = 0; s0 < splits; s0 += U) {
    T v[U], w[U];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int64_t at = (int64_t)min(s0 + j, splits - 1) * stride;
      v[j] = *reinterpret_cast<const T*>(p + at);
      w[j] = *reinterpret_cast<const T*>(q + at);
    }
#pragma unroll
    for (int j = 0; j < U; ++j)
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
