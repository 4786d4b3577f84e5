// The choice of a row's experts (moe.hip; moe_gemm.hip, whose plan takes few rows'
// logits itself).
#pragma once
#include <cfloat>

#include "common.h"

namespace arks {

// The largest of all lanes' values, by DPP moves: a shuffle goes through LDS, and
// the k passes of a row are one chain of these (64 rows of 128, k 8, 1.0 us less).
template <int CTRL>
__device__ __forceinline__ float moe_dpp(const float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(
      __float_as_int(-INFINITY), __float_as_int(v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float moe_wave_max(float v) {
  v = fmaxf(v, moe_dpp<0x111>(v));  // the lane 1, 2, 4 and 8 below in a row of 16,
  v = fmaxf(v, moe_dpp<0x112>(v));  // then the last lane of the rows below
  v = fmaxf(v, moe_dpp<0x114>(v));
  v = fmaxf(v, moe_dpp<0x118>(v));
  v = fmaxf(v, moe_dpp<0x142>(v));
  v = fmaxf(v, moe_dpp<0x143>(v));
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), WAVE_SIZE - 1));
}

// A wave's row of logits: softmax over E (<= 64 * S) then k argmax passes over
// the logits (same order as over probs), ties to the lower expert. The row
// stays in registers and a pass moves one value over the lanes (their index
// comes from a ballot); with the row read again for each pass and value and
// index both moved it took 11 us for 64 rows of 128, k 8. Lane j < k gets choice j.
template <int S>
__device__ __forceinline__ void moe_topk_row(const float* row, const int E,
                                             const int k, const int renorm,
                                             const int lane, float& weight,
                                             int& chosen) {
  float v[S];
  uint32_t open = 0;  // this lane's entries e = 64 * i + lane not yet chosen
#pragma unroll
  for (int i = 0; i < S; ++i) {
    const int e = 64 * i + lane;
    v[i] = e < E ? row[e] : -INFINITY;
    if (e < E) open |= 1u << i;
  }
  float m = -FLT_MAX;
#pragma unroll
  for (int i = 0; i < S; ++i) m = fmaxf(m, v[i]);
  m = moe_wave_max(m);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < S; ++i) s += __expf(v[i] - m);
  s = wave_reduce_sum(s);

  float mine = 0.f, wsum = 0.f;  // lane j keeps choice j
  int mine_id = 0;
  for (int j = 0; j < k; ++j) {
    float best = -INFINITY;
#pragma unroll
    for (int i = 0; i < S; ++i)
      if (open >> i & 1) best = fmaxf(best, v[i]);
    best = moe_wave_max(best);
    int id = -1, first = -1;  // first: of rows of NaN
#pragma unroll
    for (int i = S - 1; i >= 0; --i) {
      const bool is_open = open >> i & 1;
      const uint64_t any = __ballot(is_open);
      const uint64_t hit = __ballot(is_open && v[i] == best);
      if (any) first = 64 * i + __ffsll((unsigned long long)any) - 1;
      if (hit) id = 64 * i + __ffsll((unsigned long long)hit) - 1;
    }
    if (id < 0) id = first;
    if (id % 64 == lane) open &= ~(1u << (id / 64));
    const float w = __expf(best - m) / s;
    if (lane == j) {
      mine = w;
      mine_id = id;
    }
    wsum += w;
  }
  weight = mine * (renorm ? 1.f / wsum : 1.f);
  chosen = mine_id;
}

}  // namespace arks
