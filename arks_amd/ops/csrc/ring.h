// A ring of stages in LDS: 4 waves of a workgroup only load, steps ahead of the 4
// that multiply (mid_gemm.hip, seq_routed.hip).
//
// One barrier a step. In front of the barrier of step s the waves that load wait
// for their loads of step s + 1, and the others for their reads of step s: behind
// it step s + 1 may be read and the stage of step s be loaded anew (with step s +
// NS, NS stages). Rows go from memory straight into LDS, 128 B each, their 16-byte
// pieces permuted by the row's number (as in tile_engine.h).
#pragma once
#include "tile_engine.h"

namespace arks {

// 1 KB of 8 rows into LDS, 16 B a lane, `at` bytes behind its offset. ONCE: what is
// read once, the weights, passes the caches by (non-temporal): 64 rows x 37888 x
// 3584 51 -> 45 us, the rows of a stay there.
template <bool ONCE>
__device__ __forceinline__ void ring_load(const __amdgpu_buffer_rsrc_t& b, char* to,
                                          const uint32_t offset, const int at) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      b, (__attribute__((address_space(3))) char*)to, 16, offset, at, 0,
      ONCE ? 2 : 0);
}
template <int N>
__device__ __forceinline__ void ring_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void ring_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// The loads of all but the newest n steps are there (LOADS a step and wave).
template <int LOADS, int MOST>
__device__ __forceinline__ void ring_wait_steps(const int n) {
  static_assert(MOST * LOADS < 64, "waits count to 63");
  if constexpr (MOST == 0) {
    ring_wait<0>();
  } else {
    if (n >= MOST) ring_wait<MOST * LOADS>();
    else ring_wait_steps<LOADS, MOST - 1>(n);
  }
}

// What a wave that loads does: load() asks for the next of `total` steps, and
// behind(t) joins what barriers the others have behind step t. They begin with one
// barrier, and have one in each step.
template <int NS, int LOADS, typename Load, typename Behind>
__device__ __forceinline__ void ring_feed(const int total, Load load, Behind behind) {
  const int first = min(NS, total);
  for (int t = 0; t < first; ++t) load();
  ring_wait_steps<LOADS, NS - 1>(first - 1);
  ring_barrier();
  int t = 0;
  for (; t + NS < total; ++t) {
    ring_wait<(NS - 2) * LOADS>();
    ring_barrier();
    load();
    behind(t);
  }
  for (; t < total; ++t) {
    ring_wait_steps<LOADS, NS - 1>(max(0, total - 2 - t));
    ring_barrier();
    behind(t);
  }
}

}  // namespace arks
