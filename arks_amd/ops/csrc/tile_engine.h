// The product engine for many rows: a workgroup of 8 waves takes 256 rows of
// a x 256 rows of w (or, where at most 128 rows of a are left, 128 x 256), 64
// of K per step, and goes from one tile to the next without a drained memory
// queue between them.
//
// What bounds it are the matrix cores (and with them the chip's power), so the
// split is made for them: the waves form two groups of four, one wave of each
// per SIMD. A step is cut into phases of 16 matrix operations a wave
// (quadrants of the tile); while one group multiplies, the other reads the
// operands of its next phase from LDS and asks for rows further ahead, and a
// barrier swaps them. A wave holds 128 x 64 sums, which makes the LDS reads
// (94 B a cycle and CU) fit under the matrix operations.
//
// Rows go from memory straight into LDS (16 B a lane, no registers), up to 2.5
// steps ahead; waits count loads, they never drain them. LDS rows are 128 B
// without padding, as those loads need: the 16-byte pieces of a row are
// permuted by the row's number instead, on the way in (each lane asks for
// another piece of its row) and when read, so that 8 lanes that read the same
// piece of 8 rows meet 8 different bank groups.
//
// Which waits make it safe (slot: the time between two barriers; a group reads
// in one slot and multiplies in the next, the other group one slot later):
//  - a wave's reads of a phase have returned (lgkmcnt 0) before the barrier
//    that ends its slot, so what phase p read may be overwritten from phase
//    p + 1 on, by either group;
//  - loads that phase q waits for (vmcnt) before that barrier may be read from
//    phase q + 1 on. Loads return in order, so "at most n outstanding" means
//    that all but the newest n are there; stores in between only make it wait
//    longer.
#pragma once
#include "common.h"

namespace arks {

typedef __attribute__((ext_vector_type(8))) __bf16 tile_bf16x8;
typedef __attribute__((ext_vector_type(4))) float tile_f32x4;

constexpr int TILE_M = 256, TILE_HALF = 128, TILE_K = 64;
// full: 2 stages of 4 halves of 16 KB; half: 3 stages of 3
constexpr int TILE_LDS = 3 * 3 * 16384;

__device__ __forceinline__ tile_f32x4 tile_mfma(const ushort8& a,
                                                const ushort8& b,
                                                const tile_f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
      *reinterpret_cast<const tile_bf16x8*>(&a),
      *reinterpret_cast<const tile_bf16x8*>(&b), c, 0, 0, 0);
}

__device__ __forceinline__ ushort8 tile_round(const float (&v)[8]) {
  tile_bf16x8 o;
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = (__bf16)v[i];
  return *reinterpret_cast<ushort8*>(&o);
}

// g / (1 + e^-g) * u, the quotient as a division gives it: the reciprocal (of
// an eighth, which is never below the normal numbers) with one correction, half
// of a division's operations; infinities by the fix-up. Over gate and up products
// of 600 to 8192 rows and 1 to 256 rows this takes 0.8 % more time than the bare
// reciprocal, a division 1.6 % (18944 x 3584, 8192 rows 1560, 1543 and 1568 us).
__device__ __forceinline__ float tile_silu_mul(float g, float u) {
  const float n = 0.125f * g, d = __builtin_fmaf(__expf(-g), 0.125f, 0.125f);
  const float r = __builtin_amdgcn_rcpf(d), q = n * r;
  return __builtin_amdgcn_div_fixupf(
             __builtin_fmaf(__builtin_fmaf(-q, d, n), r, q), d, n) * u;
}

// A tile to compute. Rows of a and of the two halves of w are given by their
// byte offsets from a buffer's start (under 4 GiB), which the lane that loads
// them holds: half h, load j of a wave covers rows (2 * wave + j) * 8 + lane / 8
// of that half.
struct TileRows {
  __amdgpu_buffer_rsrc_t a, w[2];
  uint32_t ao[2][2], wo[2][2];
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_buffer(const void* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, 0xffffffff,
                                           0x00027000);
}

// The row of a half that load j of this lane covers.
__device__ __forceinline__ int tile_row(int wave, int lane, int j) {
  return (2 * wave + j) * 8 + lane / 8;
}
// Which 16-byte piece of the row's 128 bytes it asks for. Operand a reads rows
// base + lq, operand w rows base + 8 * (lq / 4) + lq % 4 (+ 4), so that a
// lane's sums are 8 neighbouring columns: each has the swizzle that is a
// bijection over 8 lanes in a row.
__device__ __forceinline__ uint32_t tile_piece_a(int row, int lane) {
  return ((lane % 8) ^ (row & 7)) * 16;
}
__device__ __forceinline__ uint32_t tile_piece_w(int row, int lane) {
  return ((lane % 8) ^ ((row & 3) | ((row >> 3) & 1) << 2)) * 16;
}

class Tile {
 public:
  using Lds = __attribute__((address_space(3))) char;

  __device__ __forceinline__ explicit Tile(char* lds)
      : lds_(lds),
        lane_(threadIdx.x % WAVE_SIZE),
        wave_(__builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE)),
        wm_(wave_ / 4),
        wn_(wave_ % 4) {
    const int lq = lane_ % 16, la = lane_ / 16;
    const int r = 8 * (lq / 4) + lq % 4;
    a_lo_ = (wm_ * 64 + lq) * 128 + ((la ^ (lq & 7)) * 16);
    w_lo_ = (wn_ * 32 + r) * 128 +
            ((la ^ ((r & 3) | ((r >> 3) & 1) << 2)) * 16);
  }

  // The first loads of a tile; all reads of the last tile's must be over.
  __device__ __forceinline__ void prologue(const TileRows& t, int steps,
                                           bool half) {
    if (half) {
      half_ab(t, 0, 0);
      half_b1(t, 0, 0);
      if (steps > 1) {
        half_ab(t, 1, 1);
        half_b1(t, 1, 1);
      }
    } else {
      load_a(t, 0, 0, 0);
      load_w(t, 0, 0, 0);
      load_w(t, 0, 1, 0);
      load_a(t, 0, 1, 0);
      if (steps > 1) {
        load_a(t, 1, 0, 1);
        load_w(t, 1, 0, 1);
        load_w(t, 1, 1, 1);
      }
    }
  }

  // Waits until the first phase's operands are there (this wave's loads).
  __device__ __forceinline__ void prologue_wait(int steps, bool half) {
    if (steps == 1) wait<0>();
    else if (half) wait<8>();
    else wait<10>();
  }

  // acc[rows / 128][w half][8 * la + 4 * f + r][16 * t + lq of the wave's 64
  // rows]. Entered and left by all waves together (through barriers).
  __device__ __forceinline__ void run(const TileRows& t, int steps, bool half) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            acc[i][j][f][q] = tile_f32x4{0.f, 0.f, 0.f, 0.f};
    barrier();
    if (wm_ == 1) barrier();  // the second group runs one slot behind
    if (half) {
      int at = 0, ahead = 2;
      for (int s = 0; s < steps; ++s) {
        half_step(t, s, steps, at, ahead);
        at = at == 2 ? 0 : at + 1;
        ahead = ahead == 2 ? 0 : ahead + 1;
      }
    } else {
      int s = 0;
      for (; s + 1 < steps; s += 2) {
        full_step<0>(t, s, steps);
        full_step<1>(t, s + 1, steps);
      }
      if (s < steps) full_step<0>(t, s, steps);
    }
    if (wm_ == 0) barrier();
  }

  // All waves' LDS writes before it can be read behind it; loads stay under way.
  __device__ __forceinline__ static void sync() { meet_reads(); }

  // f(group of sums 0..7, row of the tile, column of the half, [half 0's 8
  // sums], [half 1's]); the group is known to the compiler
  template <typename F>
  __device__ __forceinline__ void each(F f) const {
    const int lq = lane_ % 16, la = lane_ / 16;
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      float v[2][8];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int c = 0; c < 8; ++c)
          v[j][c] = acc[x / 4][j][c / 4][x % 4][c % 4];
      f(x, x / 4 * 128 + wm_ * 64 + x % 4 * 16 + lq, wn_ * 32 + 8 * la, v[0],
        v[1]);
    }
  }

  __device__ __forceinline__ int lane() const { return lane_; }
  __device__ __forceinline__ int wave() const { return wave_; }

 private:
  template <int N>
  __device__ __forceinline__ static void wait() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
  }
  __device__ __forceinline__ static void barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }
  // ends a slot of reads; at most N loads stay outstanding (all before: !more)
  template <int N>
  __device__ __forceinline__ static void meet(bool more) {
    __builtin_amdgcn_sched_barrier(0);
    if (more) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }
  __device__ __forceinline__ static void meet_reads() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }

  __device__ __forceinline__ void load(const __amdgpu_buffer_rsrc_t& b,
                                       const uint32_t (&o)[2], int to, int s) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          b, (Lds*)(lds_ + to + (2 * wave_ + j) * 1024), 16, o[j],
          s * (TILE_K * 2), 0, 0);
  }
  // full: a stage b half h at (2 b + h) * 16 KB, w 64 KB behind
  __device__ __forceinline__ void load_a(const TileRows& t, int b, int h,
                                         int s) {
    load(t.a, t.ao[h], (2 * b + h) * 16384, s);
  }
  __device__ __forceinline__ void load_w(const TileRows& t, int b, int h,
                                         int s) {
    load(t.w[h], t.wo[h], 65536 + (2 * b + h) * 16384, s);
  }
  // half: stage b at b * 48 KB: a, w half 0, w half 1
  __device__ __forceinline__ void half_ab(const TileRows& t, int b, int s) {
    load(t.a, t.ao[0], b * 49152, s);
    load(t.w[0], t.wo[0], b * 49152 + 16384, s);
  }
  __device__ __forceinline__ void half_b1(const TileRows& t, int b, int s) {
    load(t.w[1], t.wo[1], b * 49152 + 32768, s);
  }

  __device__ __forceinline__ void read_a(int from) {
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        af_[q][k] = *reinterpret_cast<const ushort8*>(
            lds_ + ((a_lo_ ^ (k * 64)) + from + q * 2048));
  }
  __device__ __forceinline__ void read_w(int h, int from) {
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int f = 0; f < 2; ++f)
        wf_[h][f][k] = *reinterpret_cast<const ushort8*>(
            lds_ + ((w_lo_ ^ (k * 64)) + from + f * 512));
  }
  __device__ __forceinline__ void mul(int i, int j) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          acc[i][j][f][q] = tile_mfma(wf_[j][f][k], af_[q][k], acc[i][j][f][q]);
    __builtin_amdgcn_s_setprio(0);
    barrier();
  }

  // Loads go out in the order a0, w0, w1, a1 of a step, one half a phase, two
  // steps (a1: one) ahead, each into what was read a phase or more ago.
  template <int B>
  __device__ __forceinline__ void full_step(const TileRows& t, int s,
                                            int steps) {
    const bool one = s + 1 < steps, two = s + 2 < steps;
    read_w(0, 65536 + 2 * B * 16384);
    read_a(2 * B * 16384);
    if (one) load_a(t, B ^ 1, 1, s + 1);
    meet<10>(one);  // w1 of this step
    mul(0, 0);
    read_w(1, 65536 + (2 * B + 1) * 16384);
    if (two) load_a(t, B, 0, s + 2);
    meet<10>(two);  // a1 of this step
    mul(0, 1);
    read_a((2 * B + 1) * 16384);
    if (two) load_w(t, B, 0, s + 2);
    meet_reads();
    mul(1, 1);
    if (two) load_w(t, B, 1, s + 2);
    meet<10>(two);  // a0 and w0 of the next step
    mul(1, 0);
  }

  // Loads of two steps ahead, into the stage that the last step read.
  __device__ __forceinline__ void half_step(const TileRows& t, int s, int steps,
                                            int at, int ahead) {
    const bool two = s + 2 < steps;
    read_w(0, at * 49152 + 16384);
    read_a(at * 49152);
    if (two) half_ab(t, ahead, s + 2);
    meet<10>(two);  // w1 of this step
    mul(0, 0);
    read_w(1, at * 49152 + 32768);
    if (two) half_b1(t, ahead, s + 2);
    meet<8>(two);  // a and w0 of the next step
    mul(0, 1);
  }

  char* lds_;
  int lane_, wave_, wm_, wn_, a_lo_, w_lo_;
  ushort8 af_[4][2], wf_[2][2][2];
  tile_f32x4 acc[2][2][2][4];
};

}  // namespace arks
