// The loop of wide_gemm.hip: as tile_engine.h's (8 waves in two groups of four,
// one of which multiplies while the other reads LDS and asks for rows further
// ahead), for tiles of several sizes.
//
// Two operands: X, whose rows the two groups share out (FX0 + FX1 fragments of 16
// a wave, in two halves), and Y, which the four waves of a group share out (FY
// fragments a wave). A step of 64 columns is cut into four phases: half 0 of X
// with columns 0..31, with 32..63, then half 1 with 32..63 and with 0..31, each
// times all of a wave's Y. So a wave holds one half's fragments of X for 32
// columns, and all of Y: 16 + 8 FY registers (tile_engine.h's phases, halves of
// both operands with 64 columns, hold 32 + 8 FY), and 256 x 320 sums fit beside
// them; the reads of LDS are 9, 9, 4 and 4 a phase of 20 matrix operations instead
// of 12, 4, 8 and 0.
//
// 37888 x 3584 with the activation, 8192 rows: tiles of 256 x 320 1520 us (1464
// TFLOP/s), of 256 x 256 1527, tile_engine.h's 1599 in the same run. Of a step of
// 256 x 320 the matrix operations are 2560 clocks, 3300 pass at 1.9 GHz (power;
// 2.4 at small loads). Slower: reads waited for behind the barrier and loads a
// phase later (8192 rows 1463 us for 1415), all of Y asked for in one phase (1454),
// each XCD beginning at another step (1443 for 1433).
//
// The rows' order in LDS is free (each lane asks for the row that it wants), so
// fragments are 16 rows in a row, 128 B each, their 16-byte pieces permuted by the
// row's number.
//
// Which waits make it safe: as in tile_engine.h, what phase p has read may be
// overwritten from phase p + 1 on, and what is waited for in phase q be read from
// phase q + 1 on. Half 0 of X and Y are read in phases 1 and 2, and loaded anew
// (two steps ahead) in 3 and 4; half 1 is read in 3 and 4 and loaded (a step
// ahead) in phase 1. Loads go out in the order x0, y, x1 of a step, LX + F in all,
// so that in phase 2, before x1 is read, so many newer ones may be under way, and in
// phase 4 as many behind the next step's x0 and y.
//
// A tile may have fewer rows of Y than there are places for (F fragments a wave;
// not AX, where the waves' fragments take turns).
#pragma once
#include "tile_engine.h"

namespace arks {

// AX: X is a, Y is w; else the other way round.
template <int FX0, int FX1, int FY, bool AX, int CX = 0>
class WideTile {
 public:
  using Lds = __attribute__((address_space(3))) char;
  static constexpr int X0 = 32 * FX0, X = X0 + 32 * FX1, Y = 64 * FY;
  static constexpr int STAGE = (X + Y) * 128, LDS = 2 * STAGE;
  static constexpr int LX0 = FX0 / 2, LX1 = FX1 / 2, LX = LX0 + LX1;
  static_assert(FX0 % 2 == 0 && FX1 % 2 == 0 && FX0 >= FX1 && LDS <= 160 * 1024);

  // Byte offsets of the rows that this lane loads, from the buffers' starts.
  struct Rows {
    __amdgpu_buffer_rsrc_t x, y;
    uint32_t xo[LX], yo[FY];
  };

  // The columns of a tile: `steps` of 64 from step s0 on, begun with the one `turn`
  // behind s0 and gone round from the last to the first.
  struct Span {
    int s0, steps, turn;
    __device__ __forceinline__ int at(const int s) const {
      return s0 + (s + turn < steps ? s + turn : s + turn - steps);
    }
  };

  __device__ __forceinline__ explicit WideTile(char* lds)
      : lds_(lds),
        lane_(threadIdx.x % WAVE_SIZE),
        wave_(__builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE)),
        wm_(wave_ / 4),
        wn_(wave_ % 4) {
    const int lq = lane_ % 16, la = lane_ / 16;
#pragma unroll
    for (int k = 0; k < 2; ++k) at_[k] = lq * 128 + (((la ^ (lq & 7)) * 16) ^ (k * 64));
  }

  // The row of X (Y) that load j of this lane covers, and which 16 bytes of its
  // 128 it asks for.
  __device__ __forceinline__ int row_x(int j) const {
    return j < LX0 ? (wave_ * LX0 + j) * 8 + lane_ / 8
                   : X0 + (wave_ * LX1 + j - LX0) * 8 + lane_ / 8;
  }
  __device__ __forceinline__ int row_y(int j, int f = FY) const {
    return (wave_ * f + j) * 8 + lane_ / 8;
  }
  // The first of the 16 rows of Y that this wave's fragment y is.
  __device__ __forceinline__ int frag_y(int y) const {
    return (AX ? wn_ * FY + y : 4 * y + wn_) * 16;
  }
  __device__ __forceinline__ uint32_t piece() const {
    return ((lane_ % 8) ^ (lane_ / 8)) * 16;
  }

  // The first loads of a tile's `steps` from step s0 on; all reads of the last
  // tile's must be over. F: fragments of Y a wave, up to FY.
  template <int F = FY>
  __device__ __forceinline__ void prologue(const Rows& t, const Span& k) {
    load_x<0, LX0>(t, 0, k.at(0));
    load_y<F, 0, F>(t, 0, k.at(0));
    load_x<LX0, LX>(t, 0, k.at(0));
    if (k.steps > 1) {
      load_x<0, LX0>(t, STAGE, k.at(1));
      load_y<F, 0, F>(t, STAGE, k.at(1));
    }
  }
  // Waits until the first phase's operands are there (this wave's loads).
  template <int F = FY>
  __device__ __forceinline__ void prologue_wait(int steps) {
    if (steps == 1) wait<0>();
    else wait<LX + F>();
  }

  // acc[fragment of X][fragment of Y]. Entered and left by all waves together
  // (through barriers).
  template <int F = FY>
  __device__ __forceinline__ void run(const Rows& t, const Span& k) {
#pragma unroll
    for (int i = 0; i < FX0 + FX1; ++i)
#pragma unroll
      for (int j = 0; j < FY; ++j) acc[i][j] = tile_f32x4{0.f, 0.f, 0.f, 0.f};
    barrier();
    if (wm_ == 1) barrier();  // the second group runs one slot behind
    int x0[2], x1[2], y[2], stage = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      x0[h] = at_[h] + wm_ * FX0 * 2048;
      x1[h] = FX0 == FX1 ? x0[h] : at_[h] + wm_ * FX1 * 2048;
      y[h] = at_[h] + wn_ * (AX ? FY : 1) * 2048;
    }
    for (int s = 0; s < k.steps; ++s) {
      step<F>(t, k, s, stage, x0, x1, y);
      const int turn = stage ? -STAGE : STAGE;
      stage += turn;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        x0[h] += turn;
        x1[h] = FX0 == FX1 ? x0[h] : x1[h] + turn;
        y[h] += turn;
      }
    }
    if (wm_ == 0) barrier();
  }

  // All waves' LDS writes before it can be read behind it; loads stay under way.
  __device__ __forceinline__ static void sync() { meet_reads(); }

  __device__ __forceinline__ int lane() const { return lane_; }
  __device__ __forceinline__ int wave() const { return wave_; }
  __device__ __forceinline__ int wm() const { return wm_; }
  __device__ __forceinline__ int wn() const { return wn_; }
  tile_f32x4 acc[FX0 + FX1][FY];

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
  // ends a slot of reads; at most N loads stay outstanding (none: !more)
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

  template <int CACHE>
  __device__ __forceinline__ void load(const __amdgpu_buffer_rsrc_t& b, uint32_t o,
                                       int to, int s) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(b, (Lds*)(lds_ + to), 16, o,
                                             s * (TILE_K * 2), 0, CACHE);
  }
  template <int A, int B>
  __device__ __forceinline__ void load_x(const Rows& t, int stage, int s) {
#pragma unroll
    for (int j = A; j < B; ++j)
      load<CX>(t.x, t.xo[j],
           stage + (j < LX0 ? (wave_ * LX0 + j) * 1024
                                    : X0 * 128 + (wave_ * LX1 + j - LX0) * 1024),
           s);
  }
  template <int F, int A, int B>
  __device__ __forceinline__ void load_y(const Rows& t, int stage, int s) {
#pragma unroll
    for (int j = A; j < B; ++j)
      load<0>(t.y, t.yo[j], stage + X * 128 + (wave_ * F + j) * 1024, s);
  }

  template <int H>
  __device__ __forceinline__ void read_x(int at) {
#pragma unroll
    for (int q = 0; q < (H ? FX1 : FX0); ++q)
      xf_[q] = *reinterpret_cast<const ushort8*>(lds_ + at + (H ? X0 * 128 : 0) +
                                                 q * 2048);
  }
  template <int F>
  __device__ __forceinline__ void read_y(int at, int k) {
#pragma unroll
    for (int q = 0; q < F; ++q)
      yf_[k][q] = *reinterpret_cast<const ushort8*>(lds_ + at + X * 128 +
                                                    q * (AX ? 2048 : 8192));
  }
  template <int F, int H>
  __device__ __forceinline__ void mul(int k) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int q = 0; q < (H ? FX1 : FX0); ++q)
#pragma unroll
      for (int y = 0; y < F; ++y) {
        tile_f32x4& c = acc[H * FX0 + q][y];
        c = AX ? tile_mfma(yf_[k][y], xf_[q], c) : tile_mfma(xf_[q], yf_[k][y], c);
      }
    __builtin_amdgcn_s_setprio(0);
    barrier();
  }

  template <int F>
  __device__ __forceinline__ void step(const Rows& t, const Span& k, int s, int stage,
                                       const int (&x0)[2], const int (&x1)[2],
                                       const int (&y)[2]) {
    const bool one = s + 1 < k.steps, two = s + 2 < k.steps;
    read_y<F>(y[0], 0);
    read_x<0>(x0[0]);
    if (one) load_x<LX0, LX>(t, STAGE - stage, k.at(s + 1));
    meet_reads();
    mul<F, 0>(0);
    read_y<F>(y[1], 1);
    read_x<0>(x0[1]);
    meet<LX + F>(one);  // x1 of this step
    mul<F, 0>(1);
    read_x<1>(x1[1]);
    if (two) {
      load_x<0, LX0>(t, stage, k.at(s + 2));
      load_y<F, 0, F / 2>(t, stage, k.at(s + 2));
    }
    meet_reads();
    mul<F, 1>(1);
    read_x<1>(x1[0]);
    if (two) load_y<F, F / 2, F>(t, stage, k.at(s + 2));
    meet<LX + F>(two);  // x0 and y of the next step
    mul<F, 1>(0);
  }

  char* lds_;
  int lane_, wave_, wm_, wn_, at_[2];
  ushort8 xf_[FX0], yf_[2][FY];
};

}  // namespace arks
