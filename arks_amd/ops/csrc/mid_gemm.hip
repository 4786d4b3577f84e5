// out[M, N] = a[M, K] . w[N, K]^T (+ bias), or silu(gate) * up of two such
// products, for up to 256 rows: steps that decode, short prompts.
//
// A few rows are bound by the weights' stream, 200 by both it and the matrix
// cores (200 rows x 37888 x 3584 are 45 us of weights and 39 us of matrix
// operations; tile_engine.h is for those that the cores alone bound, and
// stream_gemm.hip takes few rows of small weights, without sums for anyone to
// add). So all rows of a meet a weight row at once (it is read once), the
// weights' rows are cut as finely as gives every CU one tile of them (or, for
// small products, one run of K: fp32 sums of the runs for the consumer to
// add), and loads run NS - 1 steps of 64 columns ahead.
//
// 8 waves, 2 along the weights x 4 along the rows of a: a wave holds 16 * QT
// weight rows x 16 * FT rows of a. The two groups of four take turns: in a slot
// between two barriers one reads a whole step's operands from LDS (64 columns),
// asks for the rows of step s + NS - 1 and waits, while the other multiplies the
// step that it read in the slot before. Rows go from memory straight into LDS,
// their 16-byte pieces permuted by the row's number (as in tile_engine.h, whose
// rules for waits hold here too, a phase being such a step: what it read may be
// overwritten from the next one on, and what it waited for may be read from the
// next one on).
#include "parts.h"
#include "tile_engine.h"

namespace arks {

constexpr int MID_LDS = 160 * 1024;

// Stages of LDS: what fits, at most 5 (a workgroup's short run of K has not the
// steps for more: 4608 x 3584, 64 rows, 8 stages 11.2 us, 5 10.6).
constexpr int mid_stages(int qt, int ft) {
  return MID_LDS / ((32 * qt + 64 * ft) * 128) < 5
             ? MID_LDS / ((32 * qt + 64 * ft) * 128)
             : 5;
}

// Items of experts (moe_plan_kernel): {expert, first place, pairs, ..}; their
// places' pairs, of which top_k share a row of a (null: rows are places).
struct MidItems {
  const int4* __restrict__ items;
  const int* __restrict__ n_items;
  const int* __restrict__ perm;
  int64_t w_expert;
  int top_k;
  int expert_base;  // number of the first of these experts among all ranks'
};

// 1 KB of 8 rows into LDS, 16 B a lane, from step s of its offset. The weights
// are read once and pass the caches by (non-temporal): 64 rows x 37888 x 3584
// 51 -> 45 us, the rows of a stay there.
template <bool ONCE>
__device__ __forceinline__ void mid_load(const __amdgpu_buffer_rsrc_t& b,
                                         char* to, const uint32_t offset,
                                         const int s) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      b, (__attribute__((address_space(3))) char*)to, 16, offset,
      s * (TILE_K * 2), 0, ONCE ? 2 : 0);
}
template <int N>
__device__ __forceinline__ void mid_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void mid_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// ITEMS: the experts that rows chose. Jobs are (item, tile), an item being up to
// 64 * FT pairs of one expert, whose weights are so read once; workgroups go
// through them in turn. With plan and mix, us, here (the best of moe_gemm.hip):
// 128 experts of 2048 x 768, 8 per row: 16 rows 129 (133), 64 rows 197 (207),
// 200 rows 211 (235), 600 rows 233 (250); 8 experts of 4096 x 14336, 2 per row:
// 16 rows 425 (505), 200 rows 464 (591).
template <int QT, int FT, bool SILU, bool ITEMS>
__global__ __launch_bounds__(512, 2) void mid_gemm_kernel(
    void* __restrict__ out, const bf16* __restrict__ a,
    const bf16* __restrict__ w, const bf16* __restrict__ bias,
    const int m_rows, const int n_total, const int k_total,
    const int64_t a_stride, const int splits, const int parts,
    const int rotate, const MidItems of) {
  constexpr int NS = mid_stages(QT, FT);
  constexpr int W_ROWS = 32 * QT, COLS = SILU ? W_ROWS / 2 : W_ROWS;
  constexpr int STAGE = (W_ROWS + 64 * FT) * 128;
  constexpr int WL = (QT + 1) / 2;  // loads of weights a step, of waves 0 to 3
  constexpr bool ODD = QT % 2 != 0;  // waves 4 to 7 take one less
  static_assert(NS >= 3 && (NS - 2) * (WL + FT) < 64, "waits count to 63");
  __shared__ __attribute__((aligned(1024))) char lds[NS * STAGE];
  const int lane = threadIdx.x % WAVE_SIZE, lq = lane % 16, la = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int wm = wave / 4, wn = wave % 4;
  const int tiles = (n_total + COLS - 1) / COLS;
  const int jobs = tiles * (ITEMS ? *of.n_items : splits);
  const int all_steps = k_total / TILE_K;
  if (ITEMS && (int)blockIdx.x >= jobs) return;
  // where operand k of a fragment lies: 16 rows of 128 B, pieces permuted
  const int frag = lq * 128 + ((la ^ (lq & 7)) * 16);
  const int w_at = wm * QT * 2048 + frag;
  const int a_at = W_ROWS * 128 + wn * FT * 2048 + frag;

  // The column (of those of the tile) whose weight row stands at row `at` of a
  // wave's, so that a lane's sums are neighbours in the output: two fragments
  // make 8 columns a lane. SILU: sums 0 and 2 of a fragment are gate columns, 1
  // and 3 the up columns beside them.
  auto column = [&](const int at) {
    const int q = at / 16, i = at % 16, g = i / 4, r = i % 4;
    const bool paired = (q | 1) < QT;
    if constexpr (SILU)
      return paired ? q / 2 * 16 + 4 * g + 2 * (q & 1) + r / 2
                    : 8 * q + 2 * g + r / 2;
    else
      return paired ? q / 2 * 32 + 8 * g + 4 * (q & 1) + r : at;
  };

  // turn: the step that a job begins with (then on to the last, and from the
  // first): workgroups that read the same columns of rows a power of two apart
  // would all meet on a few memory channels (16 rows x 151936 x 2048 127 -> 102
  // us, x 57344 x 8192 164 -> 147). An expert's follows from its number and
  // the tile alone, not from the item: which item a pair is in depends on the
  // other rows of the step, and its order of sums must not.
  struct Job {
    int n0, split, s0, steps, turn;
    int expert, first, rows;
  };
  auto job = [&](const int j) {
    if constexpr (ITEMS) {
      const int4 it = of.items[j / tiles];
      const unsigned tile = j % tiles;
      const unsigned at = (unsigned)(of.expert_base + it.x) * tiles + tile;
      return Job{(int)tile * COLS, 0, 0, all_steps,
                 rotate ? (int)(at % (unsigned)all_steps) : 0,
                 it.x, it.y, it.z};
    }
    const unsigned split = j / tiles, n = splits;  // all_steps * n < 2^32
    const int s0 = all_steps * split / n;
    const int steps = all_steps * (split + 1) / n - s0;
    return Job{(int)(j % tiles) * COLS, (int)split, s0, steps,
               rotate ? (int)((unsigned)j % (unsigned)steps) : 0,
               0, 0, m_rows};
  };
  __amdgpu_buffer_rsrc_t wb, ab;
  uint32_t wo[WL], ao[FT];
  auto aim_rows = [&](const Job& b) {
#pragma unroll
    for (int j = 0; j < FT; ++j) {
      const int row = (wave + 8 * j) * 8 + lane / 8;
      uint32_t from = min(row, b.rows - 1);
      if (ITEMS && of.perm) {
        // the 8 rows' pairs are scalar loads: a vector load would be waited
        // for behind all of those that are under way (what lies up to 7 places
        // behind the last one is the plan's too, and not taken)
        const int base = min((wave + 8 * j) * 8, b.rows - 1);
        const int* at = of.perm + b.first + base;
        int pair = at[0];
#pragma unroll
        for (int i = 1; i < 8; ++i)
          pair = (int)from - base == i ? at[i] : pair;
        from = (uint32_t)pair / (uint32_t)of.top_k;
      }
      ao[j] = from * (uint32_t)(a_stride * 2) + tile_piece_a(row, lane);
    }
  };
  if (!ITEMS) aim_rows(job(blockIdx.x));
  auto aim = [&](const Job& b) {  // the loads at a job
    if (ITEMS) aim_rows(b);
    ab = tile_buffer(a + b.s0 * TILE_K +
                     (ITEMS && !of.perm ? b.first * a_stride : 0));
    wb = tile_buffer(w + (ITEMS ? b.expert * of.w_expert : 0) +
                     (int64_t)b.n0 * k_total + b.s0 * TILE_K);
#pragma unroll
    for (int j = 0; j < WL; ++j) {
      const int row = (wave + 8 * j) * 8 + lane / 8;
      const int half = row / (16 * QT), at = row % (16 * QT);
      const int col =
          min(half * (COLS / 2) + column(at), n_total - 1 - b.n0);
      wo[j] = (uint32_t)(col + (SILU && (at & 1) ? n_total : 0)) *
                  (uint32_t)(k_total * 2) +
              tile_piece_a(row, lane);
    }
  };
  auto column_step = [](const Job& b, const int s) {
    return s + b.turn < b.steps ? s + b.turn : s + b.turn - b.steps;
  };
  auto load_w = [&](const int b, const int s) {
#pragma unroll
    for (int j = 0; j < WL; ++j)
      if (!ODD || j + 1 < WL || wm == 0)
        mid_load<true>(wb, lds + b * STAGE + (wave + 8 * j) * 1024, wo[j], s);
  };
  auto load_a = [&](const int b, const int s) {
#pragma unroll
    for (int j = 0; j < FT; ++j)
      mid_load<false>(
          ab, lds + b * STAGE + W_ROWS * 128 + (wave + 8 * j) * 1024, ao[j], s);
  };
  // the loads of the next step are there: those of NS - 2 steps may be under
  // way behind them (`more`: so many were asked for)
  auto arrived = [&](const bool more) {
    if (!more) mid_wait<0>();
    else if (!ODD || wm == 0) mid_wait<(NS - 2) * (WL + FT)>();
    else mid_wait<(NS - 2) * (WL - 1 + FT)>();
  };
  auto prologue = [&](const Job& b) {
#pragma unroll
    for (int s = 0; s < NS - 1; ++s)
      if (s < b.steps) {
        load_w(s, column_step(b, s));
        load_a(s, column_step(b, s));
      }
  };

  // Up to 64 rows a chain of sums is 4 steps long, and those of 4 steps are added
  // up apart: the streamed products, which are the other choice there, add up
  // the shorter chains of several waves. 64 rows of 4608 x 3584 in 3 runs of K
  // err by 1.0e-7, in a chain per run by 2.0e-7 (streamed, 7 runs: 1.4e-7); it
  // takes 1.4 % longer over 60 sizes, in front of the multiplications (2.2 %
  // behind them). Library products, the other choice beyond, are one chain too.
  constexpr bool SETTLE = FT == 1;
  f32x4 acc[QT][FT], settled[SETTLE ? QT : 1];
  ushort8 wf[QT][2], af[FT][2];
  auto read = [&](const int b) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
      for (int q = 0; q < QT; ++q)
        wf[q][k] = *reinterpret_cast<const ushort8*>(
            lds + (b * STAGE + (w_at ^ (k * 64)) + q * 2048));
#pragma unroll
      for (int f = 0; f < FT; ++f)
        af[f][k] = *reinterpret_cast<const ushort8*>(
            lds + (b * STAGE + (a_at ^ (k * 64)) + f * 2048));
    }
  };
  auto mul = [&](const int s) {
    if constexpr (SETTLE) {
      if ((s & 3) == 0) {
#pragma unroll
        for (int q = 0; q < QT; ++q) {
          settled[q] += acc[q][0];
          acc[q][0] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
    }
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int q = 0; q < QT; ++q)
#pragma unroll
        for (int f = 0; f < FT; ++f)
          acc[q][f] = tile_mfma(wf[q][k], af[f][k], acc[q][f]);
    __builtin_amdgcn_s_setprio(0);
    mid_barrier();
  };

  int at = 0, to = NS - 1;  // the stages that are read and loaded
  auto load = [&](const Job& b, const int s) {
    load_w(to, column_step(b, s));
    load_a(to, column_step(b, s));
  };
  auto end_read = [&](const bool more) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    arrived(more);
    mid_barrier();
  };
  auto next_stage = [&] {
    at = at == NS - 1 ? 0 : at + 1;
    to = to == NS - 1 ? 0 : to + 1;
  };
  // The last steps of a job load the next job's first ones, where every job
  // has that many (16 rows x 151936 x 2048 in tiles of 64 134 -> 121 us).
  const bool chained = all_steps / splits >= NS - 1;
  int j = blockIdx.x;  // grid <= jobs
  Job now = job(j);
  aim(now);
  prologue(now);
  arrived(now.steps >= NS - 1);
  mid_barrier();
  if (wm == 1) mid_barrier();  // the second group runs one slot behind
  for (;;) {
#pragma unroll
    for (int q = 0; q < QT; ++q)
#pragma unroll
      for (int f = 0; f < FT; ++f) acc[q][f] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < (SETTLE ? QT : 1); ++q)
      settled[q] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int whole = max(0, now.steps - (NS - 1));
    for (int s = 0; s < whole; ++s) {
      read(at);
      load(now, s + NS - 1);  // into the stage that the last step read
      end_read(true);
      mul(s);
      next_stage();
    }
    j += gridDim.x;
    const bool more = j < jobs, ahead = more && chained;
    const Job next = more ? job(j) : now;
    if (ahead) aim(next);
    for (int s = whole; s < now.steps; ++s) {
      read(at);
      if (ahead) load(next, s - whole);
      end_read(ahead);
      mul(s);
      next_stage();
    }
    if constexpr (SETTLE) {
#pragma unroll
      for (int q = 0; q < QT; ++q) acc[q][0] += settled[q];
    }
    const int n0 = now.n0 + wm * (COLS / 2);
#pragma unroll
    for (int f = 0; f < FT; ++f) {
      const int m = (wn * FT + f) * 16 + lq;
      if (m >= now.rows) continue;
      const int64_t row = (int64_t)(now.first + m) * n_total;
      if constexpr (SILU) {
        bf16* to_row = reinterpret_cast<bf16*>(out) + row;
#pragma unroll
        for (int q = 0; q < QT; q += 2) {
          bf16 o[4];
#pragma unroll
          for (int x = 0; x < (q + 1 < QT ? 4 : 2); ++x)
            o[x] = float_to_bf16_bits(tile_silu_mul(
                acc[q + x / 2][f][x % 2 * 2], acc[q + x / 2][f][x % 2 * 2 + 1]));
          if (q + 1 < QT) {
            const int n = n0 + q * 8 + 4 * la;
            if (n < n_total)  // n_total % 8 == 0
              *reinterpret_cast<ushort4v*>(to_row + n) =
                  ushort4v{o[0], o[1], o[2], o[3]};
          } else {
            const int n = n0 + q * 8 + 2 * la;
            if (n < n_total)
              *reinterpret_cast<ushort2v*>(to_row + n) = ushort2v{o[0], o[1]};
          }
        }
      } else if (parts) {
        float* to_row = reinterpret_cast<float*>(out) +
                        (int64_t)now.split * m_rows * n_total + row;
#pragma unroll
        for (int q = 0; q < QT; ++q) {
          const int n = (q | 1) < QT ? n0 + q / 2 * 32 + 8 * la + 4 * (q & 1)
                                     : n0 + q * 16 + 4 * la;
          if (n < n_total) *reinterpret_cast<f32x4*>(to_row + n) = acc[q][f];
        }
      } else {
        bf16* to_row = reinterpret_cast<bf16*>(out) + row;
#pragma unroll
        for (int q = 0; q < QT; q += 2) {
          const int width = q + 1 < QT ? 8 : 4;
          const int n = n0 + q * 16 + width * la;
          if (n >= n_total) continue;  // n_total % 8 == 0
          bf16 o[8];
#pragma unroll
          for (int x = 0; x < width; ++x)
            o[x] = float_to_bf16_bits(
                acc[q + x / 4][f][x % 4] +
                (bias ? bf16_bits_to_float(bias[n + x]) : 0.f));
          if (q + 1 < QT)
            *reinterpret_cast<ushort8*>(to_row + n) =
                *reinterpret_cast<const ushort8*>(o);
          else
            *reinterpret_cast<ushort4v*>(to_row + n) =
                ushort4v{o[0], o[1], o[2], o[3]};
        }
      }
    }
    if (!more) break;
    now = next;
    if (!ahead) {
      if (wm == 0) mid_barrier();  // all reads are over
      at = 0, to = NS - 1;
      aim(now);
      prologue(now);
      arrived(now.steps >= NS - 1);
      mid_barrier();
      if (wm == 1) mid_barrier();
    }
  }
  if (wm == 0) mid_barrier();
}

}  // namespace arks

using namespace arks;

// out: bf16 [m, n], or (parts) fp32 [splits, m, n]; silu: w [2n, k], one
// split. qt: 16 * qt weight rows a wave, 2, 4 or 5; m <= 256; k % 64 == 0, at
// least one step of 64 a split; n % 8 == 0; rows of a and w on 16 bytes; all
// rows of a, and w (silu) or 160 rows of it, under 4 GiB.
extern "C" void arks_mid_gemm(void* out, const void* a, const void* w,
                              const void* bias, int m, int n, int k,
                              int64_t a_stride, int qt, int splits, int parts,
                              int silu, hipStream_t stream) {
  const int cols = silu ? 16 * qt : 32 * qt;
  const int jobs = (n + cols - 1) / cols * splits;
  // where all columns of a stay in an XCD's 4 MB of L2 (beyond: 200 rows of
  // 3584 x 18944 39 -> 48 us)
  const int rotate = (int64_t)m * k <= 1 << 20;
#define ARKS_MID(QT, FT, SILU)                                                 \
  hipLaunchKernelGGL((mid_gemm_kernel<QT, FT, SILU, false>),                   \
                     dim3(jobs < 256 ? jobs : 256), dim3(512), 0, stream, out, \
                     (const bf16*)a, (const bf16*)w, (const bf16*)bias, m, n,  \
                     k, a_stride, splits, parts, rotate, MidItems{})
#define ARKS_MID_S(QT, FT)                                                     \
  do {                                                                         \
    if (silu) ARKS_MID(QT, FT, true);                                          \
    else ARKS_MID(QT, FT, false);                                              \
  } while (0)
#define ARKS_MID_M(QT)                                                         \
  do {                                                                         \
    if (m <= 64) ARKS_MID_S(QT, 1);                                            \
    else if (m <= 128) ARKS_MID_S(QT, 2);                                      \
    else if (m <= 192) ARKS_MID_S(QT, 3);                                      \
    else ARKS_MID_S(QT, 4);                                                    \
  } while (0)
  if (qt == 2) ARKS_MID_M(2);
  else if (qt == 4) ARKS_MID_M(4);
  else ARKS_MID_M(5);
#undef ARKS_MID_M
#undef ARKS_MID_S
#undef ARKS_MID
}

// out [places, n]: the items' pairs (at most 64 * ft each) times their experts'
// weights, silu: [2n, k] each; n_items of the max_items items are there. k % 64
// == 0, n % 8 == 0; an expert's weights and (perm) all rows of a under 4 GiB; 7 ints
// behind the last of perm are there.
extern "C" void arks_mid_items(void* out, const void* a, const void* w,
                               const void* perm, const void* items,
                               const void* n_items, int64_t a_stride,
                               int64_t w_expert, int n, int k, int top_k,
                               int expert_base, int max_items, int ft, int silu,
                               hipStream_t stream) {
  const MidItems of{(const int4*)items, (const int*)n_items, (const int*)perm,
                    w_expert, top_k, expert_base};
  const int cols = silu ? 64 : 128;
  const int64_t jobs = (int64_t)((n + cols - 1) / cols) * max_items;
  const int grid = (int)(jobs < 256 ? jobs : 256);
#define ARKS_MID(QT, FT, SILU)                                                 \
  hipLaunchKernelGGL((mid_gemm_kernel<QT, FT, SILU, true>), dim3(grid),        \
                     dim3(512), 0, stream, out, (const bf16*)a,                \
                     (const bf16*)w, nullptr, 0, n, k, a_stride, 1, 0, 1, of)
  if (ft == 1 && silu) ARKS_MID(4, 1, true);
  else if (ft == 1) ARKS_MID(4, 1, false);
  else if (silu) ARKS_MID(4, 2, true);
  else ARKS_MID(4, 2, false);
#undef ARKS_MID
}
