// out[M, N] = a[M, K] . w[N, K]^T (+ bias), or silu(gate) * up of two such
// products, for up to 256 rows: steps that decode, short prompts.
//
// A few rows are bound by the weights' stream, 200 by it, the rows of a that
// every workgroup reads beside it, and the matrix cores (200 rows x 37888 x 3584
// are 40 us of weights at 6.8 TB/s and 39 us of matrix operations;
// tile_engine.h is for those that the cores alone bound, and stream_gemm.hip
// takes few rows of small weights, without sums for anyone to add). So all rows
// of a meet a weight row at once (it is read once), and the weights' rows are
// cut as finely as gives every CU one tile of them (or, for small products, one
// run of K: fp32 sums of the runs for the consumer to add).
//
// 4 waves multiply, one a SIMD, 2 along the weights x 2 along the rows of a: a
// wave holds 16 * QT weight rows x 16 * FT rows of a. 4 more waves only load:
// they go through the steps (64 columns) of all of the workgroup's jobs, NS
// ahead, whatever the others do, so that the end of a job (its stores, which the
// waits of a wave that also loads would count) does not hold up the stream. Rows
// go from memory straight into LDS, their 16-byte pieces permuted by the row's
// number (as in tile_engine.h). Rows of a are asked for in front of the weights:
// hits in L2 behind misses come as late as those do (200 rows x 37888 x 3584
// 61.8 -> 58.5 us), and 4 waves' loads are faster than 8 waves' (loads of 32 KB
// of a and 24 KB of weights a step, nothing else: 58 and 70 us in 56 steps).
//
// The ring and its waits: ring.h.
//
// us against the kernel before this one (8 waves that load and multiply in
// turns), weights cold: 37888 x 3584 with the activation, 8 rows 43.4 -> 42.3,
// 200 rows 63.5 -> 59.5; 3584 x 18944 in 8 runs of K, 64 rows 26.1 -> 25.3, 200
// rows 41.2 -> 37.5; 4608 x 3584 in 4, 8 rows 12.7 -> 9.7, 64 rows 14.5 -> 13.1;
// 152064 x 3584, 64 rows 201 -> 180, 200 rows 264 -> 247.
#include <type_traits>
#include "parts.h"
#include "ring.h"

namespace arks {

using u32x2 = __attribute__((ext_vector_type(2))) uint32_t;
using u32x4 = __attribute__((ext_vector_type(4))) uint32_t;
constexpr int MID_LDS = 160 * 1024;

// Stages of LDS: what fits, at most 6 (a workgroup's short run of K has not the
// steps for more).
constexpr int mid_stages(int qt, int ft) {
  return MID_LDS / ((32 * qt + 32 * ft) * 128) < 6
             ? MID_LDS / ((32 * qt + 32 * ft) * 128)
             : 6;
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

// The second of two products in one launch: a, w [n_total, k] of rows of its own,
// whose runs of K come behind the first one's `splits`.
struct MidPair {
  const bf16* __restrict__ a;
  const bf16* __restrict__ w;
  int64_t a_stride;
  int k_total;
  int splits;  // of the first product
};

// Lanes of neighbouring rows swap x of the odd row against y of the even one:
// a store then covers twice the columns of half the rows, whole lines.
template <typename V>
__device__ __forceinline__ void mid_swap(V& x, V& y, const bool odd) {
#pragma unroll
  for (int i = 0; i < (int)(sizeof(V) / 4); ++i) {
    const uint32_t give = odd ? x[i] : y[i];
    const uint32_t got = __builtin_amdgcn_mov_dpp(give, 0xB1, 0xF, 0xF, true);
    if (odd) x[i] = got;
    else y[i] = got;
  }
}

// Where stores go that begin below 2 GiB of p; those beyond are dropped.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t mid_out(void* p) {
  return __builtin_amdgcn_make_buffer_rsrc(p, 0, 0x80000000, 0x00027000);
}
// once: past the caches (non-temporal)
__device__ __forceinline__ void mid_store(const __amdgpu_buffer_rsrc_t& to,
                                          const uint32_t offset, const u32x4& v,
                                          const bool once) {
  if (once) __builtin_amdgcn_raw_buffer_store_b128(v, to, offset, 0, 2);
  else __builtin_amdgcn_raw_buffer_store_b128(v, to, offset, 0, 0);
}
__device__ __forceinline__ void mid_store(const __amdgpu_buffer_rsrc_t& to,
                                          const uint32_t offset, const u32x2& v,
                                          const bool once) {
  if (once) __builtin_amdgcn_raw_buffer_store_b64(v, to, offset, 0, 2);
  else __builtin_amdgcn_raw_buffer_store_b64(v, to, offset, 0, 0);
}

// ITEMS: the experts that rows chose. Jobs are (item, tile), an item being up to
// 32 * FT pairs of one expert, whose weights are so read once; workgroups go
// through them in turn (64 rows of 128 experts of 2048 x 768, 8 per row: gate and
// up 126 -> 123 us, down 71 -> 67 against the kernel before). Items of 32 are for
// up to 32 rows, where no expert has more pairs and a ring of half the rows goes
// round faster; their tiles may be of 32 * 2 weight rows, to fill the last round
// of tiles (with plan and mix, 128 experts of 2048 x 768, 8 per row: 7 rows 91.6
// us streamed, 93.3 in items of 64, 90.6 of 32, 86.1 with gate and up cut so).
//
// PAIR: two products a . w^T of different rows and K, with as many columns each, for
// a consumer that adds the sums of both: few rows of 16 to 34 million weights are
// over before the loads have come up to speed (8 rows of 4096 x 4096 take 8.6 us, at
// 3.9 TB/s), and two of them do so once (ops._pair_cut).
enum MidKind { MID_ONE, MID_ITEMS, MID_PAIR };
template <int QT, int FT, bool SILU, MidKind KIND>
__global__ __launch_bounds__(512, 2) void mid_gemm_kernel(
    void* __restrict__ out, const bf16* __restrict__ a,
    const bf16* __restrict__ w, const bf16* __restrict__ bias,
    const int m_rows, const int n_total, const int k_total,
    const int64_t a_stride, const int splits, const int parts,
    const int rotate, const MidItems of, const MidPair second) {
  constexpr bool ITEMS = KIND == MID_ITEMS, PAIR = KIND == MID_PAIR;
  constexpr int NS = mid_stages(QT, FT);
  constexpr int W_ROWS = 32 * QT, COLS = SILU ? W_ROWS / 2 : W_ROWS;
  constexpr int W_STAGE = W_ROWS * 128, STAGE = W_STAGE + 32 * FT * 128;
  constexpr int LOADS = QT + FT;  // of a step, of a wave that loads
  static_assert(NS >= 3);
  __shared__ __attribute__((aligned(1024))) char lds[NS * STAGE];
  const int lane = threadIdx.x % WAVE_SIZE, lq = lane % 16, la = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int tiles = (n_total + COLS - 1) / COLS;
  const int jobs = tiles * (ITEMS ? *of.n_items : splits);
  const int all_steps = k_total / TILE_K;
  if (ITEMS && (int)blockIdx.x >= jobs) return;

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
      return paired && !parts ? q / 2 * 32 + 8 * g + 4 * (q & 1) + r : at;
  };

  // turn: the step that a job begins with (then on to the last, and from the
  // first): workgroups that read the same columns of rows a power of two apart
  // would all meet on a few memory channels (16 rows x 151936 x 2048 127 -> 102
  // us, x 57344 x 8192 164 -> 147). An expert's follows from its number and
  // the column alone, in units of a tile of QT 4: not from the item, nor from the
  // tiles, which both depend on the other rows of the step. So a pair's sums are
  // the same bits in items of 32 and of 64, with tiles of any height (items of 128
  // and the streamed kernel of moe_gemm.hip add up in other chains).
  struct Job {
    int n0, split, s0, steps, turn;
    int expert, first, rows;
    bool other;  // of the second product
  };
  auto job = [&](const int j) {
    if constexpr (ITEMS) {
      const int4 it = of.items[j / tiles];
      constexpr unsigned UNIT = SILU ? 64 : 128;
      const unsigned n0 = j % tiles * COLS, units = (n_total + UNIT - 1) / UNIT;
      const unsigned at = (unsigned)(of.expert_base + it.x) * units + n0 / UNIT;
      return Job{(int)n0, 0, 0, all_steps,
                 rotate ? (int)(at % (unsigned)all_steps) : 0,
                 it.x, it.y, it.z, false};
    }
    if constexpr (PAIR) {
      const unsigned run = j / tiles;
      const bool other = run >= (unsigned)second.splits;
      const unsigned at = other ? run - second.splits : run;
      const unsigned n = other ? splits - second.splits : second.splits;
      const unsigned all = other ? second.k_total / TILE_K : all_steps;
      const int s0 = all * at / n, steps = all * (at + 1) / n - s0;
      return Job{(int)(j % tiles) * COLS, (int)run, s0, steps,
                 rotate ? (int)((unsigned)j % (unsigned)steps) : 0,
                 0, 0, m_rows, other};
    }
    const unsigned split = j / tiles, n = splits;  // all_steps * n < 2^32
    const int s0 = all_steps * split / n;
    const int steps = all_steps * (split + 1) / n - s0;
    return Job{(int)(j % tiles) * COLS, (int)split, s0, steps,
               rotate ? (int)((unsigned)j % (unsigned)steps) : 0,
               0, 0, m_rows, false};
  };
  if (wave >= 4) {
    const int own = wave % 4;
    __amdgpu_buffer_rsrc_t wb, ab;
    uint32_t wo[QT], ao[FT];
    auto aim = [&](const Job& b) {
      const int k = PAIR && b.other ? second.k_total : k_total;
      const int64_t stride = PAIR && b.other ? second.a_stride : a_stride;
      wb = tile_buffer((PAIR && b.other ? second.w : w) +
                       (ITEMS ? b.expert * of.w_expert : 0) +
                       (int64_t)b.n0 * k + b.s0 * TILE_K);
      ab = tile_buffer((PAIR && b.other ? second.a : a) + b.s0 * TILE_K +
                       (ITEMS && !of.perm ? b.first * stride : 0));
#pragma unroll
      for (int i = 0; i < QT; ++i) {
        const int row = (own + 4 * i) * 8 + lane / 8;
        const int side = row / (16 * QT), at = row % (16 * QT);
        const int col = min(side * (COLS / 2) + column(at), n_total - 1 - b.n0);
        wo[i] = (uint32_t)(col + (SILU && (at & 1) ? n_total : 0)) *
                    (uint32_t)(k * 2) +
                tile_piece_a(row, lane);
      }
#pragma unroll
      for (int i = 0; i < FT; ++i) {
        const int row = (own + 4 * i) * 8 + lane / 8;
        uint32_t r = min(row, b.rows - 1);
        if (ITEMS && of.perm) {
          // the 8 rows' pairs are scalar loads: a vector load would be waited
          // for behind all of those that are under way (what lies up to 7 places
          // behind the last one is the plan's too, and not taken)
          const int base = min((own + 4 * i) * 8, b.rows - 1);
          const int* at = of.perm + b.first + base;
          int pair = at[0];
#pragma unroll
          for (int k = 1; k < 8; ++k) pair = (int)r - base == k ? at[k] : pair;
          r = (uint32_t)pair / (uint32_t)of.top_k;
        }
        ao[i] = r * (uint32_t)(stride * 2) + tile_piece_a(row, lane);
      }
    };
    int total = 0;  // steps of all of this workgroup's jobs
    if (ITEMS || splits == 1)
      total = ((jobs - 1 - (int)blockIdx.x) / (int)gridDim.x + 1) * all_steps;
    else
      for (int j = blockIdx.x; j < jobs; j += gridDim.x) total += job(j).steps;
    int j = blockIdx.x, s = 0, stage = 0;
    Job b = job(j);
    aim(b);
    auto load = [&] {
      const int at = s + b.turn < b.steps ? s + b.turn : s + b.turn - b.steps;
      char* to = lds + stage * STAGE + own * 1024;
#pragma unroll
      for (int i = 0; i < FT; ++i)
        ring_load<false>(ab, to + W_STAGE + i * 4096, ao[i], at * (TILE_K * 2));
#pragma unroll
      for (int i = 0; i < QT; ++i)
        ring_load<true>(wb, to + i * 4096, wo[i], at * (TILE_K * 2));
      stage = stage == NS - 1 ? 0 : stage + 1;
      if (++s == b.steps) {
        s = 0;
        j += gridDim.x;
        if (j < jobs) {
          b = job(j);
          aim(b);
        }
      }
    };
    ring_feed<NS, LOADS>(total, load, [](int) {});
    return;
  }

  const int wm = wave / 2, wn = wave % 2;
  // where operand k of a fragment lies: 16 rows of 128 B, pieces permuted
  const int frag = lq * 128 + ((la ^ (lq & 7)) * 16);
  const int w_at = wm * QT * 2048 + frag;
  const int a_at = W_STAGE + wn * FT * 2048 + frag;
  // Up to 64 rows a chain of sums is 4 steps long, those of 4 steps are added up
  // apart, and those of 16 steps again (far): the streamed products, which are the
  // other choice there, add up the shorter chains of several waves, and the error
  // must not grow with the run of K that a cut gives. Relative to 64 bits, 8 rows,
  // chains of 4 steps in one chain -> in chains of 16: 5120 x 27648 in 3 runs
  // 1.45e-7 -> 1.17e-7 (in 8 runs 1.25e-7 before), 3584 x 18944 in 4 1.28e-7 ->
  // 1.12e-7 (in 8 1.20e-7 before), 10240 x 2048 in one 1.03e-7 -> 1.00e-7 (streamed
  // 0.98e-7); 64 rows of 4608 x 3584 in 3 runs err by 1.0e-7, in a chain per run by
  // 2.0e-7.
  // Both together take 0.3 % longer than one chain over 100 sizes and numbers of rows
  // (far as values that are chosen, and not as a branch, 3 %).
  // Library products, the other choice beyond, are one chain; there
  // ops._mid_cut keeps runs short. An expert's items have one run each, as before.
  constexpr bool SETTLE = FT <= 2, FAR = SETTLE && !ITEMS;
  f32x4 acc[QT][FT], settled[SETTLE ? QT : 1][FT], far[FAR ? QT : 1][FT];
  // The fragments of the next half step are read while this one's are
  // multiplied: those of w and the last two of a into a second set of
  // registers, the others into the same once they have been used.
  constexpr int TWO = FT < 2 ? FT : 2;
  ushort8 wf[2][QT], af[FT], al[2][TWO];
  int at = 0;  // the stage that is read
  auto read_w = [&](const int half, const int q) {
    wf[half][q] = *reinterpret_cast<const ushort8*>(
        lds + (at * STAGE + (w_at ^ (half * 64)) + q * 2048));
  };
  auto read_a = [&](const int half, const int f) {
    const ushort8 v = *reinterpret_cast<const ushort8*>(
        lds + (at * STAGE + (a_at ^ (half * 64)) + f * 2048));
    if (f >= FT - TWO) al[half][f - (FT - TWO)] = v;
    else af[f] = v;
  };
  auto half_step = [&](auto which) {
    constexpr int H = decltype(which)::value;
#pragma unroll
    for (int q = 0; q < QT; ++q) read_w(H ^ 1, q);
#pragma unroll
    for (int f = FT - TWO; f < FT; ++f) read_a(H ^ 1, f);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int f = 0; f < FT; ++f) {
#pragma unroll
      for (int q = 0; q < QT; ++q)
        acc[q][f] = tile_mfma(
            wf[H][q], f >= FT - TWO ? al[H][f - (FT - TWO)] : af[f], acc[q][f]);
      if (f < FT - TWO) {
        __builtin_amdgcn_sched_barrier(0);
        read_a(H ^ 1, f);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  int j = blockIdx.x;  // grid <= jobs
  Job now = job(j);
  ring_barrier();
  for (;;) {
#pragma unroll
  for (int q = 0; q < QT; ++q) read_w(0, q);
#pragma unroll
  for (int f = 0; f < FT; ++f) read_a(0, f);
#pragma unroll
    for (int q = 0; q < QT; ++q)
#pragma unroll
      for (int f = 0; f < FT; ++f) {
        acc[q][f] = f32x4{0.f, 0.f, 0.f, 0.f};
        if constexpr (SETTLE) settled[q][f] = f32x4{0.f, 0.f, 0.f, 0.f};
        if constexpr (FAR) far[q][f] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    for (int s = 0; s < now.steps; ++s) {
      if constexpr (SETTLE) {
        if ((s & 3) == 0) {
#pragma unroll
          for (int q = 0; q < QT; ++q)
#pragma unroll
            for (int f = 0; f < FT; ++f) {
              settled[q][f] += acc[q][f];
              acc[q][f] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
          if constexpr (FAR) {
            if ((s & 15) == 0 && s > 0) {
              asm volatile("");  // a branch
#pragma unroll
              for (int q = 0; q < QT; ++q)
#pragma unroll
                for (int f = 0; f < FT; ++f) {
                  far[q][f] += settled[q][f];
                  settled[q][f] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
            }
          }
        }
      }
      half_step(std::integral_constant<int, 0>{});
      // this step has been read, the next one is there
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      ring_barrier();
      at = at == NS - 1 ? 0 : at + 1;
      half_step(std::integral_constant<int, 1>{});
    }
    j += gridDim.x;
    const bool more = j < jobs;
    if constexpr (SETTLE) {
#pragma unroll
      for (int q = 0; q < QT; ++q)
#pragma unroll
        for (int f = 0; f < FT; ++f) {
          acc[q][f] += settled[q][f];
          if constexpr (FAR) acc[q][f] += far[q][f];
        }
    }
    const int n0 = now.n0 + wm * (COLS / 2);
#pragma unroll
    for (int f = 0; f < FT; ++f) {
      const int m0 = (wn * FT + f) * 16;
      if (m0 >= now.rows) break;
      // (worked out anew for each f, or they would fill the registers)
      int lq = lane % 16, la = lane / 16;
      asm volatile("" : "+v"(lq), "+v"(la));
      const bool odd = lq & 1;
      const int64_t row0 = (int64_t)(now.first + m0) * n_total + n0;
      if constexpr (SILU) {
        if (m0 + lq >= now.rows) continue;
        bf16* to_row = reinterpret_cast<bf16*>(out) + row0 + lq * n_total - n0;
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
      } else {
        // Pieces of 16 bytes, of two rows at a time: stores that begin at `none`
        // are not made. n_total % 8 == 0.
        constexpr uint32_t none = 1u << 31;
        // Past the caches beside the loads of other jobs, from 17 rows on: the
        // output's lines do not push out those of a (152064 x 3584, 64 rows 197
        // -> 178 us, 32 rows 179 -> 171; 8 rows 163 -> 166; 128256 x 2048, 256
        // rows 152 -> 145). Waves of 80 columns (QT 5) store parts of lines, which
        // is slower past the caches, so there only as long as the output is little
        // beside the weights: us, past the caches (not), 151936 x 896, 48 rows 56.9
        // (56.6), 64 rows 61.6 (59.2), 192 rows 95.2 (86.0); x 2048, 96 rows 124
        // (129), 192 rows 158 (154); 100352 x 2560, 128 rows 124.7 (125.1), 192
        // rows 143.7 (139.0); 152064 x 3584, 160 rows 241.7 (240.5), 224 rows 274
        // (261). Not sums: whoever adds them would read them from memory (64 rows x
        // 3584 and their norm 5.0 -> 5.4 us, 200 rows 7.4 -> 8.5).
        const bool once = jobs > (int)gridDim.x && now.rows > 16 &&
                          (QT % 4 == 0 || now.rows * 19 < k_total);
        const uint32_t size = parts ? 4 : 2;
        const uint32_t even = m0 + (lq & ~1) < now.rows
                                  ? (lq & ~1) * n_total * size : none;
        const uint32_t odds = m0 + (lq | 1) < now.rows
                                  ? (lq | 1) * n_total * size : none;
        const uint32_t own = odd ? odds : even;
        auto at = [&](const uint32_t row, const int n) {
          return n0 + n < n_total && row != none ? row + n * size : none;
        };
        if (parts) {
          const auto to = mid_out(reinterpret_cast<float*>(out) +
                                  (int64_t)now.split * m_rows * n_total + row0);
#pragma unroll
          for (int q = 0; q + 1 < QT; q += 2) {
            u32x4 x = *reinterpret_cast<const u32x4*>(&acc[q][f]);
            u32x4 y = *reinterpret_cast<const u32x4*>(&acc[q + 1][f]);
            mid_swap(x, y, odd);
            const int n = q * 16 + 4 * la + (odd ? 16 : 0);
            mid_store(to, at(even, n), x, false);
            mid_store(to, at(odds, n), y, false);
          }
          if constexpr (QT % 2)
            mid_store(to, at(own, (QT - 1) * 16 + 4 * la),
                      *reinterpret_cast<const u32x4*>(&acc[QT - 1][f]), false);
        } else {
          const auto to = mid_out(reinterpret_cast<bf16*>(out) + row0);
          const bf16* add = bias;
          asm volatile("" : "+s"(add));  // its values are not kept in registers
          auto value = [&](const int q, const int n) {
            const bf16* b = add + min(n0 + n, n_total - 8);
            bf16 o[8];
#pragma unroll
            for (int x = 0; x < 8; ++x)
              o[x] = float_to_bf16_bits(acc[q + x / 4][f][x % 4] +
                                        (add ? bf16_bits_to_float(b[x]) : 0.f));
            return *reinterpret_cast<const u32x4*>(o);
          };
#pragma unroll
          for (int q = 0; q + 3 < QT; q += 4) {
            const int n = q * 16 + 8 * la;
            u32x4 x = value(q, n), y = value(q + 2, n + 32);
            mid_swap(x, y, odd);
            mid_store(to, at(even, n + (odd ? 32 : 0)), x, once);
            mid_store(to, at(odds, n + (odd ? 32 : 0)), y, once);
          }
#pragma unroll
          for (int q = QT / 4 * 4; q + 1 < QT; q += 2)
            mid_store(to, at(own, q * 16 + 8 * la), value(q, q * 16 + 8 * la),
                      once);
          if constexpr (QT % 2) {
            const int n = (QT - 1) * 16 + 4 * la;
            bf16 o[4];
#pragma unroll
            for (int x = 0; x < 4; ++x)
              o[x] = float_to_bf16_bits(
                  acc[QT - 1][f][x] +
                  (add ? bf16_bits_to_float(add[min(n0 + n, n_total - 4) + x])
                       : 0.f));
            mid_store(to, at(own, n), *reinterpret_cast<const u32x2*>(o), once);
          }
        }
      }
    }
    if (!more) break;
    now = job(j);
  }
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
  hipLaunchKernelGGL((mid_gemm_kernel<QT, FT, SILU, MID_ONE>),                 \
                     dim3(jobs < 256 ? jobs : 256), dim3(512), 0, stream, out, \
                     (const bf16*)a, (const bf16*)w, (const bf16*)bias, m, n,  \
                     k, a_stride, splits, parts, rotate, MidItems{},           \
                     MidPair{})
#define ARKS_MID_S(QT, FT)                                                     \
  do {                                                                         \
    if (silu) ARKS_MID(QT, FT, true);                                          \
    else ARKS_MID(QT, FT, false);                                              \
  } while (0)
#define ARKS_MID_M(QT)                                                         \
  do {                                                                         \
    if (m <= 32) ARKS_MID_S(QT, 1);                                            \
    else if (m <= 64) ARKS_MID_S(QT, 2);                                       \
    else if (m <= 96) ARKS_MID_S(QT, 3);                                      \
    else if (m <= 128) ARKS_MID_S(QT, 4);                                      \
    else if (m <= 160) ARKS_MID_S(QT, 5);                                      \
    else if (m <= 192) ARKS_MID_S(QT, 6);                                      \
    else if (m <= 224) ARKS_MID_S(QT, 7);                                      \
    else ARKS_MID_S(QT, 8);                                                    \
  } while (0)
  if (qt == 2) ARKS_MID_M(2);
  else if (qt == 4) ARKS_MID_M(4);
  else ARKS_MID_M(5);
#undef ARKS_MID_M
#undef ARKS_MID_S
#undef ARKS_MID
}

// out: fp32 [splits + splits2, m, n], the sums of a . w^T in runs of k and behind
// them those of a2 . w2^T in runs of k2; m <= 64, the other conditions of
// arks_mid_gemm for both.
extern "C" void arks_mid_pair(void* out, const void* a, const void* w, int k,
                              int64_t a_stride, int splits, const void* a2,
                              const void* w2, int k2, int64_t a_stride2,
                              int splits2, int m, int n, int qt,
                              hipStream_t stream) {
  const int jobs = (n + 32 * qt - 1) / (32 * qt) * (splits + splits2);
  const int rotate = (int64_t)m * (k + k2) <= 1 << 20;
  const MidPair second{(const bf16*)a2, (const bf16*)w2, a_stride2, k2, splits};
#define ARKS_MID(QT, FT)                                                       \
  hipLaunchKernelGGL((mid_gemm_kernel<QT, FT, false, MID_PAIR>),               \
                     dim3(jobs < 256 ? jobs : 256), dim3(512), 0, stream, out, \
                     (const bf16*)a, (const bf16*)w, nullptr, m, n, k,         \
                     a_stride, splits + splits2, 1, rotate, MidItems{}, second)
#define ARKS_MID_M(QT)                                                         \
  do {                                                                         \
    if (m <= 32) ARKS_MID(QT, 1);                                              \
    else ARKS_MID(QT, 2);                                                      \
  } while (0)
  if (qt == 2) ARKS_MID_M(2);
  else if (qt == 4) ARKS_MID_M(4);
  else ARKS_MID_M(5);
#undef ARKS_MID_M
#undef ARKS_MID
}

// out [places, n]: the items' pairs (at most 32 * ft each, ft 1, 2 or 4) times
// their experts' weights, silu: [2n, k] each; n_items of the max_items items are
// there. qt: 16 * qt weight rows a wave, 4, or (ft 1) 2. k % 64 == 0, n % 8 == 0;
// an expert's weights and (perm) all rows of a under 4 GiB; 7 ints behind the
// last of perm are there.
extern "C" void arks_mid_items(void* out, const void* a, const void* w,
                               const void* perm, const void* items,
                               const void* n_items, int64_t a_stride,
                               int64_t w_expert, int n, int k, int top_k,
                               int expert_base, int max_items, int ft, int qt,
                               int silu, hipStream_t stream) {
  const MidItems of{(const int4*)items, (const int*)n_items, (const int*)perm,
                    w_expert, top_k, expert_base};
  const int cols = silu ? 16 * qt : 32 * qt;
  const int64_t jobs = (int64_t)((n + cols - 1) / cols) * max_items;
  const int grid = (int)(jobs < 256 ? jobs : 256);
#define ARKS_MID(QT, FT, SILU)                                                 \
  hipLaunchKernelGGL((mid_gemm_kernel<QT, FT, SILU, MID_ITEMS>), dim3(grid),   \
                     dim3(512), 0, stream, out, (const bf16*)a,                \
                     (const bf16*)w, nullptr, 0, n, k, a_stride, 1, 0, 1, of,  \
                     MidPair{})
#define ARKS_MID_S(QT, FT)                                                     \
  do {                                                                         \
    if (silu) ARKS_MID(QT, FT, true);                                          \
    else ARKS_MID(QT, FT, false);                                              \
  } while (0)
  if (ft == 1 && qt == 2) ARKS_MID_S(2, 1);
  else if (ft == 1) ARKS_MID_S(4, 1);
  else if (ft == 2) ARKS_MID_S(4, 2);
  else ARKS_MID_S(4, 4);
#undef ARKS_MID_S
#undef ARKS_MID
}
