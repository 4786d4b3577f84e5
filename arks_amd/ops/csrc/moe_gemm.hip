// Sparse expert feed-forward (gfx950): the (row, expert) pairs of a step run
// only the experts that they chose, without a host read of the routing.
//
//   moe_plan   pairs sorted by expert, cut into items of one expert and at
//              most `tile` pairs; every pair's place in the sorted order
//   moe_stream less than one pair per expert on the mean (from there on
//              mid_gemm.hip takes sizes of whole steps of 64 with columns for
//              the chip; others are streamed up to 8): bound by the stream of
//              the chosen experts' weights. Tiles of 16 weight rows (gate and
//              up rows side by side), the waves of a workgroup splitting K, no
//              LDS and no barrier before the final sum over the waves. 7 rows,
//              8 of 128 experts each (2048 x 768): 90 us for 46 experts' 434 MB
//              (4.8 TB/s); every expert as a batched product took 210 us.
//   moe_engine 32 and more pairs per expert on the mean (fewer tiles than CUs:
//              more than 64, ops._moe_engine): bound by the matrix cores, and by
//              the weights' one read while experts have few. Up to 320, 256 or
//              192 pairs (moe_cut) x 256 weight rows per workgroup
//              (wide_engine.h). 128 experts of 2048 x 768, 8 per row, with
//              plan: 5012 rows 452 us, 520 rows 218 us for 1.2 GB of weights; 8
//              experts of 4096 x 14336, 2 per row, 8192 rows 4.55 ms.
//   moe_tile   the same for sizes that are no multiple of 64, or leave the
//              engine without work for the chip: 128 pairs x 128 weight rows, 64
//              of K per step through double-buffered LDS and registers, 560
//              TFLOP/s.
//
// Both products exist as "up" (rows gathered by pair, silu(gate) * up in fp32
// before the one rounding) and "down". Weights lie as in checkpoints,
// [expert, out, in]: a lane reads 16 bytes along K, as the MFMA operands
// want them. Items past the last one are empty, so grids depend on the shapes
// alone and a decode step can be captured.
#include <type_traits>
#include "moe_topk.h"
#include "seq_common.h"
#include "wide_engine.h"

namespace arks {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int MOE_MAX_E = 1024;

__device__ __forceinline__ float moe_bf16(const float v) {
  return bf16_bits_to_float(float_to_bf16_bits(v));
}

__device__ __forceinline__ f32x4 moe_mfma(const ushort8& a, const ushort8& b,
                                          f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
      *reinterpret_cast<const bf16x8*>(&a), *reinterpret_cast<const bf16x8*>(&b),
      c, 0, 0, 0);
}

// perm[place] = pair, rows[pair] = place (0 where the expert is another
// rank's), weights_out[pair] = the pair's weight (0 there), items[i] = {local
// expert, first place, pairs, number within the expert | items of the expert
// << 16}, n_items; claims[16] = 0 (moe_engine's).
// Bound by the serial work of a workgroup (two LDS atomics and five accesses a
// pair), so many pairs are spread over workgroups in two launches: STAGE 1
// counts a workgroup's run of pairs per expert into counts[group][expert],
// STAGE 2 places it behind the runs before it. STAGE 0: one workgroup does
// both. 40096 pairs of 128 experts 46.9 -> 10.6 us, 131072 of 512 experts 166
// -> 16; the runs' length hardly matters (512 to 4096 pairs: 11.8 to 10.6).
// TOPK (STAGE 0, of up to MOE_TOPK_PAIRS pairs): ids and weights are found here, from
// the rows' logits [rows, experts <= 64 * TOPK], a wave a row: a launch less, while
// rows are few (ops._PLAN_ROWS).
struct MoeLogits {
  const float* __restrict__ logits;
  int experts, k, renorm;
};
constexpr int MOE_TOPK_PAIRS = 512;
// Tiles of weight rows and steps of 64 columns of the experts' two products (the
// engine's; moe_cut).
struct MoeRounds {
  int up_tiles, down_tiles, up_steps, down_steps;
};
// How many pairs the items of moe_engine may have, 320, 256 or 192, for the counts
// that the plan finds (a wave's work): items are work for 256 CUs in rounds, and a tile
// takes as long as on the mean (moe_engine: 0.5 and 0.21 for each 64 pairs). us, 320
// (256; 192), 16 experts of 4096 x 2048, 2 per row: 2000 rows 247 (325; 268), 2250 rows
// 331 (301; 354), 2500 rows 327 (314; 293); 16 of 4096 x 3584, 4 per row: 1000 rows 398
// (493; 464), 1300 rows 583 (533; 565); 32 of 2048 x 1024, 4 per row, 1700 rows 198
// (176; 166). Over 77 sizes the choice takes 1.004 of the best, always 320 1.026. It
// is 0.7 us of the plan. Against tiles of 256 pairs and of 128 for what is left, in
// tile_engine.h's loop, 79 sizes take 0.956, in the worst 8 experts of 4096 x 14336, 2
// per row, 3000 rows 1801 (1684) and 16 of 4096 x 2048, 5000 rows 513 (469).
__device__ __forceinline__ int moe_cut(const MoeRounds& r, const int* count,
                                       const int n_local, const int pairs) {
  int sum[4] = {};
  for (int e = threadIdx.x; e < n_local; e += WAVE_SIZE) {
    const int c = count[e];
    sum[0] += (c + 319) / 320;
    sum[1] += (c + 255) / 256;
    sum[2] += (c + 191) / 192;
    sum[3] += (c + 63) / 64;
  }
#pragma unroll
  for (int off = 1; off < WAVE_SIZE; off <<= 1)
#pragma unroll
    for (int j = 0; j < 4; ++j) sum[j] += __shfl_xor(sum[j], off, WAVE_SIZE);
  float best = INFINITY;
  int cap = 320;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const float n = fmaxf((float)sum[j], 1.f);
    const float time = (r.up_steps * ceilf(n * r.up_tiles / 256.f) +
                        r.down_steps * ceilf(n * r.down_tiles / 256.f)) *
                       (0.5f + 0.21f * sum[3] / n);
    // (an item's number within its expert has 15 bits)
    if (time < best && (j < 2 || pairs < 1 << 22)) {
      best = time;
      cap = 320 - 64 * j;
    }
  }
  return cap;
}
template <int STAGE, int TOPK = 0>
__global__ __launch_bounds__(1024) void moe_plan_kernel(
    int* __restrict__ perm, int* __restrict__ rows,
    float* __restrict__ weights_out, int4* __restrict__ items,
    int* __restrict__ n_items, int* __restrict__ claims,
    int* __restrict__ counts, const int* __restrict__ ids,
    const float* __restrict__ weights, const int pairs, const int expert_base,
    const int n_local, const int tile, const int max_items,
    const MoeLogits route, const MoeRounds rounds) {
  __shared__ int chosen[TOPK ? MOE_TOPK_PAIRS : 1];
  __shared__ float chosen_w[TOPK ? MOE_TOPK_PAIRS : 1];
  auto id_of = [&](const int p) { return TOPK ? chosen[TOPK ? p : 0] : ids[p]; };
  auto weight_of = [&](const int p) {
    return TOPK ? chosen_w[TOPK ? p : 0] : weights[p];
  };
  if constexpr (TOPK > 0) {
    const int lane = threadIdx.x % WAVE_SIZE;
    for (int t = threadIdx.x / WAVE_SIZE; t < pairs / route.k;
         t += 1024 / WAVE_SIZE) {
      float w;
      int id;
      moe_topk_row<TOPK>(route.logits + (int64_t)t * route.experts, route.experts,
                         route.k, route.renorm, lane, w, id);
      if (lane < route.k) {
        chosen[t * route.k + lane] = id;
        chosen_w[t * route.k + lane] = w;
      }
    }
    // (the barrier behind the counters' clearing stands in front of their use)
  }
  __shared__ int count[MOE_MAX_E], start[MOE_MAX_E], first_item[MOE_MAX_E];
  __shared__ int total_items, item_cap;
  const int tid = threadIdx.x;
  const int group = STAGE == 0 ? 0 : (int)blockIdx.x;
  const int groups = STAGE == 0 ? 1 : (int)gridDim.x;
  const int per = (pairs + groups - 1) / groups;
  const int begin = group * per, end = min(pairs, begin + per);
  constexpr int PB = 8;  // loads in flight per thread
  if constexpr (STAGE != 2) {
    for (int e = tid; e < n_local; e += 1024) count[e] = 0;
    __syncthreads();
    for (int p0 = begin + tid; p0 < end; p0 += 1024 * PB) {
      int e[PB];
#pragma unroll
      for (int j = 0; j < PB; ++j)
        e[j] = p0 + j * 1024 < end ? id_of(p0 + j * 1024) - expert_base : -1;
#pragma unroll
      for (int j = 0; j < PB; ++j)
        if (e[j] >= 0 && e[j] < n_local) atomicAdd(&count[e[j]], 1);
    }
    __syncthreads();
    if constexpr (STAGE == 1) {
      for (int e = tid; e < n_local; e += 1024)
        counts[group * n_local + e] = count[e];
      return;
    }
  }
  int before = 0;  // of this thread's expert (n_local <= 1024), in earlier runs
  if constexpr (STAGE == 2) {
    if (tid < n_local) {
      int all = 0;
      for (int g0 = 0; g0 < groups; g0 += PB) {
        int c[PB];
#pragma unroll
        for (int j = 0; j < PB; ++j)
          c[j] = g0 + j < groups ? counts[(g0 + j) * n_local + tid] : 0;
#pragma unroll
        for (int j = 0; j < PB; ++j) {
          all += c[j];
          if (g0 + j < group) before += c[j];
        }
      }
      count[tid] = all;
    }
    __syncthreads();
  }
  if (tid < WAVE_SIZE) {  // prefix sums, 64 experts at a time
    int at = 0, item = 0, cap = tile;
    if (tile > 256) cap = moe_cut(rounds, count, n_local, pairs);
    if (tid == 0) item_cap = cap;
    for (int e0 = 0; e0 < n_local; e0 += WAVE_SIZE) {
      const int e = e0 + tid;
      const int c = e < n_local ? count[e] : 0;
      const int n = (c + cap - 1) / cap;
      int sc = c, sn = n;
#pragma unroll
      for (int off = 1; off < WAVE_SIZE; off <<= 1) {
        const int vc = __shfl_up(sc, off, WAVE_SIZE);
        const int vn = __shfl_up(sn, off, WAVE_SIZE);
        if (tid >= off) {
          sc += vc;
          sn += vn;
        }
      }
      if (e < n_local) {
        start[e] = at + sc - c;
        first_item[e] = item + sn - n;
      }
      at += __shfl(sc, WAVE_SIZE - 1, WAVE_SIZE);
      item += __shfl(sn, WAVE_SIZE - 1, WAVE_SIZE);
    }
    if (tid == 0) total_items = item;
  }
  __syncthreads();
  if (group == 0) {
    if (tid < 16) claims[tid] = 0;
    if (tid == 0) *n_items = total_items;
    const int cap = item_cap;
    for (int e = tid; e < n_local; e += 1024) {
      const int c = count[e];
      const int n = (c + cap - 1) / cap;
      // (8 experts of 4096 x 14336, 2 per row, 2048 rows 1529 us with items of 320
      // and what is left, even 1448)
      const int per = tile > 256 && n ? ((c + n - 1) / n + 63) / 64 * 64 : tile;
      for (int i = 0; i < n; ++i)
        items[first_item[e] + i] = make_int4(
            e, start[e] + i * per, min(per, c - i * per), i | n << 16);
    }
    for (int i = total_items + tid; i < max_items; i += 1024)
      items[i] = make_int4(0, 0, 0, 0);
  }
  __syncthreads();
  // from here on: places given out
  for (int e = tid; e < n_local; e += 1024) count[e] = before;
  __syncthreads();
  for (int p0 = begin + tid; p0 < end; p0 += 1024 * PB) {
    int e[PB];
    float w[PB];
#pragma unroll
    for (int j = 0; j < PB; ++j) {
      const int p = min(p0 + j * 1024, end - 1);
      e[j] = id_of(p) - expert_base;
      w[j] = weight_of(p);
    }
#pragma unroll
    for (int j = 0; j < PB; ++j) {
      const int p = p0 + j * 1024;
      if (p >= end) break;
      const bool mine = e[j] >= 0 && e[j] < n_local;
      int place = 0;
      if (mine) {
        place = start[e[j]] + atomicAdd(&count[e[j]], 1);
        perm[place] = p;
      }
      rows[p] = place;
      weights_out[p] = mine ? w[j] : 0.f;
    }
  }
}

// Weight rows [n0, n0 + 16 * NF) of one item's expert (UP: 16 gate rows and
// their 16 up rows) times its up to 16 pairs; a grid of (row tiles, items). Waves take the 64-wide chunks of K in turn, two chunks of loads in
// flight each, and sum through LDS in a fixed order.
template <int NF, int WV, bool UP>
__global__ __launch_bounds__(WV * 64) void moe_stream_kernel(
    bf16* __restrict__ out,        // [pairs, n_out]
    const bf16* __restrict__ a,    // UP: [T, K] by pair / k; else [pairs, K]
    const bf16* __restrict__ w,    // expert e's rows at w + e * w_expert
    const int* __restrict__ perm, const int4* __restrict__ items,
    const int64_t a_stride, const int64_t w_expert, const int64_t w_stride,
    const int n_out, const int k_total, const int top_k) {
  const int4 item = items[blockIdx.y];
  const int cnt = item.z;
  if (cnt == 0) return;
  __shared__ f32x4 red[WV][NF][WAVE_SIZE];
  const int lane = threadIdx.x % WAVE_SIZE, lq = lane % 16, la = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int n0 = blockIdx.x * (UP ? 16 : 16 * NF);
  const int nch = k_total / 64;
  f32x4 acc[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bf16* wp[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f)
    wp[f] = w + (int64_t)item.x * w_expert +
            (int64_t)(UP ? f * n_out + n0 + lq : n0 + f * 16 + lq) * w_stride +
            8 * la + wave * 64;
  const int place = item.y + min(lq, cnt - 1);
  const bf16* ap = a + (int64_t)(UP ? perm[place] / top_k : place) * a_stride +
                   8 * la + wave * 64;
  struct Chunk {
    ushort8 w[NF][2], a[2];
  };
  auto load = [&](Chunk& c, int i, int halves) {
    const int64_t o = (int64_t)i * WV * 64;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (h >= halves) break;
#pragma unroll
      for (int f = 0; f < NF; ++f)
        c.w[f][h] = *reinterpret_cast<const ushort8*>(wp[f] + o + 32 * h);
      c.a[h] = *reinterpret_cast<const ushort8*>(ap + o + 32 * h);
    }
  };
  auto mul = [&](Chunk& c, int halves) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (h >= halves) break;
#pragma unroll
      for (int f = 0; f < NF; ++f)
        acc[f] = moe_mfma(c.w[f][h], c.a[h], acc[f]);
    }
  };
  const int own = (nch - wave + WV - 1) / WV;
  if (own > 0) {
    Chunk c0, c1;
    load(c0, 0, 2);
    if (own > 1) load(c1, 1, 2);
    int i = 0;
    for (; i + 3 < own; i += 2) {
      mul(c0, 2);
      load(c0, i + 2, 2);
      mul(c1, 2);
      load(c1, i + 3, 2);
    }
    const int left = own - i;
    mul(c0, 2);
    if (left > 2) load(c0, i + 2, 2);
    if (left > 1) mul(c1, 2);
    if (left > 2) mul(c0, 2);
  }
  if (k_total % 64 != 0 && wave == nch % WV) {  // half a chunk behind the last
    Chunk c;
    load(c, nch / WV, 1);
    mul(c, 1);
  }
#pragma unroll
  for (int f = 0; f < NF; ++f) red[wave][f][lane] = acc[f];
  __syncthreads();
  auto total = [&](int x) {
    f32x4 s = red[0][x][lane];
#pragma unroll
    for (int v = 1; v < WV; ++v) s += red[v][x][lane];
    return s;
  };
  for (int f = wave; f < (UP ? 1 : NF); f += WV) {
    f32x4 s = total(f);
    if (UP) {
      const f32x4 u = total(1);
#pragma unroll
      for (int r = 0; r < 4; ++r) s[r] = tile_silu_mul(s[r], u[r]);
    }
    if (lq < cnt) {
      ushort4v o;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = float_to_bf16_bits(s[r]);
      *reinterpret_cast<ushort4v*>(out + (int64_t)(item.y + lq) * n_out + n0 +
                                   f * 16 + 4 * la) = o;
    }
  }
}

// 128 pairs of one expert x 128 weight rows (UP: 64 gate rows and their 64 up
// rows). 4 waves of 64 x 64; the next 64 of K travel through registers while
// the present ones are multiplied out of LDS (rows padded by 16 B: reads and
// writes without conflicts). Workgroups go round the 8 XCDs in launch order:
// each XCD takes a contiguous stretch of (item, row tile) so that its L2 holds
// an item's rows and its expert's weights.
constexpr int MT_BM = 128, MT_BN = 128, MT_BK = 64, MT_LS = MT_BK + 8;

// First of the 8 columns of a row that a lane loads for the step at k0: its
// own, or the row's first ones where K ends before them (they count as zero).
__host__ __device__ constexpr int moe_stage_column(int k0, int sc, int k_total) {
  return k0 + sc < k_total ? k0 + sc : 0;
}
constexpr bool moe_stage_columns_in_rows() {
  for (int k = 8; k <= 4 * MT_BK; k += 8)
    for (int k0 = 0; k0 < k; k0 += MT_BK)
      for (int sc = 0; sc < MT_BK; sc += 8)
        if (moe_stage_column(k0, sc, k) + 8 > k) return false;
  return true;
}
static_assert(moe_stage_columns_in_rows(), "loads stay inside their rows");

template <bool UP>
__global__ __launch_bounds__(256, 2) void moe_tile_kernel(
    bf16* __restrict__ out, const bf16* __restrict__ a,
    const bf16* __restrict__ w, const int* __restrict__ perm,
    const int4* __restrict__ items, const int* __restrict__ n_items,
    const int64_t a_stride, const int64_t w_expert, const int64_t w_stride,
    const int n_out, const int k_total, const int top_k, const int row_tiles) {
  const int total = *n_items * row_tiles;
  const int per = (total + 7) / 8;
  const int slot = blockIdx.x / 8;
  const int job = blockIdx.x % 8 * per + slot;
  if (slot >= per || job >= total) return;
  const int4 item = items[job / row_tiles];
  const int cnt = item.z;
  const int n0 = job % row_tiles * (UP ? MT_BN / 2 : MT_BN);
  __shared__ __attribute__((aligned(16))) bf16 a_s[2][MT_BM][MT_LS];
  __shared__ __attribute__((aligned(16))) bf16 w_s[2][MT_BN][MT_LS];
  const int tid = threadIdx.x, lane = tid % WAVE_SIZE, lq = lane % 16,
            la = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE_SIZE);
  const int wm = wave / 2, wn = wave % 2;
  // staging: thread -> rows tid / 8 + 32 * j, columns (tid % 8) * 8
  const int sr = tid / 8, sc = tid % 8 * 8;
  const bf16* ap[4];
  const bf16* wp[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int place = item.y + min(sr + 32 * j, cnt - 1);
    ap[j] = a + (int64_t)(UP ? perm[place] / top_k : place) * a_stride;
    // UP: rows of a wave's half are 32 gate rows, then their 32 up rows
    const int r = sr + 32 * j;
    const int n = UP ? min(n0 + r / 64 * 32 + r % 32, n_out - 1) +
                           (r / 32 % 2) * n_out
                     : min(n0 + r, n_out - 1);
    wp[j] = w + (int64_t)item.x * w_expert + (int64_t)n * w_stride;
  }
  ushort8 ar[4], wr[4];
  auto load = [&](int k0) {
    const bool in = k0 + sc < k_total;  // the last 64 may be half there
    const int o = moe_stage_column(k0, sc, k_total);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      ar[j] = *reinterpret_cast<const ushort8*>(ap[j] + o);
      wr[j] = *reinterpret_cast<const ushort8*>(wp[j] + o);
    }
    if (!in) {
#pragma unroll
      for (int j = 0; j < 4; ++j) ar[j] = wr[j] = ushort8{};
    }
  };
  auto store = [&](int b) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      *reinterpret_cast<ushort8*>(&a_s[b][sr + 32 * j][sc]) = ar[j];
      *reinterpret_cast<ushort8*>(&w_s[b][sr + 32 * j][sc]) = wr[j];
    }
  };
  f32x4 acc[4][4];  // [weight rows][pairs]
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[f][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = (k_total + MT_BK - 1) / MT_BK;
  load(0);
  store(0);
  __syncthreads();
  for (int s = 0; s < steps; ++s) {
    const int b = s & 1;
    if (s + 1 < steps) load((s + 1) * MT_BK);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      ushort8 wf[4], af[4];
#pragma unroll
      for (int f = 0; f < 4; ++f)
        wf[f] = *reinterpret_cast<const ushort8*>(
            &w_s[b][wn * 64 + f * 16 + lq][q * 32 + 8 * la]);
#pragma unroll
      for (int t = 0; t < 4; ++t)
        af[t] = *reinterpret_cast<const ushort8*>(
            &a_s[b][wm * 64 + t * 16 + lq][q * 32 + 8 * la]);
#pragma unroll
      for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int t = 0; t < 4; ++t)
          acc[f][t] = moe_mfma(wf[f], af[t], acc[f][t]);
    }
    if (s + 1 < steps) store(b ^ 1);
    // (the loads of the step behind the next are not issued yet)
    __syncthreads();
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int m = wm * 64 + t * 16 + lq;
    if (m >= cnt) continue;
    bf16* row = out + (int64_t)(item.y + m) * n_out;
#pragma unroll
    for (int f = 0; f < (UP ? 2 : 4); ++f) {
      const int n = n0 + wn * (UP ? 32 : 64) + f * 16 + 4 * la;
      if (n >= n_out) continue;
      ushort4v o;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        o[r] = float_to_bf16_bits(
            UP ? tile_silu_mul(acc[f][t][r], acc[f + 2][t][r]) : acc[f][t][r]);
      *reinterpret_cast<ushort4v*>(row + n) = o;
    }
  }
}

// Up to 320 pairs of one expert x 256 weight rows (UP: 128 gate rows and their up
// rows) in the loop of wide_engine.h, whose waves take 1 to 5 fragments of 16 pairs
// each: a tile's time is a fixed part of 0.5 and 0.21 for each 64 of its pairs.
// 5012 rows of 128 experts of 2048 x 768, 8 per row, read 1.5 GB through the caches
// in 276 us of gate and up, so that weights and rows bound them as much as the
// matrix cores do (busy for 60 % of the CUs' time).
// ONCE: for experts that have one item each, mostly (up to 160 pairs on the mean):
// their weights pass the caches by, where the rows stay then, and (rotate) the tiles
// of an expert begin at different steps, so that reads of columns a power of two
// apart meet on more of the memory's channels; which step follows from the expert's
// number among all ranks', as its order of sums must. us with plan, items of up to 320,
// as they are (past the caches; and rotated): 128 experts of 2048 x 768, 8 per row, 1000
// rows 268 (251; 239), 2048 rows 309 (295; 298), 4096 rows 449 (456; 454); 16 experts of
// 4096 x 3584, 4 per row, 500 rows 319 (306; 299), 2000 rows 690 (706; 716). The line
// could lie a little higher: 200 pairs, 128 experts 346 (326; 310).
// Each XCD takes a contiguous stretch of (expert, row tile, item), so that an
// expert's items meet the same weights in its L2; its workgroups claim tiles one by
// one, as they take different times (5012 rows in tile_engine.h's tiles, dealt out in
// turn 591 us, claimed 545). The claim is made a tile ahead, so that neither it nor the
// pairs' rows are waited for. Its place in LDS belongs to the tiles' array: a second one
// made the compiler drain the loads before every read of the first.
// GLU: gate and up are rounded to bf16 before they meet, as rows of a product in
// memory would be. SCALED: scale [pairs] is a factor of both; it is loaded in front
// of the next tile's first loads, so as not to be waited for behind them, and named
// again behind them: only rows that a tile has use it, so that the compiler took the
// others' loads to be still under way, and drained all loads in every step of the
// loop for 193 to 256 pairs, whose fragments lie in these registers. us with plan,
// before (which asked at run time whether there is a scale) -> so: 16 experts of 4096
// x 3584, 4 per row, no scale, 2000 rows 719 -> 703, 3000 rows 1039 -> 961.
template <bool ONCE>
using MoeTileOf = WideTile<4, 4, 5, false, ONCE ? 2 : 0>;

// f(fragments a wave that `pairs` pairs take), as a constant
template <typename F>
__device__ __forceinline__ void moe_frags(const int pairs, F f) {
  switch ((pairs + 63) / 64) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    default: f(std::integral_constant<int, 5>{});
  }
}

template <bool UP, bool GLU, bool SCALED, bool ONCE>
__global__ __launch_bounds__(512, 2) void moe_engine_kernel(
    bf16* __restrict__ out, const bf16* __restrict__ a,
    const bf16* __restrict__ w, const int* __restrict__ perm,
    const int4* __restrict__ items, const int* __restrict__ n_items,
    int* __restrict__ claims, const float* __restrict__ scale,
    const int64_t a_stride, const int64_t w_expert, const int64_t w_stride,
    const int n_out, const int k_total, const int top_k, const int row_tiles,
    const int rotate, const int expert_base) {
  using MoeTile = MoeTileOf<ONCE>;
  constexpr int FY = 5, COLS = UP ? 128 : 256;
  __shared__ __attribute__((aligned(1024))) char lds[MoeTile::LDS + 16];
  int& claimed = *reinterpret_cast<int*>(lds + MoeTile::LDS);
  const int total = *n_items * row_tiles;
  const int xcd = blockIdx.x % 8, slots = gridDim.x / 8;
  const int j0 = (int)((int64_t)total * xcd / 8);
  const int jn = (int)((int64_t)total * (xcd + 1) / 8) - j0;
  int i = blockIdx.x / 8;
  if (i >= jn) return;
  const int steps = k_total / TILE_K;
  MoeTile tile(lds);
  const int lq = tile.lane() % 16, la = tile.lane() / 16;
  struct Job {
    int expert, first, pairs, n0;
    typename MoeTile::Span k;
  };
  auto job = [&](int i) {
    const int j = j0 + i, q = j / row_tiles, w4 = items[q].w;
    const int i0 = q - (w4 & 0xffff), r = j - i0 * row_tiles, n = w4 >> 16;
    const int4 it = items[i0 + r % n];
    const int turn = rotate ? ((expert_base + it.x) * row_tiles + r / n) % steps : 0;
    return Job{it.x, it.y, it.z, r / n * COLS, {0, steps, turn}};
  };
  // The rows of a that this wave loads, each in a lane of its own (so they are one
  // register beside a tile's sums).
  auto places = [&](const Job& b) {
    const int f = (b.pairs + 63) / 64;
    const int r = min(tile.wave() * f * 8 + tile.lane(), b.pairs - 1);
    return UP ? perm[b.first + r] : r;
  };
  auto rows = [&](const Job& b, const int p) {
    typename MoeTile::Rows t;
    t.x = tile_buffer(w + b.expert * w_expert);
    t.y = tile_buffer(a + (UP ? 0 : b.first * a_stride));
#pragma unroll
    for (int j = 0; j < MoeTile::LX; ++j) {
      // A wave's 64 weight rows: as in wide_gemm.hip, 8 neighbouring columns of a
      // lane are 2 fragments, or (UP) 4, with a column's gate and up row in turns.
      const int row = tile.row_x(j), q = row / 16 % 4, g = row % 16 / 4, r = row % 4;
      const int base = row / 64 * (UP ? 32 : 64);
      const int col = base + (UP ? 8 * g + 2 * q + r / 2
                                 : q / 2 * 32 + 8 * g + 4 * (q & 1) + r);
      t.xo[j] = (uint32_t)(min(b.n0 + col, n_out - 1) + (UP && (r & 1) ? n_out : 0)) *
                    (uint32_t)(w_stride * 2) +
                tile.piece();
    }
#pragma unroll
    for (int j = 0; j < FY; ++j)
      t.yo[j] = (uint32_t)__shfl(UP ? p / top_k : p, j * 8 + tile.lane() / 8) *
                    (uint32_t)(a_stride * 2) +
                tile.piece();
    return t;
  };
  Job now = job(i);
  int p = places(now);
  typename MoeTile::Rows t = rows(now, p);
  moe_frags(now.pairs, [&](auto f) { tile.template prologue<f>(t, now.k); });
  // workgroups' first tiles are theirs, the others are claimed
  if (threadIdx.x == 0) claimed = slots + atomicAdd(&claims[xcd], 1);
  MoeTile::sync();
  i = __builtin_amdgcn_readfirstlane(claimed);
  moe_frags(now.pairs, [&](auto f) { tile.template prologue_wait<f>(steps); });
  for (;;) {
    const bool more = i < jn;
    const Job next = more ? job(i) : now;
    if (more) p = places(next);
    moe_frags(now.pairs, [&](auto f) { tile.template run<f>(t, now.k); });
    float by[SCALED ? FY : 1];
    if constexpr (SCALED) {
      int at[FY];
#pragma unroll
      for (int y = 0; y < FY; ++y)
        at[y] = perm[now.first + min(tile.frag_y(y) + lq, now.pairs - 1)];
#pragma unroll
      for (int y = 0; y < FY; ++y) by[y] = scale[at[y]];
    }
    int c;
    if (more) {
      if (threadIdx.x == 0) c = atomicAdd(&claims[xcd], 1);
      // its loads travel while this tile is stored
      t = rows(next, p);
      moe_frags(next.pairs, [&](auto f) { tile.template prologue<f>(t, next.k); });
    }
    // the sums' columns: 8 of each half (UP), 8 of each half's two pairs of fragments
    constexpr int P = UP ? 1 : 2;
    ushort8 o[FY][2 * P];
#pragma unroll
    for (int y = 0; y < FY; ++y)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int q = 0; q < P; ++q) {
          float v[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            if constexpr (UP) {
              const float g = tile.acc[4 * h + e / 2][y][e % 2 * 2];
              const float u = tile.acc[4 * h + e / 2][y][e % 2 * 2 + 1];
              if constexpr (SCALED)
                v[e] = silu_f(by[y] * moe_bf16(g)) * (by[y] * moe_bf16(u));
              else
                v[e] = GLU ? silu_f(moe_bf16(g)) * moe_bf16(u) : tile_silu_mul(g, u);
            } else {
              v[e] = tile.acc[4 * h + 2 * q + e / 4][y][e % 4];
            }
          }
          o[y][h * P + q] = tile_round(v);
        }
    if constexpr (SCALED) {
#pragma unroll
      for (int y = 0; y < FY; ++y) asm volatile("" : "+v"(by[y]));
    }
    if (more) {
      if (threadIdx.x == 0) claimed = slots + c;
      moe_frags(next.pairs, [&](auto f) { tile.template prologue_wait<f>(steps); });
    }
#pragma unroll
    for (int y = 0; y < FY; ++y) {
      const int m = tile.frag_y(y) + lq;
      if (m >= now.pairs) break;  // fragments are in the rows' order
      bf16* row = out + (int64_t)(now.first + m) * n_out + now.n0;
#pragma unroll
      for (int x = 0; x < 2 * P; ++x) {
        const int col = x / P * (COLS / 2) + tile.wm() * (UP ? 32 : 64) +
                        x % P * 32 + 8 * la;
        if (now.n0 + col < n_out) *reinterpret_cast<ushort8*>(row + col) = o[y][x];
      }
    }
    if (!more) return;
    now = next;
    MoeTile::sync();
    i = __builtin_amdgcn_readfirstlane(claimed);
  }
}

}  // namespace arks

using namespace arks;

// groups: workgroups that the pairs are spread over; more than one need
// counts [groups, n_local]. tile above 256 (moe_engine's): items of the
// size that moe_cut finds for products of these MoeRounds, an expert's even, in whole
// 64 pairs; max_items holds those of up to 192.
extern "C" void arks_moe_plan(void* perm, void* rows, void* weights_out,
                              void* items, void* n_items, void* claims,
                              void* counts, const void* ids,
                              const void* weights, int pairs, int expert_base,
                              int n_local, int tile, int max_items, int groups,
                              const int* rounds, hipStream_t stream) {
  const MoeRounds rounds_of{rounds[0], rounds[1], rounds[2], rounds[3]};
#define ARKS_PLAN(STAGE)                                                      \
  hipLaunchKernelGGL((moe_plan_kernel<STAGE>), dim3(groups), dim3(1024), 0,   \
                     stream, (int*)perm, (int*)rows, (float*)weights_out,     \
                     (int4*)items, (int*)n_items, (int*)claims, (int*)counts, \
                     (const int*)ids, (const float*)weights, pairs,           \
                     expert_base, n_local, tile, max_items, MoeLogits{}, rounds_of)
  if (groups == 1) {
    ARKS_PLAN(0);
  } else {
    ARKS_PLAN(1);
    ARKS_PLAN(2);
  }
#undef ARKS_PLAN
}

// arks_moe_plan of one group whose ids and weights come from logits [pairs / k,
// experts]: at most 512 pairs, 128 experts in all, k <= 64.
extern "C" void arks_moe_plan_topk(void* perm, void* rows, void* weights_out,
                                   void* items, void* n_items, void* claims,
                                   const void* logits, int experts, int k,
                                   int renorm, int pairs, int expert_base,
                                   int n_local, int tile, int max_items,
                                   const int* rounds, hipStream_t stream) {
  hipLaunchKernelGGL((moe_plan_kernel<0, 2>), dim3(1), dim3(1024), 0, stream,
                     (int*)perm, (int*)rows, (float*)weights_out, (int4*)items,
                     (int*)n_items, (int*)claims, nullptr, nullptr, nullptr, pairs,
                     expert_base, n_local, tile, max_items,
                     MoeLogits{(const float*)logits, experts, k, renorm},
                     MoeRounds{rounds[0], rounds[1], rounds[2], rounds[3]});
}

// tile: pairs of an item, 16 (streamed; n_out % 32 == k_total % 32 == 0) or 128
// (tiles through LDS; n_out % 8 == k_total % 8 == 0) or 256 (the engine, whose items
// have up to 320; n_out % 8 == k_total % 64 == 0, an expert's weights and (up) all
// rows of a under 4 GiB; up: 1, or 2 for GLU, with scale [pairs] or null; once: 0,
// 1, or 2 for rotated columns, by an expert's number from expert_base on).
extern "C" void arks_moe_gemm(void* out, const void* a, const void* w,
                              const void* perm, const void* items,
                              const void* n_items, void* claims,
                              const void* scale, int64_t a_stride, int64_t w_expert,
                              int64_t w_stride, int n_out, int k_total,
                              int top_k, int max_items, int tile, int up,
                              int once, int expert_base, hipStream_t stream) {
  const bool glu = up == 2;
#define ARKS_STREAM(NF, WV, UP)                                               \
  hipLaunchKernelGGL((moe_stream_kernel<NF, WV, UP>),                         \
                     dim3(n_out / (UP ? 16 : 16 * NF), max_items),            \
                     dim3(WV * 64), 0, stream, (bf16*)out, (const bf16*)a,    \
                     (const bf16*)w, (const int*)perm, (const int4*)items,    \
                     a_stride, w_expert, w_stride, n_out, k_total, top_k)
  // waves that split K: enough to cover it in a few chunks each
  if (tile == 16) {
    if (up) {
      if (k_total >= 1024) ARKS_STREAM(2, 8, true);
      else ARKS_STREAM(2, 4, true);
    } else {
      if (k_total >= 4096) ARKS_STREAM(2, 8, false);
      else ARKS_STREAM(2, 4, false);
    }
  } else if (tile == 256) {
    const int row_tiles = (n_out + (up ? 127 : 255)) / (up ? 128 : 256);
    const int64_t jobs = (int64_t)max_items * row_tiles;
    const dim3 grid(jobs < 256 ? (jobs + 7) / 8 * 8 : 256), block(512);
#define ARKS_ENGINE_O(UP, GLU, SCALED, ONCE)                                  \
  hipLaunchKernelGGL((moe_engine_kernel<UP, GLU, SCALED, ONCE>), grid, block, 0, \
                     stream, (bf16*)out, (const bf16*)a, (const bf16*)w,      \
                     (const int*)perm, (const int4*)items,                    \
                     (const int*)n_items, (int*)claims + (up ? 0 : 8),        \
                     (const float*)scale, a_stride, w_expert, w_stride, n_out, \
                     k_total, top_k, row_tiles, (int)(once == 2), expert_base)
#define ARKS_ENGINE(UP, GLU, SCALED)                                          \
  do {                                                                        \
    if (once) ARKS_ENGINE_O(UP, GLU, SCALED, true);                           \
    else ARKS_ENGINE_O(UP, GLU, SCALED, false);                               \
  } while (0)
    if (up && glu && scale) ARKS_ENGINE(true, true, true);
    else if (up && glu) ARKS_ENGINE(true, true, false);
    else if (up) ARKS_ENGINE(true, false, false);
    else ARKS_ENGINE(false, false, false);
#undef ARKS_ENGINE
#undef ARKS_ENGINE_O
  } else {
    const int cols = up ? MT_BN / 2 : MT_BN;
    const int row_tiles = (n_out + cols - 1) / cols;
    const dim3 grid((max_items * row_tiles + 7) / 8 * 8), block(256);
    if (up)
      hipLaunchKernelGGL((moe_tile_kernel<true>), grid, block, 0, stream,
                         (bf16*)out, (const bf16*)a, (const bf16*)w,
                         (const int*)perm, (const int4*)items,
                         (const int*)n_items, a_stride, w_expert, w_stride,
                         n_out, k_total, top_k, row_tiles);
    else
      hipLaunchKernelGGL((moe_tile_kernel<false>), grid, block, 0, stream,
                         (bf16*)out, (const bf16*)a, (const bf16*)w,
                         (const int*)perm, (const int4*)items,
                         (const int*)n_items, a_stride, w_expert, w_stride,
                         n_out, k_total, top_k, row_tiles);
  }
#undef ARKS_STREAM
}
