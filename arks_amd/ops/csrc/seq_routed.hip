// Experts of a few rows (a step that decodes): the gate and up products of the
// experts that rows chose, with their activation, and the down product over
// those experts' columns. Experts that no row chose are not read.
//
// What bounds them is the weights' stream. 4 waves multiply and 4 only load, NS
// steps ahead (ring.h).
//
// The order of sums is the same for any number of rows: K is cut into chunks of
// CHUNK columns, a chunk into 4 parts, and wave p adds up part p of every chunk in
// one chain; the 4 sums are added in order. Near a tie the last bits of a row
// decide between two experts, and no choice may turn with the rows that share a
// step. The columns of experts that nobody chose are products with 0, so that
// leaving them out changes nothing. (The chunks are those in which the library's
// products of 1 and of 8 rows, which were here before, were seen to add up with
// weights of 114688 x 4096 and 4096 x 57344: such steps kept their bits.)
//
// 16 experts of ff 3584 on 4096 columns, 4 per row, weights cold, us (the
// library's products over all experts): gate and up with the activation, 1 row
// (4 experts chosen) 42.7 (157 and 4.6 for the activation), 8 rows (11) 111 (158
// and 4.3), 16 rows (16) 161 (190 and 4.5), 5.5 to 6.1 TB/s; down 23.8 (82), 56
// (82), 87 (114).
#include <type_traits>

#include "ring.h"
#include "seq_common.h"

namespace arks {

struct RoutedAct {
  int scale_in;  // silu: the scale on gate and up, not on the product
  int clamped;   // min(g, l) sigmoid(alpha g) (clamp(u, -l, l) + 1)
  float limit, alpha;
};

// Stages of LDS: what fits beside the sums that waves hand over, at most 8.
constexpr int routed_stages(int qt) {
  return (160 - 4 * qt) / (8 * (qt + 1)) < 8 ? (160 - 4 * qt) / (8 * (qt + 1))
                                             : 8;
}

// UP: out [M, E * ff] = the activated products of x [M, K] with gate and up rows
// w [E][gate ff | up ff][K], 0 where a row did not choose the expert; else out
// [M, N] = x [M, E * ff] . w [N, E * ff]^T. scale [M, E]: weights of the experts
// that a row chose, 0 elsewhere. QT: 16 * QT weight rows a tile.
template <int QT, bool UP>
__global__ __launch_bounds__(512, 2) void routed_gemm_kernel(
    bf16* __restrict__ out, const bf16* __restrict__ x, const int64_t x_stride,
    const bf16* __restrict__ w, const float* __restrict__ scale,
    const int64_t scale_stride, const int m_rows, const int n_total,
    const int k_total, const int experts, const int ff, const RoutedAct act) {
  constexpr int NS = routed_stages(QT);
  constexpr int PART = (QT + 1) * 2048, STAGE = 4 * PART;  // of wave p; of all
  constexpr int LOADS = 2 * QT + 2;
  constexpr int COLS = UP ? 8 * QT : 16 * QT;
  constexpr int CHUNK = UP ? 512 : 1024, OWN = CHUNK / 4;  // columns; of a wave
  static_assert(NS >= 3 && (!UP || QT % 2 == 0));
  __shared__ __attribute__((aligned(1024))) char lds[NS * STAGE];
  __shared__ tile_f32x4 sums[4][QT][WAVE_SIZE];
  const int lane = threadIdx.x % WAVE_SIZE, lq = lane % 16, la = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int p = wave % 4;

  // the experts that somebody chose (none: all rows of the first one's are 0)
  bool mine = false;
  for (int m = 0; m < m_rows; ++m)
    mine |= lane < experts && scale[m * scale_stride + min(lane, experts - 1)] != 0.f;
  uint64_t chosen = __ballot(mine);
  if (chosen == 0) chosen = 1;

  // which chunks' part of a wave is a chosen expert's, 64 of them from `first`
  const int chunks = k_total / CHUNK;
  auto active = [&](const int first, const int of) -> uint64_t {
    const int c = first + lane;
    const int e = (c * CHUNK + of * OWN) / ff;
    return __ballot(c < chunks && (chosen >> min(e, 63) & 1));
  };
  const int per = UP ? k_total / 256 : 1;  // steps of a job
  int steps = per, own_steps = per;
  if constexpr (!UP) {
    steps = 0;
    for (int of = 0; of < 4; ++of) {
      int n = 0;
      for (int c = 0; c < chunks; c += 64) n += __popcll(active(c, of));
      n *= OWN / 64;
      steps = max(steps, n);
      if (of == p) own_steps = n;
    }
  }
  const int tiles = (UP ? ff : n_total) / COLS + ((UP ? ff : n_total) % COLS != 0);
  const int jobs = UP ? tiles * __popcll(chosen) : tiles;
  struct Job {
    int expert, at;  // first column of the tile, among the expert's
  };
  auto job = [&](const int j) {
    if constexpr (!UP) return Job{0, j * COLS};
    uint64_t left = chosen;
    for (int i = j / tiles; i > 0; --i) left &= left - 1;
    return Job{__ffsll((unsigned long long)left) - 1, j % tiles * COLS};
  };
  if ((int)blockIdx.x >= jobs) return;
  const int total =
      ((jobs - 1 - (int)blockIdx.x) / (int)gridDim.x + 1) * steps;

  if (wave >= 4) {
    __amdgpu_buffer_rsrc_t wb;
    const __amdgpu_buffer_rsrc_t xb = tile_buffer(x);
    uint32_t wo[2 * QT], xo[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = i * 8 + lane / 8;
      xo[i] = (uint32_t)min(row, m_rows - 1) * (uint32_t)(x_stride * 2) +
              tile_piece_a(row, lane);
    }
    auto aim = [&](const Job& b) {
      const int64_t row0 = UP ? (int64_t)b.expert * 2 * ff + b.at : b.at;
      wb = tile_buffer(w + row0 * k_total);
#pragma unroll
      for (int i = 0; i < 2 * QT; ++i) {
        const int row = i * 8 + lane / 8;
        int at = row;
        if constexpr (UP)  // 16 gate rows, the up rows beside them, and again
          at = min(row / 32 * 16 + row % 16, ff - 1 - b.at) +
               (row / 16 % 2 ? ff : 0);
        else
          at = min(row, n_total - 1 - b.at);
        wo[i] = (uint32_t)at * (uint32_t)(k_total * 2) + tile_piece_a(row, lane);
      }
    };
    int j = blockIdx.x, s = 0, stage = 0;
    int group = 0, c = 0, sub = 0;  // !UP: the chunk, and the step in its part
    uint64_t left = 0;
    auto next_chunk = [&] {
      while (left == 0 && group < chunks) {
        left = active(group, p);
        group += 64;
      }
      if (left) {
        c = group - 64 + __ffsll((unsigned long long)left) - 1;
        left &= left - 1;
      }
    };
    aim(job(j));
    if constexpr (!UP) next_chunk();
    auto load = [&] {
      int col;  // of this wave's step s
      if constexpr (UP) {
        const int i = s * 64;
        col = i / OWN * CHUNK + p * OWN + i % OWN;
      } else {
        col = c * CHUNK + p * OWN + sub * 64;
        if (++sub == OWN / 64) {
          sub = 0;
          next_chunk();
        }
      }
      char* to = lds + stage * STAGE + p * PART;
#pragma unroll
      for (int i = 0; i < 2; ++i)
        ring_load<false>(xb, to + QT * 2048 + i * 1024, xo[i], col * 2);
#pragma unroll
      for (int i = 0; i < 2 * QT; ++i)
        ring_load<true>(wb, to + i * 1024, wo[i], col * 2);
      stage = stage == NS - 1 ? 0 : stage + 1;
      if (++s == steps) {
        s = 0;
        j += gridDim.x;
        if (j < jobs) {
          aim(job(j));
          if constexpr (!UP) {
            group = 0, sub = 0, left = 0;
            next_chunk();
          }
        }
      }
    };
    int end = steps;  // of the job that is multiplied
    ring_feed<NS, LOADS>(total, load, [&](const int t) {
      if (t + 1 == end) {  // the sums are handed over
        ring_barrier();
        end += steps;
      }
    });
    return;
  }

  // where a step's operands lie: 16 rows of 128 B, pieces permuted
  const int frag = lq * 128 + ((la ^ (lq & 7)) * 16);
  int at = 0;  // the stage that is read
  ring_barrier();
  for (int j = blockIdx.x; j < jobs; j += gridDim.x) {
    const Job b = job(j);
    tile_f32x4 acc[QT];
#pragma unroll
    for (int q = 0; q < QT; ++q) acc[q] = tile_f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < steps; ++s) {
      ushort8 wf[2][QT], xf[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const char* rows = lds + at * STAGE + p * PART + (frag ^ (h * 64));
        xf[h] = *reinterpret_cast<const ushort8*>(rows + QT * 2048);
#pragma unroll
        for (int q = 0; q < QT; ++q)
          wf[h][q] = *reinterpret_cast<const ushort8*>(rows + q * 2048);
      }
      // this step has been read, the next one is there
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      ring_barrier();
      at = at == NS - 1 ? 0 : at + 1;
      if (UP || s < own_steps) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int q = 0; q < QT; ++q)
            acc[q] = tile_mfma(wf[h][q], xf[h], acc[q]);
      }
    }
#pragma unroll
    for (int q = 0; q < QT; ++q) sums[p][q][lane] = acc[q];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    ring_barrier();
    auto sum = [&](const int q) {
      tile_f32x4 v = sums[0][q][lane];
#pragma unroll
      for (int i = 1; i < 4; ++i) v += sums[i][q][lane];
      return v;
    };
    if constexpr (UP) {
      const int n = b.at + p * 16 + 4 * la;
      if (p < QT / 2 && lq < m_rows && n < ff) {  // ff % 16 == 0
        const tile_f32x4 gate = sum(2 * p), up = sum(2 * p + 1);
        const float s = scale[lq * scale_stride + b.expert];
        const float sg = act.scale_in ? s : 1.f;
        ushort4v o;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          // rounded as the products alone are, then as moe_glu_scaled has it
          const float gv = bf16_bits_to_float(float_to_bf16_bits(gate[r]));
          const float uv = bf16_bits_to_float(float_to_bf16_bits(up[r]));
          if (act.clamped) {
            const float g = fminf(gv, act.limit);
            const float u = fminf(fmaxf(uv, -act.limit), act.limit) + 1.f;
            o[r] = float_to_bf16_bits(s * (g / (1.f + __expf(-act.alpha * g)) * u));
          } else {
            const float g = sg * gv;
            const float u = s * uv;
            o[r] = float_to_bf16_bits(g / (1.f + __expf(-g)) * u);
          }
          if (s == 0.f) o[r] = 0;  // an expert the row does not use
        }
        *reinterpret_cast<ushort4v*>(
            out + ((int64_t)lq * experts + b.expert) * ff + n) = o;
      }
    } else if (p < QT) {
      const int n = b.at + p * 16 + 4 * la;
      if (lq < m_rows && n < n_total) {  // n_total % 16 == 0
        const tile_f32x4 v = sum(p);
        ushort4v o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = float_to_bf16_bits(v[r]);
        *reinterpret_cast<ushort4v*>(out + (int64_t)lq * n_total + n) = o;
      }
    }
  }
}

}  // namespace arks

using namespace arks;

// m <= 16, experts <= 64, ff % 16 == 0, k % 512 == 0; an expert's rows and all of
// x under 4 GiB, rows of x and w on 16 bytes.
extern "C" void arks_seq_routed_up(void* out, const void* x, int64_t x_stride,
                                   const void* w, const void* scale,
                                   int64_t scale_stride, int m, int k,
                                   int experts, int ff, int scale_in,
                                   int clamped, float limit, float alpha,
                                   hipStream_t stream) {
  const RoutedAct act{scale_in, clamped, limit, alpha};
  const int64_t jobs = (int64_t)((ff + 31) / 32) * experts;
  hipLaunchKernelGGL((routed_gemm_kernel<4, true>),
                     dim3((unsigned)(jobs < 256 ? jobs : 256)), dim3(512), 0,
                     stream, (bf16*)out, (const bf16*)x, x_stride, (const bf16*)w,
                     (const float*)scale, scale_stride, m, 0, k, experts, ff, act);
}

// x [m, experts * ff], w [n, experts * ff], n % 16 == 0, ff % 256 == 0, experts *
// ff % 1024 == 0; 16 rows of w and all of x under 4 GiB.
extern "C" void arks_seq_routed_down(void* out, const void* x, int64_t x_stride,
                                     const void* w, const void* scale,
                                     int64_t scale_stride, int m, int n,
                                     int experts, int ff, hipStream_t stream) {
  const int jobs = n / 16;
  hipLaunchKernelGGL((routed_gemm_kernel<1, false>),
                     dim3(jobs < 256 ? jobs : 256), dim3(512), 0, stream,
                     (bf16*)out, (const bf16*)x, x_stride, (const bf16*)w,
                     (const float*)scale, scale_stride, m, n, experts * ff,
                     experts, ff, RoutedAct{});
}
