// out[M, N] = a[M, K] . w[N, K]^T (+ bias), its fp32 sums over runs of K, or
// silu(gate) * up of two such products, for more than 256 rows.
//
// What bounds it are the matrix cores, as long as all CUs have work. A few hundred
// rows are few tiles, so there are several sizes of them (128 x 256 to 256 x 320
// and 320 x 256), and K may be cut into runs whose sums the consumer adds
// (ops._wide_cut chooses both). us of a product alone, with a launch for the sums
// (library): 3584 x 18944, 300 rows in 320 x 128 and 9 runs 60 (101), 700 rows in
// 256 x 256 and 6 97 (165); gate and up of 18944 x 3584 with the activation, 400
// rows in 256 x 320 104 (library and activation 144, tile_gemm.hip 157), 1000 rows
// 194 (316, 236). Writing the sums, 50 to 60 MB, is 8 to 14 us of these, whole
// lines at a time, past the caches or not.
//
// A workgroup of 8 waves goes from one tile to the next, whose first loads travel
// while the sums are stored. Rows of tiles go in groups of 8 that share the weights
// they read; each XCD takes a contiguous stretch of (run, group, columns, row of
// tiles), so that its L2 serves both operands.
#include "parts.h"
#include "wide_engine.h"

namespace arks {

enum WideOut { WIDE_BF16, WIDE_SUMS, WIDE_SILU };

template <int FX0, int FX1, int FY, bool AX, WideOut OUT>
__global__ __launch_bounds__(512, 2) void wide_gemm_kernel(
    void* __restrict__ out, const bf16* __restrict__ a,
    const bf16* __restrict__ w, const bf16* __restrict__ bias,
    const int m_rows, const int n_total, const int k_total,
    const int64_t a_stride, const int splits) {
  using T = WideTile<FX0, FX1, FY, AX>;
  constexpr bool SILU = OUT == WIDE_SILU;
  constexpr int TM = AX ? T::X : T::Y, TW = AX ? T::Y : T::X;
  constexpr int COLS = SILU ? TW / 2 : TW;
  __shared__ __attribute__((aligned(1024))) char lds[T::LDS];
  T tile(lds);
  const int tm = (m_rows + TM - 1) / TM, tn = (n_total + COLS - 1) / COLS;
  const int tiles = tm * tn, jobs = tiles * splits;
  const int xcd = blockIdx.x % 8, slots = gridDim.x / 8;
  const int j0 = (int)((int64_t)jobs * xcd / 8);
  const int jn = (int)((int64_t)jobs * (xcd + 1) / 8) - j0;
  int i = blockIdx.x / 8;
  if (i >= jn) return;
  const int all = k_total / TILE_K;

  struct Job {
    int m0, n0, split;
    typename T::Span k;
  };
  auto job = [&](int i) {
    constexpr int G = 8;
    const int j = j0 + i, split = j / tiles, at = j % tiles;
    const int g = at / (G * tn), r = at % (G * tn);
    const int gm = min(G, tm - g * G);
    const int s0 = (int)((int64_t)all * split / splits);
    return Job{(g * G + r % gm) * TM, r / gm * COLS, split,
               {s0, (int)((int64_t)all * (split + 1) / splits) - s0, 0}};
  };
  // The column (of those of a wave's f fragments) whose weights stand at row `at`
  // of them, so that a lane's sums are neighbours in the output: 8 columns of two
  // fragments, or of four with the activation, where sums 0 and 2 of a fragment
  // are gate columns, 1 and 3 the up columns beside them. Sums in fp32 are 4
  // columns, 16 bytes, as they are.
  auto column = [](int at, int f) {
    const int q = at / 16, i = at % 16, g = i / 4, r = i % 4;
    if constexpr (SILU) {
      if (q / 4 * 4 + 3 < f) return q / 4 * 32 + 8 * g + 2 * (q % 4) + r / 2;
      if ((q | 1) < f) return q / 2 * 16 + 4 * g + 2 * (q & 1) + r / 2;
      return 8 * q + 2 * g + r / 2;
    } else {
      if (OUT == WIDE_BF16 && (q | 1) < f) return q / 2 * 32 + 8 * g + 4 * (q & 1) + r;
      return at;
    }
  };
  // The row of w, from the tile's first column on, that stands at row `row` of
  // the tile's.
  auto weight = [&](int row, int n0) {
    int base, at, f;
    if constexpr (AX) {
      base = row / (16 * FY) * 16 * FY, at = row % (16 * FY), f = FY;
    } else {
      const bool h = row >= T::X0;
      const int in = h ? row - T::X0 : row, per = 16 * (h ? FX1 : FX0);
      base = (h ? T::X0 : 0) + in / per * per, at = in % per, f = h ? FX1 : FX0;
    }
    const int col = min((SILU ? base / 2 : base) + column(at, f), n_total - 1 - n0);
    return col + (SILU && (at & 1) ? n_total : 0);
  };
  auto rows = [&](const Job& b) {
    typename T::Rows t;
    const auto ab = tile_buffer(a + b.m0 * a_stride);
    const auto wb = tile_buffer(w + (int64_t)b.n0 * k_total);
    t.x = AX ? ab : wb;
    t.y = AX ? wb : ab;
    auto of_a = [&](int r) {
      return (uint32_t)min(r, m_rows - 1 - b.m0) * (uint32_t)(a_stride * 2) +
             tile.piece();
    };
    auto of_w = [&](int r) {
      return (uint32_t)weight(r, b.n0) * (uint32_t)(k_total * 2) + tile.piece();
    };
#pragma unroll
    for (int j = 0; j < T::LX; ++j)
      t.xo[j] = AX ? of_a(tile.row_x(j)) : of_w(tile.row_x(j));
#pragma unroll
    for (int j = 0; j < FY; ++j)
      t.yo[j] = AX ? of_w(tile.row_y(j)) : of_a(tile.row_y(j));
    return t;
  };
  Job now = job(i);
  typename T::Rows t = rows(now);
  tile.prologue(t, now.k);
  tile.prologue_wait(now.k.steps);
  for (;;) {
    tile.run(t, now.k);
    i += slots;
    const bool more = i < jn;
    const Job next = more ? job(i) : now;
    if (more) {
      t = rows(next);
      tile.prologue(t, next.k);
    }
    const int lq = tile.lane() % 16, la = tile.lane() / 16;
    // a row's sums, of the fragments of weights from column n on
    auto store = [&](int m, int n, auto frags, auto sum) {
      constexpr int F = decltype(frags)::value;
      const int row = now.m0 + m;
      if (row >= m_rows) return;
      if constexpr (OUT == WIDE_SUMS) {
        float* to = reinterpret_cast<float*>(out) +
                    ((int64_t)now.split * m_rows + row) * n_total + now.n0;
#pragma unroll
        for (int q = 0; q < F; ++q) {
          const int col = n + q * 16 + 4 * la;
          if (now.n0 + col < n_total) *reinterpret_cast<f32x4*>(to + col) = sum(q);
        }
      } else {
        bf16* to = reinterpret_cast<bf16*>(out) + (int64_t)row * n_total + now.n0;
        if constexpr (OUT == WIDE_BF16) {
#pragma unroll
          for (int q = 0; q < F; q += 2) {
            const bool pair = q + 1 < F;
            const int col = n + q * 16 + (pair ? 8 : 4) * la;
            if (now.n0 + col >= n_total) continue;
            float v[8];
#pragma unroll
            for (int e = 0; e < (pair ? 8 : 4); ++e)
              v[e] = sum(q + e / 4)[e % 4] +
                     (bias ? bf16_bits_to_float(bias[now.n0 + col + e]) : 0.f);
            if (pair) {
              *reinterpret_cast<ushort8*>(to + col) = tile_round(v);
            } else {
              ushort4v o;
#pragma unroll
              for (int e = 0; e < 4; ++e) o[e] = float_to_bf16_bits(v[e]);
              *reinterpret_cast<ushort4v*>(to + col) = o;
            }
          }
        } else {
          constexpr int QUADS = F / 4 * 4;
#pragma unroll
          for (int q = 0; q < QUADS; q += 4) {
            const int col = n + q * 8 + 8 * la;
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e)
              v[e] = tile_silu_mul(sum(q + e / 2)[e % 2 * 2],
                                   sum(q + e / 2)[e % 2 * 2 + 1]);
            if (now.n0 + col < n_total)
              *reinterpret_cast<ushort8*>(to + col) = tile_round(v);
          }
          if constexpr (F % 4 >= 2) {
            const int col = n + QUADS * 8 + 4 * la;
            ushort4v o;
#pragma unroll
            for (int e = 0; e < 4; ++e)
              o[e] = float_to_bf16_bits(
                  tile_silu_mul(sum(QUADS + e / 2)[e % 2 * 2],
                                sum(QUADS + e / 2)[e % 2 * 2 + 1]));
            if (now.n0 + col < n_total) *reinterpret_cast<ushort4v*>(to + col) = o;
          }
          if constexpr (F % 2) {
            const int col = n + (F - 1) * 8 + 2 * la;
            ushort2v o;
#pragma unroll
            for (int e = 0; e < 2; ++e)
              o[e] = float_to_bf16_bits(
                  tile_silu_mul(sum(F - 1)[e * 2], sum(F - 1)[e * 2 + 1]));
            if (now.n0 + col < n_total) *reinterpret_cast<ushort2v*>(to + col) = o;
          }
        }
      }
    };
    constexpr int S = SILU ? 2 : 1;
    if constexpr (AX) {
#pragma unroll
      for (int x = 0; x < FX0 + FX1; ++x)
        store(x < FX0 ? (tile.wm() * FX0 + x) * 16 + lq
                      : T::X0 + (tile.wm() * FX1 + x - FX0) * 16 + lq,
              tile.wn() * FY * 16 / S, std::integral_constant<int, FY>{},
              [&](int q) { return tile.acc[x][q]; });
    } else {
#pragma unroll
      for (int y = 0; y < FY; ++y) {
        const int m = tile.frag_y(y) + lq;
        store(m, tile.wm() * FX0 * 16 / S, std::integral_constant<int, FX0>{},
              [&](int q) { return tile.acc[q][y]; });
        store(m, (T::X0 + tile.wm() * FX1 * 16) / S,
              std::integral_constant<int, FX1>{},
              [&](int q) { return tile.acc[FX0 + q][y]; });
      }
    }
    if (!more) return;
    tile.prologue_wait(next.k.steps);
    now = next;
  }
}

}  // namespace arks

using namespace arks;

// kind: out is bf16 [m, n] (0), fp32 [splits, m, n] (1), or bf16 [m, n] with w
// [2n, k] (2). a rows on 16 bytes, w and out contiguous and on 16 bytes; k % 64 ==
// 0, at least one step of 64 a split, n % 8 == 0; tm rows of a and tw of w (kind 2:
// n + tw / 2 of them) under 4 GiB. Returns 0 if there is no tile of tm x tw.
extern "C" int arks_wide_gemm(void* out, const void* a, const void* w,
                              const void* bias, int m, int n, int k,
                              int64_t a_stride, int tm, int tw, int splits,
                              int kind, hipStream_t stream) {
  const int cols = kind == WIDE_SILU ? tw / 2 : tw;
  const int64_t jobs =
      (int64_t)((m + tm - 1) / tm) * ((n + cols - 1) / cols) * splits;
  const int grid = (int)(jobs < 256 ? (jobs + 7) / 8 * 8 : 256);
#define ARKS_WIDE(FX0, FX1, FY, AX, OUT)                                       \
  hipLaunchKernelGGL((wide_gemm_kernel<FX0, FX1, FY, AX, OUT>), dim3(grid),    \
                     dim3(512), 0, stream, out, (const bf16*)a,                \
                     (const bf16*)w, (const bf16*)bias, m, n, k, a_stride,     \
                     splits)
#define ARKS_WIDE_TILE(TM, TW, FX0, FX1, FY, AX)                               \
  if (tm == TM && tw == TW) {                                                  \
    if (kind == WIDE_BF16) ARKS_WIDE(FX0, FX1, FY, AX, WIDE_BF16);             \
    else if (kind == WIDE_SUMS) ARKS_WIDE(FX0, FX1, FY, AX, WIDE_SUMS);        \
    else ARKS_WIDE(FX0, FX1, FY, AX, WIDE_SILU);                               \
    return 1;                                                                  \
  }
  ARKS_WIDE_TILE(128, 256, 2, 2, 4, true)
  ARKS_WIDE_TILE(192, 256, 4, 2, 4, true)
  ARKS_WIDE_TILE(256, 128, 2, 2, 4, false)
  ARKS_WIDE_TILE(256, 192, 4, 4, 3, true)
  ARKS_WIDE_TILE(256, 256, 4, 4, 4, true)
  ARKS_WIDE_TILE(256, 320, 4, 4, 5, true)
  ARKS_WIDE_TILE(320, 128, 2, 2, 5, false)
  ARKS_WIDE_TILE(320, 256, 4, 4, 5, false)
#undef ARKS_WIDE_TILE
#undef ARKS_WIDE
  return 0;
}
