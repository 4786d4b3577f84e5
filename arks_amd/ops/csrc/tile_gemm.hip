// out[M, N] = silu(a w_gate^T) * (a w_up^T) for many rows, w [2N, K] the gate
// rows, then the up rows: the product of tile_engine.h with a tile's two halves of w
// as 128 gate rows and their up rows, so that the activation is taken on the fp32
// sums and neither product travels through memory. It has what fills 0.98 of its
// rounds (28672 x 4096, 8192 rows 1303 us, wide_gemm.hip 1381), weights that stay out
// of wide_gemm.hip (ops.plain_prompts) and those beyond its 32-bit offsets (from 2^31
// gate elements on). 18944 x
// 3584: 8192 rows 1511 us (1473 TFLOP/s; a library product and the activation
// behind it 1633), 3150 rows 612 us (1398 TFLOP/s; 798), 2048 rows 397 us
// (420). One workgroup per CU goes from tile to tile, the next one's first
// loads under way while the sums are stored: launched tile by tile 8192 rows
// took 1.016 of the time, 3150 rows (with the last 78 of them as a tile of 256)
// 1.05.
#include "tile_engine.h"

namespace arks {

// Rows of tiles go in groups of 8 that share the weights they read; each XCD
// takes a contiguous stretch of (group, columns, row of tiles), so that its L2
// serves both. Tiles of the last 1 to 128 rows cost about 0.55 of a full one and
// come last, spread over the XCDs likewise.
__global__ __launch_bounds__(512, 2) void tile_silu_kernel(
    bf16* __restrict__ out, const bf16* __restrict__ a,
    const bf16* __restrict__ w, const int m_rows, const int n_total,
    const int k_total, const int64_t a_stride) {
  __shared__ __attribute__((aligned(1024))) char lds[TILE_LDS];
  const int cols = (n_total + 127) / 128;
  const int left = m_rows % TILE_M;
  const bool tail = left > 0 && left <= TILE_HALF;
  const int full_rows = m_rows / TILE_M + (left > TILE_HALF ? 1 : 0);
  const int full = full_rows * cols;
  const int xcd = blockIdx.x % 8, slots = gridDim.x / 8;
  const int f0 = (int)((int64_t)full * xcd / 8);
  const int fn = (int)((int64_t)full * (xcd + 1) / 8) - f0;
  const int h0 = tail ? cols * xcd / 8 : 0;
  const int hn = tail ? cols * (xcd + 1) / 8 - h0 : 0;
  int i = blockIdx.x / 8;
  if (i >= fn + hn) return;
  const int steps = k_total / TILE_K;
  Tile tile(lds);
  struct Job {
    int m0, n0;
    bool half;
  };
  auto job = [&](int i) {
    constexpr int G = 8;
    if (i >= fn) return Job{full_rows * TILE_M, (h0 + i - fn) * 128, true};
    const int j = f0 + i, g = j / (G * cols), r = j % (G * cols);
    const int gm = min(G, full_rows - g * G);
    return Job{(g * G + r % gm) * TILE_M, r / gm * 128, false};
  };
  auto rows = [&](const Job& b) {
    TileRows t;
    t.a = tile_buffer(a + b.m0 * a_stride);
    t.w[0] = tile_buffer(w + (int64_t)b.n0 * k_total);
    t.w[1] = tile_buffer(w + (int64_t)(n_total + b.n0) * k_total);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r = tile_row(tile.wave(), tile.lane(), j);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        t.ao[h][j] = (uint32_t)min(h * 128 + r, m_rows - 1 - b.m0) *
                         (uint32_t)(a_stride * 2) +
                     tile_piece_a(r, tile.lane());
        t.wo[h][j] = (uint32_t)min(r, n_total - 1 - b.n0) *
                         (uint32_t)(k_total * 2) +
                     tile_piece_w(r, tile.lane());
      }
    }
    return t;
  };
  Job now = job(i);
  TileRows t = rows(now);
  tile.prologue(t, steps, now.half);
  tile.prologue_wait(steps, now.half);
  for (;;) {
    tile.run(t, steps, now.half);
    i += slots;
    const bool more = i < fn + hn;
    const Job next = more ? job(i) : now;
    if (more) {  // its loads travel while this tile is stored
      t = rows(next);
      tile.prologue(t, steps, next.half);
    }
    ushort8 o[8];
    tile.each([&](int x, int, int, const float(&g)[8], const float(&u)[8]) {
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = tile_silu_mul(g[j], u[j]);
      o[x] = tile_round(v);
    });
    if (more) tile.prologue_wait(steps, next.half);
    tile.each([&](int x, int m, int n, const float(&)[8], const float(&)[8]) {
      const int row = now.m0 + m, col = now.n0 + n;
      if (row < m_rows && col < n_total)  // n_total % 8 == 0
        *reinterpret_cast<ushort8*>(out + (int64_t)row * n_total + col) = o[x];
    });
    if (!more) return;
    now = next;
  }
}

}  // namespace arks

using namespace arks;

// a rows on 16 bytes, w and out contiguous and on 16 bytes; k % 64 == 0,
// n % 8 == 0, 256 rows of a and 128 of w under 4 GiB.
extern "C" void arks_tile_silu(void* out, const void* a, const void* w, int m,
                               int n, int k, int64_t a_stride,
                               hipStream_t stream) {
  const int64_t tiles = (int64_t)((m + 255) / 256) * ((n + 127) / 128);
  const int grid = (int)(tiles < 256 ? (tiles + 7) / 8 * 8 : 256);
  hipLaunchKernelGGL(tile_silu_kernel, dim3(grid), dim3(512), 0, stream,
                     (bf16*)out, (const bf16*)a, (const bf16*)w, m, n, k,
                     a_stride);
}
