// Elementwise / normalization kernels for the decode hot path (bf16, gfx950).
// All memory-bound: vectorized 16 B/lane loads (guide G13), grid-stride, f32
// accumulation. Ops: rmsnorm, fused residual-add + rmsnorm, silu_mul (SwiGLU),
// neox-style RoPE (in-place on q and k).
#include "common.h"
#include "parts.h"

namespace arks {

// ---------------------------------------------------------------------------
// RMSNorm: one workgroup per row, of 4 waves (8 where it adds split sums: such
// rows are few, and a row is one pass then).
// hidden must be a multiple of 8 (bf16x8 vector loads).
// IN_PARTS: the input is the sum of fp32 splits [splits, rows, hidden] of the
// product before it; adding 8 of them here takes 0.5 us at 64 x 3584, a launch
// of its own 5.
// IN_MIX: the input is the mix of the experts' rows that a token chose, rounded
// as moe_mix_rows stores it (behind 4 layers of 128 experts, 8 per row, one
// step of 64 rows 1289 -> 1282 us, of 7 rows 724 -> 719, a prompt pass 3810 ->
// 3792: a launch and, for many rows, one write and read of the mix less).
// NV: vectors of a thread that stay in registers, with the weights loaded
// beside them: few rows are bound by the chain of loads, sum and store, many
// by the bytes. Rows that are longer (NV 0) are read again from L2 behind the
// sum, as all were before: 64 x 3584 and 4 splits 5.3 us, held 4.9.
// The arguments fill one line of 64 bytes: a dimension of the grid, which lies
// behind them, would be one more load in front of the sums' addresses (64 x 3584
// and 4 splits 3.84 us back to back, with the rows as an argument 3.69).
// ---------------------------------------------------------------------------
enum NormInput { IN_ROWS, IN_PARTS, IN_MIX };
template <bool FUSED_ADD, NormInput IN, int NV, int U = 8>
__global__ void rmsnorm_kernel(bf16* __restrict__ out,
                               const void* __restrict__ input,
                               bf16* __restrict__ residual,  // null unless FUSED_ADD
                               const bf16* __restrict__ weight,
                               const float eps, const int hidden,
                               const int rows,
                               const int n_in,  // splits, or k of a mix
                               const float* __restrict__ mix_weights,  // [rows, k]
                               const int* __restrict__ mix_rows) {     // [rows, k]
  constexpr bool PARTS = IN == IN_PARTS;
  constexpr int BLOCK = PARTS ? 512 : 256;
  const int row = blockIdx.x;
  const bf16* in_row =
      reinterpret_cast<const bf16*>(input) + (int64_t)row * hidden;
  const float* part_row =
      reinterpret_cast<const float*>(input) + (int64_t)row * hidden;
  const int64_t part_stride = (int64_t)rows * hidden;
  bf16* res_row = FUSED_ADD ? residual + (int64_t)row * hidden : nullptr;
  bf16* out_row = out + (int64_t)row * hidden;

  const int nvec = hidden / 8;
  float ss = 0.f;
  // the row's values at vector i (with the residual, stored back)
  auto load = [&](const int i) {
    float x[8];
    ushort8 r{}, s;
    if constexpr (FUSED_ADD) r = *reinterpret_cast<const ushort8*>(res_row + i * 8);
    if constexpr (PARTS) {
      f32x4 lo, hi;
      sum_parts_pair<U>(part_row + i * 8, part_row + i * 8 + 4, part_stride,
                        n_in, lo, hi);
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = j < 4 ? lo[j % 4] : hi[j % 4];
    } else {
      if constexpr (IN == IN_MIX) {
        // weights and rows are the same in all lanes: scalar loads, no barrier
        const float* w = mix_weights + (int64_t)row * n_in;
        const int* rows_in = mix_rows + (int64_t)row * n_in;
        s = mix_rows8(
            reinterpret_cast<const bf16*>(input), n_in, i * 8,
            [&](int j) { return (int64_t)rows_in[min(j, n_in - 1)] * hidden; },
            [&](int j) { return j < n_in ? w[min(j, n_in - 1)] : 0.f; });
      } else {
        s = *reinterpret_cast<const ushort8*>(in_row + i * 8);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = bf16_bits_to_float(s[j]);
    }
    if constexpr (FUSED_ADD) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        s[j] = float_to_bf16_bits(x[j] + bf16_bits_to_float(r[j]));
        // the sum of squares is that of the rounded values, which are normed
        x[j] = bf16_bits_to_float(s[j]);
      }
      *reinterpret_cast<ushort8*>(res_row + i * 8) = s;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) ss += x[j] * x[j];
    return s;
  };
  __shared__ float red[BLOCK / WAVE_SIZE];
  float rrms;
  auto store = [&](const int i, const ushort8& x, const ushort8& w) {
    ushort8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      o[j] = float_to_bf16_bits(bf16_bits_to_float(x[j]) * rrms *
                                bf16_bits_to_float(w[j]));
    *reinterpret_cast<ushort8*>(out_row + i * 8) = o;
  };
  auto weights = [&](const int i) {
    return *reinterpret_cast<const ushort8*>(weight + i * 8);
  };
  if constexpr (NV > 0) {
    ushort8 x[NV], w[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int i = threadIdx.x + v * BLOCK;
      if (i < nvec) w[v] = weights(i);
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int i = threadIdx.x + v * BLOCK;
      if (i < nvec) x[v] = load(i);
    }
    rrms = rsqrtf(block_reduce_sum<BLOCK>(ss, red) / (float)hidden + eps);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int i = threadIdx.x + v * BLOCK;
      if (i < nvec) store(i, x[v], w[v]);
    }
  } else {
    for (int i = threadIdx.x; i < nvec; i += BLOCK) load(i);
    rrms = rsqrtf(block_reduce_sum<BLOCK>(ss, red) / (float)hidden + eps);
    const bf16* src_row = FUSED_ADD ? res_row : in_row;
    for (int i = threadIdx.x; i < nvec; i += BLOCK)
      store(i, *reinterpret_cast<const ushort8*>(src_row + i * 8), weights(i));
  }
}

// ---------------------------------------------------------------------------
// SiLU-mul: input [rows, 2*d] = [gate | up], output [rows, d].
// ---------------------------------------------------------------------------
__global__ void silu_mul_kernel(bf16* __restrict__ out,
                                const bf16* __restrict__ gate_up,
                                const int d, const int64_t total_vec) {
  // Grid-stride over row-major output in 8-element vectors.
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
       idx < total_vec; idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t row = idx / (d / 8);
    const int col8 = (int)(idx % (d / 8)) * 8;
    const bf16* g = gate_up + row * (2 * (int64_t)d) + col8;
    const bf16* u = g + d;
    ushort8 gv = *reinterpret_cast<const ushort8*>(g);
    ushort8 uv = *reinterpret_cast<const ushort8*>(u);
    ushort8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float x = bf16_bits_to_float(gv[j]);
      float silu = x / (1.f + __expf(-x));
      o[j] = float_to_bf16_bits(silu * bf16_bits_to_float(uv[j]));
    }
    *reinterpret_cast<ushort8*>(out + row * d + col8) = o;
  }
}

// ---------------------------------------------------------------------------
// RoPE (neox / rotate-half), in place on q [T, Hq*D] and k [T, Hkv*D].
// cos_sin: [max_pos, D] f32, first half cos, second half sin (host-precomputed
// — guide App. B: never sinf/cosf on device for RoPE).
// One workgroup per token; threads cover (head, pair) space, 2 pairs each.
// ---------------------------------------------------------------------------
__global__ void rope_kernel(const int64_t* __restrict__ positions,
                            bf16* __restrict__ q, bf16* __restrict__ k,
                            const float* __restrict__ cos_sin,
                            const int head_dim, const int num_q_heads,
                            const int num_kv_heads, const int64_t q_stride,
                            const int64_t k_stride) {
  const int token = blockIdx.x;
  const int half = head_dim / 2;
  const int64_t pos = positions[token];
  const float* cs = cos_sin + pos * head_dim;
  const int total_heads = num_q_heads + num_kv_heads;
  // Each thread handles 2 consecutive rotary pairs (4 bf16 values).
  const int pairs2 = half / 2;  // pair-couples per head
  for (int idx = threadIdx.x; idx < total_heads * pairs2; idx += blockDim.x) {
    const int h = idx / pairs2;
    const int p2 = (idx % pairs2) * 2;  // first pair index of the couple
    bf16* base = (h < num_q_heads)
                     ? q + (int64_t)token * q_stride + (int64_t)h * head_dim
                     : k + (int64_t)token * k_stride +
                           (int64_t)(h - num_q_heads) * head_dim;
    ushort2v x1 = *reinterpret_cast<const ushort2v*>(base + p2);
    ushort2v x2 = *reinterpret_cast<const ushort2v*>(base + half + p2);
    ushort2v o1, o2;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float c = cs[p2 + j];
      const float s = cs[half + p2 + j];
      const float a = bf16_bits_to_float(x1[j]);
      const float b = bf16_bits_to_float(x2[j]);
      o1[j] = float_to_bf16_bits(a * c - b * s);
      o2[j] = float_to_bf16_bits(b * c + a * s);
    }
    *reinterpret_cast<ushort2v*>(base + p2) = o1;
    *reinterpret_cast<ushort2v*>(base + half + p2) = o2;
  }
}

}  // namespace arks

// ------------------------------- launchers ---------------------------------
using namespace arks;

extern "C" {

#define ARKS_NORM_U(FUSED, IN, NV, U)                                          \
  hipLaunchKernelGGL((rmsnorm_kernel<FUSED, IN, NV, U>), dim3(rows),           \
                     dim3(IN == IN_PARTS ? 512 : 256), 0, stream, (bf16*)out,  \
                     input, (bf16*)residual, (const bf16*)weight, eps, hidden, \
                     rows, n_in, (const float*)mix_weights, (const int*)mix_rows)
#define ARKS_NORM(FUSED, IN, NV)                                               \
  do {                                                                         \
    constexpr bool P = IN == IN_PARTS;                                         \
    const int u = P ? parts_flight(n_in) : 8;                                  \
    if (u == 2) ARKS_NORM_U(FUSED, IN, NV, (P ? 2 : 8));                       \
    else if (u == 4) ARKS_NORM_U(FUSED, IN, NV, (P ? 4 : 8));                  \
    else ARKS_NORM_U(FUSED, IN, NV, 8);                                        \
  } while (0)
#define ARKS_NORM_V(FUSED, IN)                                                 \
  do {                                                                         \
    const int block = IN == IN_PARTS ? 512 : 256;                              \
    const int per = (hidden / 8 + block - 1) / block;                          \
    if (per <= 1) ARKS_NORM(FUSED, IN, 1);                                     \
    else if (per <= 2) ARKS_NORM(FUSED, IN, 2);                                \
    else if (per <= 4) ARKS_NORM(FUSED, IN, 4);                                \
    else ARKS_NORM(FUSED, IN, 0);                                              \
  } while (0)

void arks_rmsnorm(void* out, const void* input, const void* weight, float eps,
                  int rows, int hidden, hipStream_t stream) {
  void* const residual = nullptr;
  const int n_in = 0;
  const void *const mix_weights = nullptr, *const mix_rows = nullptr;
  ARKS_NORM_V(false, IN_ROWS);
}

void arks_fused_add_rmsnorm(void* out, const void* input, void* residual,
                            const void* weight, float eps, int rows, int hidden,
                            hipStream_t stream) {
  const int n_in = 0;
  const void *const mix_weights = nullptr, *const mix_rows = nullptr;
  ARKS_NORM_V(true, IN_ROWS);
}

void arks_fused_add_rmsnorm_parts(void* out, const void* input, int splits,
                                  void* residual, const void* weight, float eps,
                                  int rows, int hidden, hipStream_t stream) {
  const int n_in = splits;
  const void *const mix_weights = nullptr, *const mix_rows = nullptr;
  ARKS_NORM_V(true, IN_PARTS);
}

// input [any, hidden]: row r gets the k (at most 16) rows mix_rows[r] of it,
// times mix_weights[r]
void arks_fused_add_rmsnorm_mix(void* out, const void* input,
                                const void* mix_weights, const void* mix_rows,
                                int k, void* residual, const void* weight,
                                float eps, int rows, int hidden,
                                hipStream_t stream) {
  const int n_in = k;
  ARKS_NORM_V(true, IN_MIX);
}
#undef ARKS_NORM_V
#undef ARKS_NORM
#undef ARKS_NORM_U

void arks_silu_mul(void* out, const void* gate_up, int64_t rows, int d,
                   hipStream_t stream) {
  int64_t total_vec = rows * (d / 8);
  int blocks = (int)std::min<int64_t>((total_vec + 255) / 256, 2048);
  if (blocks == 0) blocks = 1;
  hipLaunchKernelGGL(silu_mul_kernel, dim3(blocks), dim3(256), 0, stream,
                     (bf16*)out, (const bf16*)gate_up, d, total_vec);
}

void arks_rope_inplace(const void* positions, void* q, void* k,
                       const void* cos_sin, int num_tokens, int head_dim,
                       int num_q_heads, int num_kv_heads, int64_t q_stride,
                       int64_t k_stride, hipStream_t stream) {
  dim3 grid(num_tokens), block(256);
  hipLaunchKernelGGL(rope_kernel, grid, block, 0, stream,
                     (const int64_t*)positions, (bf16*)q, (bf16*)k,
                     (const float*)cos_sin, head_dim, num_q_heads,
                     num_kv_heads, q_stride, k_stride);
}

}  // extern "C"
