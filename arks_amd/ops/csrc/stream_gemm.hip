// out[M, N] = a[M, K] . w[N, K]^T for few rows: the weights are read once and
// bound it. A workgroup takes 16 * NF weight rows; its WV waves split K into
// chunks of 64 in turn (each lane loads 16 B of a weight row straight into a
// matrix operand, two chunks in flight per wave) and meet in LDS, so no
// partial sums travel through memory and no second launch adds them. One row:
// 3584 x 3584 in 7.4 us (3.5 TB/s; split over workgroups with a second launch
// 14.1), 28672 x 4096 in 46 us (5.1 TB/s; library 64), 151936 x 2048 in
// 108 us (5.8 TB/s; library 205). 128 x 2048 in fp32 (a router): 5 us, a
// library product with its conversion 11 us. With more rows the loads of a,
// one set per workgroup, take over: 151936 x 2048, 16 rows 134 us.
#include "common.h"

namespace arks {

namespace {

using bf16x8_sg = __attribute__((ext_vector_type(8))) __bf16;
using f32x4 = __attribute__((ext_vector_type(4))) float;

__device__ __forceinline__ f32x4 stream_mfma(const ushort8& w, const ushort8& a,
                                             const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
      *reinterpret_cast<const bf16x8_sg*>(&w),
      *reinterpret_cast<const bf16x8_sg*>(&a), c, 0, 0, 0);
}

}  // namespace

__device__ __forceinline__ float stream_silu_mul(float g, float u) {
  return g / (1.f + __expf(-g)) * u;
}

// Grid (tiles of 16 * NF weight rows, tiles of 16 * MT rows of a). Rows past
// the end of a or w repeat the last one and are not stored. SILU (NF 2): w is
// [2 * n_total, K], a workgroup takes 16 gate rows and their up rows and
// stores silu(gate) * up.
template <int MT, int NF, int WV, bool SILU, typename OUT>
__global__ __launch_bounds__(WV * 64) void stream_gemm_kernel(
    OUT* __restrict__ out, const bf16* __restrict__ a,
    const bf16* __restrict__ w, const bf16* __restrict__ bias,
    const int m_rows, const int n_total, const int k_total,
    const int64_t a_stride) {
  __shared__ f32x4 red[WV][NF * MT][WAVE_SIZE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE, lq = lane % 16, la = lane / 16;
  const int n0 = blockIdx.x * (SILU ? 16 : 16 * NF), m0 = blockIdx.y * 16 * MT;
  const int chunks = k_total / 64;
  const int own = (chunks - wave + WV - 1) / WV;  // chunks of this wave
  f32x4 acc[NF][MT];
  const bf16* wp[NF];
  const bf16* ap[MT];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[f][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int64_t n = min(n0 + (SILU ? 0 : f * 16) + lq, n_total - 1);
    wp[f] = w + (n + (SILU ? (int64_t)f * n_total : 0)) * k_total + 8 * la +
            wave * 64;
  }
#pragma unroll
  for (int t = 0; t < MT; ++t)
    ap[t] = a + (int64_t)min(m0 + t * 16 + lq, m_rows - 1) * a_stride + 8 * la +
            wave * 64;
  struct Chunk {
    ushort8 w[NF][2], a[MT][2];
  };
  auto load_half = [&](Chunk& c, const int64_t o, const int h) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
      c.w[f][h] = *reinterpret_cast<const ushort8*>(wp[f] + o + 32 * h);
#pragma unroll
    for (int t = 0; t < MT; ++t)
      c.a[t][h] = *reinterpret_cast<const ushort8*>(ap[t] + o + 32 * h);
  };
  auto load = [&](Chunk& c, const int i) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        c.w[f][h] = *reinterpret_cast<const ushort8*>(
            wp[f] + (int64_t)i * WV * 64 + 32 * h);
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        c.a[t][h] = *reinterpret_cast<const ushort8*>(
            ap[t] + (int64_t)i * WV * 64 + 32 * h);
  };
  auto mul_half = [&](const Chunk& c, const int h) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int t = 0; t < MT; ++t)
        acc[f][t] = stream_mfma(c.w[f][h], c.a[t][h], acc[f][t]);
  };
  auto mul = [&](const Chunk& c) {
    mul_half(c, 0);
    mul_half(c, 1);
  };
  if (own > 0) {
    Chunk c0, c1;
    load(c0, 0);
    if (own > 1) load(c1, 1);
    int i = 0;
    for (; i + 3 < own; i += 2) {
      mul(c0);
      load(c0, i + 2);
      mul(c1);
      load(c1, i + 3);
    }
    const int left = own - i;
    mul(c0);
    if (left > 2) load(c0, i + 2);
    if (left > 1) mul(c1);
    if (left > 2) mul(c0);
  }
  // K % 64 == 32: the half chunk goes to the wave whose turn it is
  if (k_total % 64 != 0 && wave == chunks % WV) {
    Chunk c0;
    load_half(c0, (int64_t)own * WV * 64, 0);
    mul_half(c0, 0);
  }
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int t = 0; t < MT; ++t) red[wave][f * MT + t][lane] = acc[f][t];
  __syncthreads();
  auto total = [&](const int x) {
    f32x4 s = red[0][x][lane];
#pragma unroll
    for (int v = 1; v < WV; ++v) s += red[v][x][lane];
    return s;
  };
  for (int x = wave; x < (SILU ? MT : NF * MT); x += WV) {
    f32x4 s = total(x);
    if constexpr (SILU) {
      const f32x4 u = total(MT + x);
#pragma unroll
      for (int r = 0; r < 4; ++r) s[r] = stream_silu_mul(s[r], u[r]);
    }
    const int m = m0 + (x % MT) * 16 + lq, n = n0 + (x / MT) * 16 + 4 * la;
    if (m >= m_rows) continue;
    OUT o[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float b =
          bias ? bf16_bits_to_float(bias[min(n + r, n_total - 1)]) : 0.f;
      if constexpr (sizeof(OUT) == 2) o[r] = float_to_bf16_bits(s[r] + b);
      else o[r] = s[r] + b;
    }
    OUT* to = out + (int64_t)m * n_total + n;
    if (n_total % 4 == 0) {  // n_total - n is a multiple of 4 too
      if (n < n_total)
        __builtin_memcpy(__builtin_assume_aligned(to, 4 * sizeof(OUT)), o,
                         sizeof(o));
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < n_total) to[r] = o[r];
    }
  }
}

}  // namespace arks

using namespace arks;

// mt: row tiles of 16 per workgroup (1, 2); nf: groups of 16 weight rows (1,
// 2); wv: waves. (nf, wv) is one of (1, 4), (1, 16), (2, 8), (2, 16). out is
// contiguous, bf16 or (f32) fp32, silu: bf16 of n columns under w [2n, k];
// bias null or bf16 [n]; k % 32 == 0, rows of a and w on 16 bytes.
extern "C" void arks_stream_gemm(void* out, const void* a, const void* w,
                                 const void* bias, int m, int n, int k,
                                 int64_t a_stride, int mt, int nf, int wv,
                                 int f32, int silu, hipStream_t stream) {
#define ARKS_SG(MT, NF, WV, SILU, OUT)                                         \
  hipLaunchKernelGGL((stream_gemm_kernel<MT, NF, WV, SILU, OUT>),              \
                     dim3((n + (SILU ? 16 : 16 * NF) - 1) /                    \
                              (SILU ? 16 : 16 * NF),                           \
                          (m + 16 * MT - 1) / (16 * MT)),                      \
                     dim3(WV * 64), 0, stream, (OUT*)out, (const bf16*)a,      \
                     (const bf16*)w, (const bf16*)bias, m, n, k, a_stride)
#define ARKS_SG_O(MT, NF, WV)                                                  \
  do {                                                                         \
    if (f32) ARKS_SG(MT, NF, WV, false, float);                                \
    else ARKS_SG(MT, NF, WV, false, bf16);                                     \
  } while (0)
  if (silu) {
    if (mt == 1 && wv == 16) ARKS_SG(1, 2, 16, true, bf16);
    else if (mt == 1) ARKS_SG(1, 2, 8, true, bf16);
    else if (wv == 16) ARKS_SG(2, 2, 16, true, bf16);
    else ARKS_SG(2, 2, 8, true, bf16);
  } else if (mt == 1) {
    if (nf == 1 && wv == 4) ARKS_SG_O(1, 1, 4);
    else if (nf == 1) ARKS_SG_O(1, 1, 16);
    else if (wv == 8) ARKS_SG_O(1, 2, 8);
    else ARKS_SG_O(1, 2, 16);
  } else {
    if (nf == 1 && wv == 4) ARKS_SG_O(2, 1, 4);
    else if (nf == 1) ARKS_SG_O(2, 1, 16);
    else if (wv == 8) ARKS_SG_O(2, 2, 8);
    else ARKS_SG_O(2, 2, 16);
  }
#undef ARKS_SG_O
#undef ARKS_SG
}
