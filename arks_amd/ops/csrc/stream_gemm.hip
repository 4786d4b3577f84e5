// out[M, N] = a[M, K] . w[N, K]^T for few rows: the weights are read once and
// bound it. A workgroup takes 16 * NF weight rows; its WV waves split K into
// chunks of 64 in turn (each lane loads 16 B of a weight row straight into a
// matrix operand, two chunks in flight per wave) and meet in LDS, so no
// partial sums travel through memory. 128 x 2048 in fp32 (a router): 5 us,
// a library product with its conversion 11 us.
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

// Grid (tiles of 16 * NF weight rows, tiles of 16 rows of a). Rows past the
// end of a or w repeat the last one and are not stored.
template <int NF, int WV, typename OUT>
__global__ __launch_bounds__(WV * 64) void stream_gemm_kernel(
    OUT* __restrict__ out, const bf16* __restrict__ a,
    const bf16* __restrict__ w, const bf16* __restrict__ bias,
    const int m_rows, const int n_total, const int k_total,
    const int64_t a_stride) {
  __shared__ f32x4 red[WV][NF][WAVE_SIZE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lane = threadIdx.x % WAVE_SIZE, lq = lane % 16, la = lane / 16;
  const int n0 = blockIdx.x * 16 * NF, m0 = blockIdx.y * 16;
  const int own = (k_total / 64 - wave + WV - 1) / WV;  // chunks of this wave
  f32x4 acc[NF];
  const bf16* wp[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
    wp[f] = w + (int64_t)min(n0 + f * 16 + lq, n_total - 1) * k_total + 8 * la +
            wave * 64;
  }
  const bf16* ap =
      a + (int64_t)min(m0 + lq, m_rows - 1) * a_stride + 8 * la + wave * 64;
  struct Chunk {
    ushort8 w[NF][2], a[2];
  };
  auto load = [&](Chunk& c, const int i) {
    const int64_t o = (int64_t)i * WV * 64;
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        c.w[f][h] = *reinterpret_cast<const ushort8*>(wp[f] + o + 32 * h);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      c.a[h] = *reinterpret_cast<const ushort8*>(ap + o + 32 * h);
  };
  auto mul = [&](const Chunk& c) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int f = 0; f < NF; ++f)
        acc[f] = stream_mfma(c.w[f][h], c.a[h], acc[f]);
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
#pragma unroll
  for (int f = 0; f < NF; ++f) red[wave][f][lane] = acc[f];
  __syncthreads();
  for (int f = wave; f < NF; f += WV) {
    f32x4 s = red[0][f][lane];
#pragma unroll
    for (int v = 1; v < WV; ++v) s += red[v][f][lane];
    const int m = m0 + lq, n = n0 + f * 16 + 4 * la;
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
    if (n_total % 4 == 0) {  // n_total - n is one too
      if (n < n_total) __builtin_memcpy(__builtin_assume_aligned(to, 4 * sizeof(OUT)), o, sizeof(o));
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < n_total) to[r] = o[r];
    }
  }
}

}  // namespace arks

using namespace arks;

// nf: 1 or 2 row groups per workgroup; wv: 8 or 16 waves. out is contiguous,
// bf16 or (f32) fp32; bias null or bf16 [n]; k % 64 == 0, a rows 16 B aligned.
extern "C" void arks_stream_gemm(void* out, const void* a, const void* w,
                                 const void* bias, int m, int n, int k,
                                 int64_t a_stride, int nf, int wv, int f32,
                                 hipStream_t stream) {
#define ARKS_SG(NF, WV, OUT)                                                   \
  hipLaunchKernelGGL((stream_gemm_kernel<NF, WV, OUT>),                        \
                     dim3((n + 16 * NF - 1) / (16 * NF), (m + 15) / 16),       \
                     dim3(WV * 64), 0, stream, (OUT*)out, (const bf16*)a,      \
                     (const bf16*)w, (const bf16*)bias, m, n, k, a_stride)
#define ARKS_SG_O(NF, WV)                                                      \
  do {                                                                         \
    if (f32) ARKS_SG(NF, WV, float);                                           \
    else ARKS_SG(NF, WV, bf16);                                                \
  } while (0)
  if (nf == 1 && wv == 16) ARKS_SG_O(1, 16);
  else if (nf == 1) ARKS_SG_O(1, 8);
  else if (wv == 16) ARKS_SG_O(2, 16);
  else ARKS_SG_O(2, 8);
#undef ARKS_SG_O
#undef ARKS_SG
}
