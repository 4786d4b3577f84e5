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
#include "parts.h"

namespace arks {

namespace {

using bf16x8_sg = __attribute__((ext_vector_type(8))) __bf16;

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

// For more rows than stream_gemm_kernel takes, and for few weight rows with
// long K: K is split over blockIdx.y too, and the fp32 sums of a split go to
// part [splits, M, N] for the consumer to add. 8 waves take 16 weight rows
// each and share the rows of a: KC columns of them at a time through two LDS
// buffers, fetched three chunks ahead, the weights PF chunks ahead in
// registers. The barriers wait for LDS alone, so the loads stay in flight.
// 3584 x 18944 (136 MB) in 8 splits: 8 rows 27 us, 64 rows 34 us, and 3 us
// for the sums where no consumer adds them; with barriers that drain the loads
// and 64 weight rows a workgroup 40 and 5 us, in the library 33 and 50 us.
// run: chunks of KC that a split takes, the last what is left; 0: even splits.
template <int MT, int KC, int PF>
__global__ __launch_bounds__(512) void stream_split_kernel(
    float* __restrict__ part, const bf16* __restrict__ a,
    const bf16* __restrict__ w, const int m_rows, const int n_total,
    const int k_total, const int64_t a_stride, const int splits,
    const int run) {
  static_assert(PF % 2 == 0, "buffers alternate over a round");
  constexpr int S = KC / 32, CPR = KC / 8, ITEMS = MT * 16 * CPR;
  constexpr int AI = (ITEMS + 511) / 512;
  __shared__ __attribute__((aligned(16))) bf16 lds[2][MT * 16][KC + 8];
  const int tid = threadIdx.x, lane = tid % WAVE_SIZE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE_SIZE);
  const int lq = lane % 16, la = lane / 16;
  const int n0 = (blockIdx.x * 8 + wave) * 16;
  const int chunks = k_total / KC;
  const int first = run > 0 ? blockIdx.y * run
                            : (int)((int64_t)chunks * blockIdx.y / splits);
  const int n = run > 0 ? min(run, chunks - first)
                        : (int)((int64_t)chunks * (blockIdx.y + 1) / splits) -
                              first;
  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bf16* wp = w + (int64_t)min(n0 + lq, n_total - 1) * k_total + 8 * la +
                   (int64_t)first * KC;
  const bf16* ap[AI];
#pragma unroll
  for (int t = 0; t < AI; ++t) {
    const int i = tid + t * 512;
    ap[t] = a + (int64_t)min(i / CPR, m_rows - 1) * a_stride + i % CPR * 8 +
            (int64_t)first * KC;
  }
  ushort8 wr[PF][S], ar[2][AI];
  auto load_w = [&](ushort8 (&r)[S], const int i) {
#pragma unroll
    for (int q = 0; q < S; ++q)
      r[q] = *reinterpret_cast<const ushort8*>(wp + (int64_t)i * KC + q * 32);
  };
  auto load_a = [&](ushort8 (&r)[AI], const int i) {
#pragma unroll
    for (int t = 0; t < AI; ++t)
      r[t] = *reinterpret_cast<const ushort8*>(ap[t] + (int64_t)i * KC);
  };
  auto store_a = [&](const ushort8 (&r)[AI], const int b) {
#pragma unroll
    for (int t = 0; t < AI; ++t) {
      const int i = tid + t * 512;
      if (ITEMS % 512 == 0 || i < ITEMS)
        *reinterpret_cast<ushort8*>(&lds[b][i / CPR][i % CPR * 8]) = r[t];
    }
  };
  auto mul = [&](const ushort8 (&r)[S], const int b) {
#pragma unroll
    for (int q = 0; q < S; ++q)
#pragma unroll
      for (int t = 0; t < MT; ++t)
        acc[t] = stream_mfma(r[q],
                             *reinterpret_cast<const ushort8*>(
                                 &lds[b][t * 16 + lq][q * 32 + 8 * la]),
                             acc[t]);
  };
  auto meet = [] {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  load_a(ar[0], 0);
#pragma unroll
  for (int j = 0; j < PF; ++j)
    if (j < n) load_w(wr[j], j);
  if (n > 1) load_a(ar[1], 1);
  store_a(ar[0], 0);
  if (n > 2) load_a(ar[0], 2);
  meet();
  int i = 0;
  for (; i + 2 * PF <= n && i + PF + 2 < n; i += PF) {
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      store_a(ar[(j + 1) & 1], (j + 1) & 1);
      load_a(ar[(j + 1) & 1], i + j + 3);
      mul(wr[j], j & 1);
      load_w(wr[j], i + j + PF);
      meet();
    }
  }
  for (; i < n; i += PF) {
#pragma unroll
    for (int j = 0; j < PF; ++j)
      if (i + j < n) {
        if (i + j + 1 < n) store_a(ar[(j + 1) & 1], (j + 1) & 1);
        if (i + j + 3 < n) load_a(ar[(j + 1) & 1], i + j + 3);
        mul(wr[j], j & 1);
        if (i + j + PF < n) load_w(wr[j], i + j + PF);
        meet();
      }
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = t * 16 + lq, col = n0 + 4 * la;
    if (m < m_rows && col < n_total)  // n_total % 4 == 0
      *reinterpret_cast<f32x4*>(
          part + ((int64_t)blockIdx.y * m_rows + m) * n_total + col) = acc[t];
  }
}

// out = the sum of the splits (+ bias), 4 columns a thread.
template <int U>
__global__ __launch_bounds__(256) void stream_sum_kernel(
    bf16* __restrict__ out, const float* __restrict__ part,
    const bf16* __restrict__ bias, const int64_t total, const int n_total,
    const int splits) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= total) return;
  f32x4 s = sum_parts4<U>(part + i, total, splits);
  ushort4v o;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    o[r] = float_to_bf16_bits(
        s[r] + (bias ? bf16_bits_to_float(bias[i % n_total + r]) : 0.f));
  *reinterpret_cast<ushort4v*>(out + i) = o;
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

// part [splits, m, n] fp32; m <= 64, n % 4 == 0. per 0: even splits, k % 64
// == 0; else columns of a split, k % 32 == per % 32 == 0 and (splits - 1) * per
// < k <= splits * per. Up to 32 rows chunks of 128 columns where K has them:
// 3584 x 18944, 32 rows 28.9 us, 64 of them 30.2.
extern "C" void arks_stream_split(void* part, const void* a, const void* w,
                                  int m, int n, int k, int64_t a_stride,
                                  int splits, int per, hipStream_t stream) {
#define ARKS_SS(MT, KC, PF)                                                    \
  hipLaunchKernelGGL((stream_split_kernel<MT, KC, PF>),                        \
                     dim3((n + 127) / 128, splits), dim3(512), 0, stream,      \
                     (float*)part, (const bf16*)a, (const bf16*)w, m, n, k,    \
                     a_stride, splits, per / KC)
  const int kc = per == 0 ? (k % 128 == 0 && splits <= k / 128 ? 128 : 64)
                 : (k | per) % 128 == 0 ? 128
                 : (k | per) % 64 == 0  ? 64
                                        : 32;
#define ARKS_SS_M(MT)                                                          \
  do {                                                                         \
    if (kc == 32) ARKS_SS(MT, 32, 8);                                          \
    else if (kc == 128) ARKS_SS(MT, 128, 2);                                   \
    else ARKS_SS(MT, 64, 4);                                                   \
  } while (0)
  switch ((m + 15) / 16) {
    case 1: ARKS_SS_M(1); break;
    case 2: ARKS_SS_M(2); break;
    case 3:
      if (kc == 32) ARKS_SS(3, 32, 8);
      else ARKS_SS(3, 64, 4);
      break;
    default:
      if (kc == 32) ARKS_SS(4, 32, 8);
      else ARKS_SS(4, 64, 4);
      break;
  }
#undef ARKS_SS_M
#undef ARKS_SS
}

extern "C" void arks_stream_sum(void* out, const void* part, const void* bias,
                                int64_t m, int n, int splits,
                                hipStream_t stream) {
  const int64_t total = m * n;
#define ARKS_SUM(U)                                                            \
  hipLaunchKernelGGL((stream_sum_kernel<U>), dim3((total / 4 + 255) / 256),    \
                     dim3(256), 0, stream, (bf16*)out, (const float*)part,     \
                     (const bf16*)bias, total, n, splits)
  const int u = parts_flight(splits);
  if (u == 2) ARKS_SUM(2);
  else if (u == 4) ARKS_SUM(4);
  else ARKS_SUM(8);
#undef ARKS_SUM
}
