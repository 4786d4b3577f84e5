// Paged KV-cache scatter: write the new tokens' K/V into their assigned slots.
// Cache layout: [num_blocks, num_kv_heads, block_size, head_dim] bf16
// slot = block_id * block_size + offset  (flat, per token)
#include "common.h"
#include "parts.h"

#include <hip/hip_fp8.h>

namespace arks {

__global__ void reshape_and_cache_kernel(
    const bf16* __restrict__ k,  // [T, Hkv, D], token rows strided
    const bf16* __restrict__ v,
    bf16* __restrict__ k_cache,  // [B, Hkv, block_size, D]
    bf16* __restrict__ v_cache,
    const int64_t* __restrict__ slot_mapping,  // [T]
    const int num_kv_heads, const int head_dim, const int block_size,
    const int64_t kv_stride) {
  const int token = blockIdx.x;
  const int64_t slot = slot_mapping[token];
  if (slot < 0) return;  // padding slot
  const int64_t block_id = slot / block_size;
  const int offset = (int)(slot % block_size);
  const int nvec = num_kv_heads * head_dim / 8;
  const bf16* k_src = k + (int64_t)token * kv_stride;
  const bf16* v_src = v + (int64_t)token * kv_stride;
  for (int i = threadIdx.x; i < nvec; i += blockDim.x) {
    const int h = (i * 8) / head_dim;
    const int d = (i * 8) % head_dim;
    const int64_t dst = ((block_id * num_kv_heads + h) * block_size + offset) *
                            head_dim + d;
    *reinterpret_cast<ushort8*>(k_cache + dst) =
        *reinterpret_cast<const ushort8*>(k_src + i * 8);
    *reinterpret_cast<ushort8*>(v_cache + dst) =
        *reinterpret_cast<const ushort8*>(v_src + i * 8);
  }
}

__global__ void reshape_and_cache_fp8_kernel(
    const bf16* __restrict__ k,  // [T, Hkv, D], token rows strided
    const bf16* __restrict__ v,
    uint8_t* __restrict__ k_cache,  // [B, Hkv, block_size, D] e4m3
    uint8_t* __restrict__ v_cache,
    const int64_t* __restrict__ slot_mapping,  // [T]
    const int num_kv_heads, const int head_dim, const int block_size,
    const int64_t kv_stride) {
  const int token = blockIdx.x;
  const int64_t slot = slot_mapping[token];
  if (slot < 0) return;  // padding slot
  const int64_t block_id = slot / block_size;
  const int offset = (int)(slot % block_size);
  const int nvec = num_kv_heads * head_dim / 8;
  const bf16* k_src = k + (int64_t)token * kv_stride;
  const bf16* v_src = v + (int64_t)token * kv_stride;
  for (int i = threadIdx.x; i < nvec; i += blockDim.x) {
    const int h = (i * 8) / head_dim;
    const int d = (i * 8) % head_dim;
    const int64_t dst = ((block_id * num_kv_heads + h) * block_size + offset) *
                            head_dim + d;
    ushort8 kv8 = *reinterpret_cast<const ushort8*>(k_src + i * 8);
    ushort8 vv8 = *reinterpret_cast<const ushort8*>(v_src + i * 8);
    uchar8 ko, vo;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      __hip_fp8_e4m3 kq(bf16_bits_to_float(kv8[e]));
      __hip_fp8_e4m3 vq(bf16_bits_to_float(vv8[e]));
      ko[e] = kq.__x;
      vo[e] = vq.__x;
    }
    *reinterpret_cast<uchar8*>(k_cache + dst) = ko;
    *reinterpret_cast<uchar8*>(v_cache + dst) = vo;
  }
}

}  // namespace arks

using namespace arks;

extern "C" void arks_reshape_and_cache_fp8(
    const void* k, const void* v, void* k_cache, void* v_cache,
    const void* slot_mapping, int num_tokens, int num_kv_heads, int head_dim,
    int block_size, int64_t kv_stride, hipStream_t stream) {
  if (num_tokens == 0) return;
  int threads = std::min(256, num_kv_heads * head_dim / 8);
  hipLaunchKernelGGL(reshape_and_cache_fp8_kernel, dim3(num_tokens),
                     dim3(threads), 0, stream, (const bf16*)k, (const bf16*)v,
                     (uint8_t*)k_cache, (uint8_t*)v_cache,
                     (const int64_t*)slot_mapping, num_kv_heads, head_dim,
                     block_size, kv_stride);
}

extern "C" void arks_reshape_and_cache(const void* k, const void* v,
                                       void* k_cache, void* v_cache,
                                       const void* slot_mapping, int num_tokens,
                                       int num_kv_heads, int head_dim,
                                       int block_size, int64_t kv_stride,
                                       hipStream_t stream) {
  if (num_tokens == 0) return;
  int threads = std::min(256, num_kv_heads * head_dim / 8);
  hipLaunchKernelGGL(reshape_and_cache_kernel, dim3(num_tokens), dim3(threads),
                     0, stream, (const bf16*)k, (const bf16*)v, (bf16*)k_cache,
                     (bf16*)v_cache, (const int64_t*)slot_mapping, num_kv_heads,
                     head_dim, block_size, kv_stride);
}

namespace arks {

// ---------------------------------------------------------------------------
// Fused RoPE + cache write: rotate q/k in place AND scatter the rotated k
// (plus v) into the paged cache in one launch — the separate
// rope_kernel + reshape_and_cache pair cost a kernel boundary and a full
// re-read of k every layer on the decode path. The rotating thread already
// holds the rotated k values in registers, so the cache store is free.
// Thread space: [q heads | kv heads] x pair-couples for the rotation, then
// the v copy strided over the same block.
// NORM: q and k heads are RMS-normed on the way (a head's head_dim / 4
// consecutive lanes share its sum of squares; the normed values stay fp32
// until the rotated ones are rounded). As separate passes the two norms and
// the contiguous copies that they need cost 14 us per layer at 7 rows and
// 100 us at 5012 (32/4 heads x 128).
// PARTS: q, k and v are the sums of fp32 splits [splits, T, q | k | v] of the
// projection (+ bias); k and v go to the cache alone. Saves the launch that
// would add them (5 us at 64 rows of 4608).
// W: pairs of a thread. Many tokens take 8 where rows and bases lie on 16 bytes:
// one access of 16 bytes per half of a head instead of four, and a workgroup of
// as many threads as a token has work. 5012 rows of 32/4 heads x 128 with norms
// 35.3 -> 28.4 us, 8192 of 28/4 without 35 -> 30.6 (of about 27 for the bytes).
// Few tokens and split sums keep 2: a thread's chain of loads is what they wait
// for.
// ---------------------------------------------------------------------------
template <bool FP8, bool NORM, bool PARTS, int W, int U = 8>
__global__ void rope_cache_kernel(
    const int64_t* __restrict__ positions,
    bf16* __restrict__ q,        // [T, Hq*D] rows strided
    bf16* __restrict__ k,        // [T, Hkv*D] rows strided
    const bf16* __restrict__ v,  // [T, Hkv*D] rows strided (k_stride)
    void* __restrict__ k_cache,  // [B, Hkv, block_size, D] bf16 or e4m3
    void* __restrict__ v_cache,
    const int64_t* __restrict__ slot_mapping,  // [T] (-1 = no cache write)
    const float* __restrict__ cos_sin,         // [max_pos, D]
    const int head_dim, const int num_q_heads, const int num_kv_heads,
    const int block_size, const int64_t q_stride, const int64_t k_stride,
    const bf16* __restrict__ q_norm, const bf16* __restrict__ k_norm,
    const float eps, const float* __restrict__ part,
    const bf16* __restrict__ bias, const int splits) {
  const int token = blockIdx.x;
  const int width = (num_q_heads + 2 * num_kv_heads) * head_dim;
  const int64_t part_stride = (int64_t)gridDim.x * width;
  const float* part_row = part + (int64_t)token * width;
  const int half = head_dim / 2;
  const int64_t pos = positions[token];
  const float* cs = cos_sin + pos * head_dim;
  const int64_t slot = slot_mapping[token];
  const bool cache = slot >= 0;
  // (a division of 64 bits would be a long chain in front of the stores)
  int64_t block_id = 0;
  int offset = 0;
  if (cache && slot <= 0x7fffffff) {
    block_id = (uint32_t)slot / (uint32_t)block_size;
    offset = (uint32_t)slot % (uint32_t)block_size;
  } else if (cache) {
    block_id = slot / block_size;
    offset = (int)(slot % block_size);
  }
  const int64_t cbase =
      (block_id * num_kv_heads) * (int64_t)block_size * head_dim +
      (int64_t)offset * head_dim;
  const int64_t hstride = (int64_t)block_size * head_dim;

  const int total_heads = num_q_heads + num_kv_heads;
  typedef __attribute__((ext_vector_type(W))) unsigned short bits;
  const int lanes = half / W;  // threads of a head
  const int first = blockIdx.y * blockDim.x + threadIdx.x;
  const int step = gridDim.y * blockDim.x;
  for (int idx = first; idx < total_heads * lanes; idx += step) {
    const int h = idx / lanes;
    const int p2 = (idx % lanes) * W;
    const bool is_q = h < num_q_heads;
    bf16* base = is_q
                     ? q + (int64_t)token * q_stride + (int64_t)h * head_dim
                     : k + (int64_t)token * k_stride +
                           (int64_t)(h - num_q_heads) * head_dim;
    bits o1, o2;
    float a2[W], b2[W];
    if constexpr (PARTS) {
      static_assert(W == 2);
      const int c = h * head_dim + p2;
      f32x2 f1, f2;
      sum_parts_pair<U>(part_row + c, part_row + c + half, part_stride, splits,
                        f1, f2);
      a2[0] = f1.x, a2[1] = f1.y, b2[0] = f2.x, b2[1] = f2.y;
      if (bias) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          a2[j] += bf16_bits_to_float(bias[c + j]);
          b2[j] += bf16_bits_to_float(bias[c + half + j]);
        }
      }
    } else {
      const bits x1 = *reinterpret_cast<const bits*>(base + p2);
      const bits x2 = *reinterpret_cast<const bits*>(base + half + p2);
#pragma unroll
      for (int j = 0; j < W; ++j) {
        a2[j] = bf16_bits_to_float(x1[j]);
        b2[j] = bf16_bits_to_float(x2[j]);
      }
    }
    if constexpr (NORM) {
      float sa = 0.f, sb = 0.f;
#pragma unroll
      for (int j = 0; j < W; ++j) {
        sa += a2[j] * a2[j];
        sb += b2[j] * b2[j];
      }
      float ss = sa + sb;
      for (int off = lanes / 2; off > 0; off >>= 1)
        ss += __shfl_xor(ss, off, WAVE_SIZE);
      const float r = rsqrtf(ss / (float)head_dim + eps);
      const bf16* nw = is_q ? q_norm : k_norm;
#pragma unroll
      for (int j = 0; j < W; ++j) {
        a2[j] *= r * bf16_bits_to_float(nw[p2 + j]);
        b2[j] *= r * bf16_bits_to_float(nw[half + p2 + j]);
      }
    }
#pragma unroll
    for (int j = 0; j < W; ++j) {
      const float c = cs[p2 + j];
      const float s = cs[half + p2 + j];
      const float a = a2[j];
      const float b = b2[j];
      o1[j] = float_to_bf16_bits(a * c - b * s);
      o2[j] = float_to_bf16_bits(b * c + a * s);
    }
    if (!PARTS || is_q) {
      *reinterpret_cast<bits*>(base + p2) = o1;
      *reinterpret_cast<bits*>(base + half + p2) = o2;
    }
    if (!is_q && cache) {
      const int64_t dst = cbase + (int64_t)(h - num_q_heads) * hstride;
      if constexpr (FP8) {
        uint8_t* kc = reinterpret_cast<uint8_t*>(k_cache);
        typedef __attribute__((ext_vector_type(W))) unsigned char bytes;
        bytes y1, y2;
#pragma unroll
        for (int j = 0; j < W; ++j) {
          // convert from the bf16-ROUNDED values so the cache is
          // bit-identical to the separate rope + reshape_and_cache path
          __hip_fp8_e4m3 a(bf16_bits_to_float(o1[j]));
          __hip_fp8_e4m3 b(bf16_bits_to_float(o2[j]));
          y1[j] = a.__x;
          y2[j] = b.__x;
        }
        *reinterpret_cast<bytes*>(kc + dst + p2) = y1;
        *reinterpret_cast<bytes*>(kc + dst + half + p2) = y2;
      } else {
        bf16* kc = reinterpret_cast<bf16*>(k_cache);
        *reinterpret_cast<bits*>(kc + dst + p2) = o1;
        *reinterpret_cast<bits*>(kc + dst + half + p2) = o2;
      }
    }
  }
  if (!cache) return;
  // v: plain copy into the page (vectorized 8)
  const bf16* v_src = v + (int64_t)token * k_stride;
  const int nvec = num_kv_heads * head_dim / 8;
  for (int i = first; i < nvec; i += step) {
    const int h = (i * 8) / head_dim;
    const int d = (i * 8) % head_dim;
    const int64_t dst = cbase + (int64_t)h * hstride + d;
    ushort8 vv8;
    if constexpr (PARTS) {
      const int c = (num_q_heads + num_kv_heads) * head_dim + i * 8;
      f32x4 lo, hi;
      sum_parts_pair<U>(part_row + c, part_row + c + 4, part_stride, splits, lo,
                        hi);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float b = bias ? bf16_bits_to_float(bias[c + e]) : 0.f;
        vv8[e] = float_to_bf16_bits((e < 4 ? lo[e % 4] : hi[e % 4]) + b);
      }
    } else {
      vv8 = *reinterpret_cast<const ushort8*>(v_src + i * 8);
    }
    if constexpr (FP8) {
      uchar8 vo;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        __hip_fp8_e4m3 vq(bf16_bits_to_float(vv8[e]));
        vo[e] = vq.__x;
      }
      *reinterpret_cast<uchar8*>(reinterpret_cast<uint8_t*>(v_cache) + dst) = vo;
    } else {
      *reinterpret_cast<ushort8*>(reinterpret_cast<bf16*>(v_cache) + dst) = vv8;
    }
  }
}

}  // namespace arks

// Workgroups per token: few tokens leave most CUs idle, so each thread gets one
// couple of pairs. 64 tokens of 28/4 heads x 128, with 8 splits to add: 1 group
// 12.2 us, 4 groups 7.1 us.
static int rope_groups(int num_tokens, int heads, int head_dim) {
  return num_tokens > 256 ? 1 : (heads * (head_dim / 4) + 255) / 256;
}

// q_norm, k_norm: null, or bf16 [head_dim] weights of the heads' RMS norms
// (head_dim 32, 64, 128 or 256).
extern "C" void arks_rope_and_cache(
    const void* positions, void* q, void* k, const void* v, void* k_cache,
    void* v_cache, const void* slot_mapping, const void* cos_sin,
    int num_tokens, int head_dim, int num_q_heads, int num_kv_heads,
    int block_size, int64_t q_stride, int64_t k_stride, int kv_fp8,
    const void* q_norm, const void* k_norm, float eps, hipStream_t stream) {
  if (num_tokens == 0) return;
  const int heads = num_q_heads + num_kv_heads;
  const bool wide =
      num_tokens > 256 && head_dim % 16 == 0 && q_stride % 8 == 0 &&
      k_stride % 8 == 0 &&
      (((uintptr_t)q | (uintptr_t)k | (uintptr_t)k_cache | (uintptr_t)cos_sin |
        (uintptr_t)q_norm | (uintptr_t)k_norm) & 15) == 0;
  dim3 grid(num_tokens, rope_groups(num_tokens, heads, head_dim)), block(256);
  if (wide) block.x = std::min(512, (heads * (head_dim / 16) + 63) / 64 * 64);
#define ARKS_ROPE(FP8, NORM)                                                   \
  if (wide) ARKS_ROPE_W(FP8, NORM, 8); else ARKS_ROPE_W(FP8, NORM, 2)
#define ARKS_ROPE_W(FP8, NORM, W)                                              \
  hipLaunchKernelGGL((rope_cache_kernel<FP8, NORM, false, W>), grid, block, 0, \
                     stream,                                                   \
                     (const int64_t*)positions, (bf16*)q, (bf16*)k,            \
                     (const bf16*)v, k_cache, v_cache,                         \
                     (const int64_t*)slot_mapping, (const float*)cos_sin,      \
                     head_dim, num_q_heads, num_kv_heads, block_size,          \
                     q_stride, k_stride, (const bf16*)q_norm,                  \
                     (const bf16*)k_norm, eps, nullptr, nullptr, 0)
  if (kv_fp8 && q_norm) {
    ARKS_ROPE(true, true);
  } else if (kv_fp8) {
    ARKS_ROPE(true, false);
  } else if (q_norm) {
    ARKS_ROPE(false, true);
  } else {
    ARKS_ROPE(false, false);
  }
#undef ARKS_ROPE_W
#undef ARKS_ROPE
}

extern "C" void arks_rope_and_cache_parts(
    const void* positions, void* q, const void* part, const void* bias,
    int splits, void* k_cache, void* v_cache, const void* slot_mapping,
    const void* cos_sin, int num_tokens, int head_dim, int num_q_heads,
    int num_kv_heads, int block_size, int kv_fp8, const void* q_norm,
    const void* k_norm, float eps, hipStream_t stream) {
  dim3 grid(num_tokens,
            rope_groups(num_tokens, num_q_heads + num_kv_heads, head_dim)),
      block(256);
#define ARKS_ROPE(FP8, NORM)                                                   \
  do {                                                                         \
    const int u = parts_flight(splits);                                        \
    if (u == 2) ARKS_ROPE_U(FP8, NORM, 2);                                     \
    else if (u == 4) ARKS_ROPE_U(FP8, NORM, 4);                                \
    else ARKS_ROPE_U(FP8, NORM, 8);                                            \
  } while (0)
#define ARKS_ROPE_U(FP8, NORM, U)                                              \
  hipLaunchKernelGGL((rope_cache_kernel<FP8, NORM, true, 2, U>), grid, block,  \
                     0, stream, (const int64_t*)positions, (bf16*)q, nullptr,     \
                     nullptr, k_cache, v_cache, (const int64_t*)slot_mapping,  \
                     (const float*)cos_sin, head_dim, num_q_heads,             \
                     num_kv_heads, block_size,                                 \
                     (int64_t)num_q_heads * head_dim, 0, (const bf16*)q_norm,  \
                     (const bf16*)k_norm, eps, (const float*)part,             \
                     (const bf16*)bias, splits)
  if (kv_fp8) {
    if (q_norm) ARKS_ROPE(true, true); else ARKS_ROPE(true, false);
  } else {
    if (q_norm) ARKS_ROPE(false, true); else ARKS_ROPE(false, false);
  }
#undef ARKS_ROPE
#undef ARKS_ROPE_U
}
