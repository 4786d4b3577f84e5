// MoE routing + mixing kernels (gfx950), around the expert products of
// moe_gemm.hip. In torch the same steps (softmax -> topk -> renorm, then float
// casts and an einsum for the weighted mix) are about 10 small kernels a layer.
//
//   moe_topk:      probs = softmax(logits[T,E]); per row select top-k
//                  (ties -> lower expert id, matching torch.topk), optional
//                  renormalization; emits (weights[T,k] f32, ids[T,k] i32).
//   moe_mix_rows:  out[t] = sum_j w[t,j] * y[rows[t,j]], the weighted mix over
//                  the experts' rows y [R, H].
//
// The reference delegates MoE serving to external images; these kernels are
// internals of its runtime slot.
#include "common.h"
#include "moe_topk.h"
#include "parts.h"

namespace arks {

// One wave per token row.
template <int S>
__global__ __launch_bounds__(64) void moe_topk_kernel(
    float* __restrict__ weights,    // [T, k]
    int* __restrict__ ids,          // [T, k]
    const float* __restrict__ logits,  // [T, E]
    const int E, const int k, const int renorm) {
  const int t = blockIdx.x;
  const int lane = threadIdx.x;
  float weight;
  int id;
  moe_topk_row<S>(logits + (int64_t)t * E, E, k, renorm, lane, weight, id);
  if (lane < k) {
    weights[(int64_t)t * k + lane] = weight;
    ids[(int64_t)t * k + lane] = id;
  }
}

// One block per token over a flat [R, H] buffer of expert rows, in any order;
// rows[t,k] addresses each token's k of them. Reading them bounds it (no
// scatter, no atomics); zero-weight slots point at row 0.
__global__ __launch_bounds__(256) void moe_mix_rows_kernel(
    bf16* __restrict__ out,          // [T, H]
    const bf16* __restrict__ y,      // [R, H]
    const float* __restrict__ weights,  // [T, k]
    const int* __restrict__ rows,       // [T, k]
    const int T, const int H, const int k) {
  const int t = blockIdx.x;
  // by lanes of their own, the places behind the last row filled (as scalars, as
  // the norm that mixes has them, 16 tokens of 2 rows x 4096 take 3.8 us, so 3.4)
  __shared__ float w[16];
  __shared__ int64_t base[16];
  if (threadIdx.x < 16) {
    const int j = min((int)threadIdx.x, k - 1);
    w[threadIdx.x] = (int)threadIdx.x < k ? weights[(int64_t)t * k + j] : 0.f;
    base[threadIdx.x] = (int64_t)rows[(int64_t)t * k + j] * H;
  }
  __syncthreads();
  // loads of 16 bytes where rows start there
  if (H % 8 == 0 &&
      (reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(out)) % 16 == 0) {
    for (int h = threadIdx.x * 8; h < H; h += 256 * 8)
      *reinterpret_cast<ushort8*>(out + (int64_t)t * H + h) =
          mix_rows8(y, k, h, [&](int j) { return base[j]; },
                    [&](int j) { return w[j]; });
    return;
  }
  for (int h = threadIdx.x * 2; h < H; h += 256 * 2) {
    float a0 = 0.f, a1 = 0.f;
    for (int j = 0; j < k; ++j) {
      const uint32_t u = *reinterpret_cast<const uint32_t*>(y + base[j] + h);
      a0 += w[j] == 0.f ? 0.f : w[j] * bf16_bits_to_float((uint16_t)u);
      a1 += w[j] == 0.f ? 0.f : w[j] * bf16_bits_to_float((uint16_t)(u >> 16));
    }
    uint32_t packed = (uint32_t)float_to_bf16_bits(a0) |
                      ((uint32_t)float_to_bf16_bits(a1) << 16);
    *reinterpret_cast<uint32_t*>(out + (int64_t)t * H + h) = packed;
  }
}

}  // namespace arks

using namespace arks;

extern "C" void arks_moe_topk(void* weights, void* ids, const void* logits,
                              int T, int E, int k, int renorm,
                              hipStream_t stream) {
  dim3 grid(T), block(64);
#define ARKS_TOPK(S)                                                          \
  hipLaunchKernelGGL((moe_topk_kernel<S>), grid, block, 0, stream,            \
                     (float*)weights, (int*)ids, (const float*)logits, E, k,  \
                     renorm)
  if (E <= 128) ARKS_TOPK(2);
  else if (E <= 512) ARKS_TOPK(8);
  else ARKS_TOPK(16);
#undef ARKS_TOPK
}

extern "C" void arks_moe_mix_rows(void* out, const void* y,
                                  const void* weights, const void* rows,
                                  int T, int H, int k, hipStream_t stream) {
  dim3 grid(T), block(256);
  hipLaunchKernelGGL(moe_mix_rows_kernel, grid, block, 0, stream, (bf16*)out,
                     (const bf16*)y, (const float*)weights, (const int*)rows,
                     T, H, k);
}
