// Python bindings for the arks_amd gfx950 kernels (torch extension).
// Host-side validation lives here; kernels are in the *.hip files.
#include <torch/extension.h>

#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>

#include <array>
#include <cstring>
#include <string>
#include <vector>

namespace py = pybind11;

#include "attn_bindings.h"

// --- kernel launchers (see the .hip files) ---
extern "C" {
void arks_rmsnorm(void* out, const void* input, const void* weight, float eps,
                  int rows, int hidden, hipStream_t stream);
void arks_fused_add_rmsnorm(void* out, const void* input, void* residual,
                            const void* weight, float eps, int rows, int hidden,
                            hipStream_t stream);
void arks_fused_add_rmsnorm_parts(void* out, const void* part, int splits,
                                  void* residual, const void* weight, float eps,
                                  int rows, int hidden, hipStream_t stream);
void arks_fused_add_rmsnorm_mix(void* out, const void* input,
                                const void* mix_weights, const void* mix_rows,
                                int k, void* residual, const void* weight,
                                float eps, int rows, int hidden,
                                hipStream_t stream);
void arks_rope_and_cache_parts(const void* positions, void* q, const void* part,
                               const void* bias, int splits, void* k_cache,
                               void* v_cache, const void* slot_mapping,
                               const void* cos_sin, int num_tokens,
                               int head_dim, int num_q_heads, int num_kv_heads,
                               int block_size, int kv_fp8, const void* q_norm,
                               const void* k_norm, float eps,
                               hipStream_t stream);
void arks_silu_mul(void* out, const void* gate_up, int64_t rows, int d,
                   hipStream_t stream);
void arks_rope_inplace(const void* positions, void* q, void* k,
                       const void* cos_sin, int num_tokens, int head_dim,
                       int num_q_heads, int num_kv_heads, int64_t q_stride,
                       int64_t k_stride, hipStream_t stream);
void arks_reshape_and_cache(const void* k, const void* v, void* k_cache,
                            void* v_cache, const void* slot_mapping,
                            int num_tokens, int num_kv_heads, int head_dim,
                            int block_size, int64_t kv_stride,
                            hipStream_t stream);
void arks_reshape_and_cache_fp8(const void* k, const void* v, void* k_cache,
                                void* v_cache, const void* slot_mapping,
                                int num_tokens, int num_kv_heads, int head_dim,
                                int block_size, int64_t kv_stride,
                                hipStream_t stream);
void arks_rope_and_cache(const void* positions, void* q, void* k,
                         const void* v, void* k_cache, void* v_cache,
                         const void* slot_mapping, const void* cos_sin,
                         int num_tokens, int head_dim, int num_q_heads,
                         int num_kv_heads, int block_size, int64_t q_stride,
                         int64_t k_stride, int kv_fp8, const void* q_norm,
                         const void* k_norm, float eps, hipStream_t stream);
void arks_attn_prefill_varlen(void* out, const void* q, const void* k,
                              const void* v, const void* cu_seqlens,
                              const void* tile_info, int ntiles, float scale,
                              int num_q_heads, int num_kv_heads, int head_dim,
                              int64_t q_stride, int64_t kv_stride, int window,
                              hipStream_t stream);
void arks_quant_fp8_rows(void* out, void* inv_scale, const void* x, int rows,
                         int cols, hipStream_t stream);
void arks_rmsnorm_fp8(void* out, void* inv_scale, const void* input,
                      void* residual, const void* weight, float eps, int rows,
                      int hidden, int fused_add, hipStream_t stream);
void arks_silu_mul_fp8(void* out, void* inv_scale, const void* gate_up,
                       int rows, int d, hipStream_t stream);
void arks_sample(void* out, void* part_val, void* part_idx, const void* logits,
                 const void* temperatures, const void* uniform, int rows,
                 int vocab, int parts, hipStream_t stream);
void arks_ar_seq_inc(void* seq, hipStream_t stream);
void arks_one_shot_allreduce(void* out, const void* src, void* mail_ptrs[8],
                             void* flag_ptrs[8], void* seq, int rank,
                             int world, int64_t n, hipStream_t stream);
void arks_moe_topk(void* weights, void* ids, const void* logits, int T,
                   int E, int k, int renorm, hipStream_t stream);
void arks_moe_mix_rows(void* out, const void* y, const void* weights,
                       const void* rows, int T, int H, int k,
                       hipStream_t stream);
void arks_stream_gemm(void* out, const void* a, const void* w, const void* bias,
                      int m, int n, int k, int64_t a_stride, int mt, int nf,
                      int wv, int f32, int silu, hipStream_t stream);
void arks_stream_split(void* part, const void* a, const void* w, int m, int n,
                       int k, int64_t a_stride, int splits, int per,
                       hipStream_t stream);
void arks_stream_sum(void* out, const void* part, const void* bias, int64_t m,
                     int n, int splits, hipStream_t stream);
void arks_tile_silu(void* out, const void* a, const void* w, int m, int n,
                    int k, int64_t a_stride, hipStream_t stream);
int arks_wide_gemm(void* out, const void* a, const void* w, const void* bias,
                   int m, int n, int k, int64_t a_stride, int tm, int tw,
                   int splits, int kind, hipStream_t stream);
void arks_mid_gemm(void* out, const void* a, const void* w, const void* bias,
                   int m, int n, int k, int64_t a_stride, int qt, int splits,
                   int parts, int silu, hipStream_t stream);
void arks_mid_pair(void* out, const void* a, const void* w, int k,
                   int64_t a_stride, int splits, const void* a2, const void* w2,
                   int k2, int64_t a_stride2, int splits2, int m, int n, int qt,
                   hipStream_t stream);
void arks_mid_items(void* out, const void* a, const void* w, const void* perm,
                    const void* items, const void* n_items, int64_t a_stride,
                    int64_t w_expert, int n, int k, int top_k, int expert_base,
                    int max_items, int ft, int qt, int silu,
                    hipStream_t stream);
void arks_moe_plan(void* perm, void* rows, void* weights_out, void* items,
                   void* n_items, void* claims, void* counts, const void* ids,
                   const void* weights, int pairs, int expert_base, int n_local,
                   int tile, int max_items, int groups, const int* rounds,
                   hipStream_t stream);
void arks_moe_plan_topk(void* perm, void* rows, void* weights_out, void* items,
                        void* n_items, void* claims, const void* logits,
                        int experts, int k, int renorm, int pairs, int expert_base,
                        int n_local, int tile, int max_items, const int* rounds,
                        hipStream_t stream);
void arks_moe_gemm(void* out, const void* a, const void* w, const void* perm,
                   const void* items, const void* n_items, void* claims, const void* scale,
                   int64_t a_stride, int64_t w_expert, int64_t w_stride, int n_out, int k_total,
                   int top_k, int max_items, int tile, int up,
                   int once, int expert_base, hipStream_t stream);
void arks_mfma_probe(void* d, const void* a, const void* b, hipStream_t stream);
void arks_mfma_probe32(void* d, const void* a, const void* b, hipStream_t stream);
void arks_tr16_probe(void* out, int stride_bytes, hipStream_t stream);
}

namespace {

hipStream_t current_stream() {
  return c10::hip::getCurrentHIPStream().stream();
}

// KV caches may be bf16 or fp8 e4m3 (kv_cache_dtype="fp8"); returns fp8?


// bf16 tensor whose trailing dims are contiguous; dim-0 rows may be strided
// (a view into the fused QKV buffer).

void check_parts(const torch::Tensor& part) {
  TORCH_CHECK(part.is_cuda() && part.is_contiguous() && part.dim() == 3 &&
                  part.scalar_type() == torch::kFloat32 && part.size(0) >= 1 &&
                  part.size(2) % 4 == 0 &&
                  reinterpret_cast<uintptr_t>(part.data_ptr()) % 16 == 0,
              "parts must be fp32 [splits, rows, columns], columns % 4 == 0");
}

void rmsnorm(torch::Tensor out, torch::Tensor input, torch::Tensor weight,
             double eps) {
  check_bf16_contig(out, "out");
  check_bf16_contig(input, "input");
  check_bf16_contig(weight, "weight");
  const int hidden = input.size(-1);
  TORCH_CHECK(hidden % 8 == 0, "hidden must be a multiple of 8");
  const int rows = input.numel() / hidden;
  arks_rmsnorm(out.data_ptr(), input.data_ptr(), weight.data_ptr(), (float)eps,
               rows, hidden, current_stream());
}

void fused_add_rmsnorm(torch::Tensor out, torch::Tensor input,
                       torch::Tensor residual, torch::Tensor weight,
                       double eps) {
  check_bf16_contig(out, "out");
  check_bf16_contig(input, "input");
  check_bf16_contig(residual, "residual");
  const int hidden = input.size(-1);
  TORCH_CHECK(hidden % 8 == 0, "hidden must be a multiple of 8");
  const int rows = input.numel() / hidden;
  arks_fused_add_rmsnorm(out.data_ptr(), input.data_ptr(), residual.data_ptr(),
                         weight.data_ptr(), (float)eps, rows, hidden,
                         current_stream());
}

// fused_add_rmsnorm of the sum of part's splits
void fused_add_rmsnorm_parts(torch::Tensor out, torch::Tensor part,
                             torch::Tensor residual, torch::Tensor weight,
                             double eps) {
  check_bf16_contig(out, "out");
  check_bf16_contig(residual, "residual");
  check_bf16_contig(weight, "weight");
  check_parts(part);
  const int64_t hidden = part.size(2), rows = part.size(1);
  TORCH_CHECK(hidden % 8 == 0 && out.numel() == rows * hidden &&
              residual.numel() == rows * hidden && weight.numel() == hidden);
  arks_fused_add_rmsnorm_parts(out.data_ptr(), part.data_ptr(),
                               (int)part.size(0), residual.data_ptr(),
                               weight.data_ptr(), (float)eps, (int)rows,
                               (int)hidden, current_stream());
}

// fused_add_rmsnorm of the mix (moe_mix_rows) of the rows y of experts
void fused_add_rmsnorm_mix(torch::Tensor out, torch::Tensor y,
                           torch::Tensor mix_weights, torch::Tensor mix_rows,
                           torch::Tensor residual, torch::Tensor weight,
                           double eps) {
  check_bf16_contig(out, "out");
  check_bf16_contig(y, "y");
  check_bf16_contig(residual, "residual");
  check_bf16_contig(weight, "weight");
  check_rows_16b(y, "y");
  TORCH_CHECK(y.dim() == 2 && mix_weights.dim() == 2 &&
              mix_rows.sizes() == mix_weights.sizes() &&
              mix_weights.is_cuda() && mix_rows.is_cuda() &&
              mix_weights.scalar_type() == torch::kFloat32 &&
              mix_rows.scalar_type() == torch::kInt32 &&
              mix_weights.is_contiguous() && mix_rows.is_contiguous());
  const int64_t hidden = y.size(1), rows = mix_weights.size(0);
  const int64_t k = mix_weights.size(1);
  TORCH_CHECK(hidden % 8 == 0 && out.numel() == rows * hidden &&
              residual.numel() == rows * hidden && weight.numel() == hidden &&
              k >= 1 && k <= 16 && (y.size(0) > 0 || rows == 0));
  if (rows == 0) return;
  arks_fused_add_rmsnorm_mix(out.data_ptr(), y.data_ptr(),
                             mix_weights.data_ptr(), mix_rows.data_ptr(),
                             (int)k, residual.data_ptr(), weight.data_ptr(),
                             (float)eps, (int)rows, (int)hidden,
                             current_stream());
}

void silu_mul(torch::Tensor out, torch::Tensor gate_up) {
  check_bf16_contig(out, "out");
  check_bf16_contig(gate_up, "gate_up");
  const int d = out.size(-1);
  TORCH_CHECK(gate_up.size(-1) == 2 * d, "gate_up last dim must be 2*d");
  TORCH_CHECK(d % 8 == 0, "d must be a multiple of 8");
  const int64_t rows = out.numel() / d;
  arks_silu_mul(out.data_ptr(), gate_up.data_ptr(), rows, d, current_stream());
}

void rope_inplace(torch::Tensor positions, torch::Tensor q, torch::Tensor k,
                  torch::Tensor cos_sin, int64_t head_dim) {
  check_bf16_rowstrided(q, "q");
  check_bf16_rowstrided(k, "k");
  TORCH_CHECK(q.dim() == 2 && k.dim() == 2, "q/k must be 2-D [T, H*D]");
  TORCH_CHECK(positions.scalar_type() == torch::kInt64, "positions must be i64");
  TORCH_CHECK(cos_sin.scalar_type() == torch::kFloat32, "cos_sin must be f32");
  TORCH_CHECK(head_dim % 4 == 0, "head_dim must be a multiple of 4");
  const int num_tokens = q.size(0);
  const int num_q_heads = q.size(-1) / head_dim;
  const int num_kv_heads = k.size(-1) / head_dim;
  arks_rope_inplace(positions.data_ptr(), q.data_ptr(), k.data_ptr(),
                    cos_sin.data_ptr(), num_tokens, (int)head_dim, num_q_heads,
                    num_kv_heads, q.stride(0), k.stride(0), current_stream());
}

void reshape_and_cache(torch::Tensor k, torch::Tensor v, torch::Tensor k_cache,
                       torch::Tensor v_cache, torch::Tensor slot_mapping) {
  check_bf16_rowstrided(k, "k");
  check_bf16_rowstrided(v, "v");
  const bool fp8 = check_kv_cache(k_cache, "k_cache");
  check_kv_cache(v_cache, "v_cache");
  TORCH_CHECK(slot_mapping.scalar_type() == torch::kInt64);
  TORCH_CHECK(k.stride(0) == v.stride(0), "k/v must share row stride");
  const int num_tokens = k.size(0);
  const int num_kv_heads = k_cache.size(1);
  const int block_size = k_cache.size(2);
  const int head_dim = k_cache.size(3);
  TORCH_CHECK(head_dim % 8 == 0);
  auto fn = fp8 ? arks_reshape_and_cache_fp8 : arks_reshape_and_cache;
  fn(k.data_ptr(), v.data_ptr(), k_cache.data_ptr(),
     v_cache.data_ptr(), slot_mapping.data_ptr(),
     num_tokens, num_kv_heads, head_dim, block_size,
     k.stride(0), current_stream());
}

void rope_and_cache(torch::Tensor positions, torch::Tensor q,
                    torch::Tensor k, torch::Tensor v, torch::Tensor k_cache,
                    torch::Tensor v_cache, torch::Tensor slot_mapping,
                    torch::Tensor cos_sin, int64_t head_dim,
                    c10::optional<torch::Tensor> q_norm,
                    c10::optional<torch::Tensor> k_norm, double eps) {
  TORCH_CHECK(positions.scalar_type() == torch::kInt64);
  TORCH_CHECK(slot_mapping.scalar_type() == torch::kInt64);
  TORCH_CHECK(q_norm.has_value() == k_norm.has_value());
  if (q_norm.has_value()) {
    check_bf16_contig(*q_norm, "q_norm");
    check_bf16_contig(*k_norm, "k_norm");
    TORCH_CHECK(q_norm->numel() == head_dim && k_norm->numel() == head_dim);
    TORCH_CHECK(head_dim == 32 || head_dim == 64 || head_dim == 128 ||
                    head_dim == 256,
                "head norms need head_dim 32, 64, 128 or 256");
  }
  TORCH_CHECK(cos_sin.scalar_type() == torch::kFloat32 &&
              cos_sin.is_contiguous());
  check_bf16_rowstrided(q, "q");
  check_bf16_rowstrided(k, "k");
  check_bf16_rowstrided(v, "v");
  const bool kv_fp8 = check_kv_cache(k_cache, "k_cache");
  check_kv_cache(v_cache, "v_cache");
  TORCH_CHECK(k.stride(0) == v.stride(0), "k/v must share row stride");
  const int T = q.size(0);
  const int nq = (int)(q.numel() / std::max<int64_t>(T, 1) / head_dim);
  const int nkv = (int)(k.numel() / std::max<int64_t>(T, 1) / head_dim);
  const int block_size = k_cache.size(2);
  arks_rope_and_cache(positions.data_ptr(), q.data_ptr(), k.data_ptr(),
                      v.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
                      slot_mapping.data_ptr(), cos_sin.data_ptr(), T,
                      (int)head_dim, nq, nkv, block_size, q.stride(0),
                      k.stride(0), kv_fp8 ? 1 : 0,
                      q_norm.has_value() ? q_norm->data_ptr() : nullptr,
                      k_norm.has_value() ? k_norm->data_ptr() : nullptr,
                      (float)eps, current_stream());
}

// rope_and_cache of the projection's split sums part [splits, T, (q heads + 2
// kv heads) * head_dim] (+ bias): rotated q to q, k and v to the cache only
void rope_and_cache_parts(torch::Tensor positions, torch::Tensor q,
                          torch::Tensor part, c10::optional<torch::Tensor> bias,
                          torch::Tensor k_cache, torch::Tensor v_cache,
                          torch::Tensor slot_mapping, torch::Tensor cos_sin,
                          int64_t head_dim, c10::optional<torch::Tensor> q_norm,
                          c10::optional<torch::Tensor> k_norm, double eps) {
  for (const auto& t : {positions, slot_mapping})
    TORCH_CHECK(t.is_cuda() && t.is_contiguous() &&
                    t.scalar_type() == torch::kInt64,
                "positions and slots must be int64 on GPU");
  TORCH_CHECK(cos_sin.is_cuda() && cos_sin.is_contiguous() &&
                  cos_sin.scalar_type() == torch::kFloat32 &&
                  cos_sin.size(-1) == head_dim,
              "cos_sin must be fp32 [positions, head_dim] on GPU");
  check_bf16_contig(q, "q");
  check_parts(part);
  const int64_t T = part.size(1), width = part.size(2);
  const int nkv = k_cache.size(1), block_size = k_cache.size(2);
  TORCH_CHECK(head_dim % 8 == 0 && k_cache.size(3) == head_dim &&
              k_cache.is_cuda() && v_cache.is_cuda() && k_cache.is_contiguous() && v_cache.is_contiguous() &&
              v_cache.sizes() == k_cache.sizes());
  TORCH_CHECK(q.dim() == 2 && q.size(0) == T && q.size(1) % head_dim == 0 &&
              width == q.size(1) + 2 * nkv * head_dim &&
              positions.numel() == T && slot_mapping.numel() == T);
  const bool kv_fp8 = k_cache.scalar_type() != torch::kBFloat16;
  TORCH_CHECK(v_cache.scalar_type() == k_cache.scalar_type() &&
              k_cache.element_size() == (kv_fp8 ? 1 : 2));
  if (bias.has_value()) {
    check_bf16_contig(*bias, "bias");
    TORCH_CHECK(bias->numel() == width);
  }
  TORCH_CHECK(q_norm.has_value() == k_norm.has_value());
  if (q_norm.has_value()) {
    check_bf16_contig(*q_norm, "q_norm");
    check_bf16_contig(*k_norm, "k_norm");
    TORCH_CHECK(q_norm->numel() == head_dim && k_norm->numel() == head_dim);
    TORCH_CHECK(head_dim == 32 || head_dim == 64 || head_dim == 128 ||
                    head_dim == 256,
                "head norms need head_dim 32, 64, 128 or 256");
  }
  arks_rope_and_cache_parts(
      positions.data_ptr(), q.data_ptr(), part.data_ptr(),
      bias.has_value() ? bias->data_ptr() : nullptr, (int)part.size(0),
      k_cache.data_ptr(), v_cache.data_ptr(), slot_mapping.data_ptr(),
      cos_sin.data_ptr(), (int)T, (int)head_dim, (int)(q.size(1) / head_dim),
      nkv, block_size, kv_fp8 ? 1 : 0,
      q_norm.has_value() ? q_norm->data_ptr() : nullptr,
      k_norm.has_value() ? k_norm->data_ptr() : nullptr, (float)eps,
      current_stream());
}


void attention_prefill_varlen(torch::Tensor out, torch::Tensor q,
                              torch::Tensor k, torch::Tensor v,
                              torch::Tensor cu_seqlens, torch::Tensor tile_info,
                              double scale, int64_t window) {
  check_bf16_contig(out, "out");
  check_bf16_rowstrided(q, "q");
  check_bf16_rowstrided(k, "k");
  check_bf16_rowstrided(v, "v");
  TORCH_CHECK(k.stride(0) == v.stride(0), "k/v must share row stride");
  TORCH_CHECK(cu_seqlens.scalar_type() == torch::kInt32);
  TORCH_CHECK(tile_info.scalar_type() == torch::kInt32);
  TORCH_CHECK(tile_info.dim() == 2 && tile_info.size(1) == 2);
  const int num_q_heads = q.size(1);
  const int head_dim = q.size(2);
  const int num_kv_heads = k.size(1);
  TORCH_CHECK(head_dim == 64 || head_dim == 128, "head_dim must be 64 or 128");
  const int ntiles = tile_info.size(0);
  arks_attn_prefill_varlen(out.data_ptr(), q.data_ptr(), k.data_ptr(),
                           v.data_ptr(), cu_seqlens.data_ptr(),
                           tile_info.data_ptr(), ntiles, (float)scale,
                           num_q_heads, num_kv_heads, head_dim, q.stride(0),
                           k.stride(0), (int)window, current_stream());
}


// 8-wave 32x32-MFMA ladder (attn_extend2.hip): 256-row q tiles, bf16 KV.


void rmsnorm_fp8(torch::Tensor out, torch::Tensor inv_scale,
                 torch::Tensor input, c10::optional<torch::Tensor> residual,
                 torch::Tensor weight, double eps) {
  check_bf16_contig(input, "input");
  check_bf16_contig(weight, "weight");
  TORCH_CHECK(out.scalar_type() == torch::kFloat8_e4m3fn && out.is_contiguous());
  TORCH_CHECK(inv_scale.scalar_type() == torch::kFloat32);
  const int hidden = input.size(-1);
  TORCH_CHECK(hidden % 8 == 0 && hidden <= 8192,
              "rmsnorm_fp8 requires hidden % 8 == 0 and hidden <= 8192");
  const int rows = input.numel() / hidden;
  void* res_ptr = nullptr;
  if (residual.has_value()) {
    check_bf16_contig(*residual, "residual");
    res_ptr = residual->data_ptr();
  }
  arks_rmsnorm_fp8(out.data_ptr(), inv_scale.data_ptr(), input.data_ptr(),
                   res_ptr, weight.data_ptr(), (float)eps, rows, hidden,
                   residual.has_value() ? 1 : 0, current_stream());
}

void silu_mul_fp8(torch::Tensor out, torch::Tensor inv_scale,
                  torch::Tensor gate_up) {
  check_bf16_contig(gate_up, "gate_up");
  TORCH_CHECK(out.scalar_type() == torch::kFloat8_e4m3fn && out.is_contiguous());
  TORCH_CHECK(inv_scale.scalar_type() == torch::kFloat32);
  const int d = out.size(-1);
  TORCH_CHECK(gate_up.size(-1) == 2 * d && d % 8 == 0);
  TORCH_CHECK((int64_t)d * 2 <= 160 * 1024, "row too large for LDS staging");
  const int rows = out.numel() / d;
  arks_silu_mul_fp8(out.data_ptr(), inv_scale.data_ptr(), gate_up.data_ptr(),
                    rows, d, current_stream());
}

void quant_fp8_rows(torch::Tensor out, torch::Tensor inv_scale,
                    torch::Tensor x) {
  check_bf16_contig(x, "x");
  TORCH_CHECK(out.scalar_type() == torch::kFloat8_e4m3fn && out.is_contiguous());
  TORCH_CHECK(inv_scale.scalar_type() == torch::kFloat32);
  TORCH_CHECK(x.size(1) % 8 == 0, "cols must be a multiple of 8");
  arks_quant_fp8_rows(out.data_ptr(), inv_scale.data_ptr(), x.data_ptr(),
                      x.size(0), x.size(1), current_stream());
}

// Workgroups per row: ~1024 in all (4 per CU), each with at least 2048 values.
void sample_rows(torch::Tensor out, torch::Tensor logits, const void* temps,
                 const void* uniform) {
  const int64_t rows = logits.size(0), vocab = logits.size(1);
  const int64_t parts = std::max<int64_t>(
      1, std::min<int64_t>({64, vocab / 2048,
                            1024 / std::max<int64_t>(rows, 1)}));
  torch::Tensor val, idx;
  if (parts > 1) {
    val = torch::empty({rows * parts}, logits.options().dtype(torch::kFloat32));
    idx = torch::empty({rows * parts}, logits.options().dtype(torch::kInt32));
  }
  if (rows > 0)
    arks_sample(out.data_ptr(), parts > 1 ? val.data_ptr() : nullptr,
                parts > 1 ? idx.data_ptr() : nullptr, logits.data_ptr(), temps,
                uniform, (int)rows, (int)vocab, (int)parts, current_stream());
}

void greedy_sample(torch::Tensor out, torch::Tensor logits) {
  check_bf16_contig(logits, "logits");
  TORCH_CHECK(out.scalar_type() == torch::kInt64);
  sample_rows(out, logits, nullptr, nullptr);
}

void gumbel_sample(torch::Tensor out, torch::Tensor logits,
                   torch::Tensor temperatures, torch::Tensor uniform) {
  check_bf16_contig(logits, "logits");
  TORCH_CHECK(out.scalar_type() == torch::kInt64);
  TORCH_CHECK(temperatures.scalar_type() == torch::kFloat32);
  TORCH_CHECK(uniform.scalar_type() == torch::kFloat32);
  sample_rows(out, logits, temperatures.data_ptr(), uniform.data_ptr());
}

// D[16,16] = A[16,32] @ B[32,16], all bf16 in / f32 out. Verifies the MFMA
// fragment layout assumption on hardware.
void tr16_probe(torch::Tensor out, int64_t stride_bytes) {
  TORCH_CHECK(out.scalar_type() == torch::kInt16 && out.numel() >= 256);
  arks_tr16_probe(out.data_ptr(), (int)stride_bytes, current_stream());
}

void mfma_probe32(torch::Tensor d, torch::Tensor a, torch::Tensor b) {
  check_bf16_contig(a, "a");
  check_bf16_contig(b, "b");
  TORCH_CHECK(d.scalar_type() == torch::kFloat32 && d.is_contiguous());
  TORCH_CHECK(a.size(0) == 32 && a.size(1) == 16);
  TORCH_CHECK(b.size(0) == 16 && b.size(1) == 32);
  arks_mfma_probe32(d.data_ptr(), a.data_ptr(), b.data_ptr(), current_stream());
}

// --- p2p one-shot all-reduce plumbing (allreduce.hip) ---
// IPC-shared buffers are raw hipMalloc allocations: a handle for a torch
// caching-allocator tensor maps the UNDERLYING block, so the opened peer
// pointer would miss the tensor's offset inside it.
py::tuple ipc_alloc(int64_t nbytes) {
  void* ptr = nullptr;
  auto err = hipMalloc(&ptr, (size_t)nbytes);
  TORCH_CHECK(err == hipSuccess, "hipMalloc: ", hipGetErrorString(err));
  (void)hipMemset(ptr, 0, (size_t)nbytes);
  hipIpcMemHandle_t h;
  err = hipIpcGetMemHandle(&h, ptr);
  TORCH_CHECK(err == hipSuccess, "hipIpcGetMemHandle: ",
              hipGetErrorString(err));
  return py::make_tuple(
      reinterpret_cast<int64_t>(ptr),
      py::bytes(reinterpret_cast<const char*>(&h), sizeof(h)));
}

void ipc_alloc_free(int64_t ptr) {
  (void)hipFree(reinterpret_cast<void*>(ptr));
}

// test hook: arm a raw flag buffer with huge values (0x7f per byte) so the
// single-GPU sequential harness never spins
void arm_flags(int64_t ptr, int64_t n) {
  (void)hipMemset(reinterpret_cast<void*>(ptr), 0x7f, (size_t)n * 8);
}

py::bytes ipc_handle(torch::Tensor t) {
  TORCH_CHECK(t.is_cuda(), "ipc_handle wants a CUDA tensor");
  hipIpcMemHandle_t h;
  auto err = hipIpcGetMemHandle(&h, t.data_ptr());
  TORCH_CHECK(err == hipSuccess, "hipIpcGetMemHandle: ",
              hipGetErrorString(err));
  return py::bytes(reinterpret_cast<const char*>(&h), sizeof(h));
}

int64_t ipc_open(py::bytes handle) {
  std::string s = handle;
  TORCH_CHECK(s.size() == sizeof(hipIpcMemHandle_t), "bad handle size");
  hipIpcMemHandle_t h;
  memcpy(&h, s.data(), sizeof(h));
  void* ptr = nullptr;
  auto err = hipIpcOpenMemHandle(&ptr, h, hipIpcMemLazyEnablePeerAccess);
  TORCH_CHECK(err == hipSuccess, "hipIpcOpenMemHandle: ",
              hipGetErrorString(err));
  return reinterpret_cast<int64_t>(ptr);
}

void ipc_close(int64_t ptr) {
  (void)hipIpcCloseMemHandle(reinterpret_cast<void*>(ptr));
}

void one_shot_allreduce(torch::Tensor out, torch::Tensor src,
                        std::vector<int64_t> mail,
                        std::vector<int64_t> flags, torch::Tensor seq,
                        int64_t rank) {  // mail/flags: ipc_alloc'd raw ptrs
  check_bf16_contig(out, "out");
  check_bf16_contig(src, "src");
  TORCH_CHECK(seq.is_cuda() && seq.scalar_type() == torch::kInt64);
  const int world = (int)mail.size();
  TORCH_CHECK(world == (int)flags.size());
  TORCH_CHECK(world == 1 || world == 2 || world == 4 || world == 8,
              "world must be 1/2/4/8");
  const int64_t n = src.numel();
  TORCH_CHECK(n % 8 == 0, "numel must be a multiple of 8");
  TORCH_CHECK(out.numel() == n);
  void* mp[8] = {};
  void* fp[8] = {};
  for (int p = 0; p < world; ++p) {
    mp[p] = reinterpret_cast<void*>(mail[p]);
    fp[p] = reinterpret_cast<void*>(flags[p]);
  }
  auto stream = current_stream();
  arks_ar_seq_inc(seq.data_ptr(), stream);
  arks_one_shot_allreduce(out.data_ptr(), src.data_ptr(), mp, fp,
                          seq.data_ptr(), (int)rank, world, n, stream);
}

void moe_topk(torch::Tensor weights, torch::Tensor ids,
              torch::Tensor logits, int64_t k, int64_t renorm) {
  TORCH_CHECK(logits.is_cuda() && logits.is_contiguous() &&
              logits.scalar_type() == torch::kFloat32, "logits f32 contig");
  TORCH_CHECK(weights.scalar_type() == torch::kFloat32 &&
              ids.scalar_type() == torch::kInt32);
  const int T = logits.size(0), E = logits.size(1);
  TORCH_CHECK(k >= 1 && k <= 16 && E <= 1024 && k <= E,
              "need 1 <= k <= min(16, E), E <= 1024");
  arks_moe_topk(weights.data_ptr(), ids.data_ptr(), logits.data_ptr(), T, E,
                (int)k, (int)renorm, current_stream());
}

void moe_mix_rows(torch::Tensor out, torch::Tensor y,
                  torch::Tensor weights, torch::Tensor rows) {
  check_bf16_contig(out, "out");
  check_bf16_contig(y, "y");
  TORCH_CHECK(weights.scalar_type() == torch::kFloat32 &&
              rows.scalar_type() == torch::kInt32);
  const int T = out.size(0), H = out.size(1);
  const int k = weights.size(1);
  TORCH_CHECK(k <= 16 && H % 2 == 0);
  TORCH_CHECK(rows.size(0) == T && rows.size(1) == k);
  arks_moe_mix_rows(out.data_ptr(), y.data_ptr(), weights.data_ptr(),
                    rows.data_ptr(), T, H, k, current_stream());
}

// out [M, N] (bf16 or fp32) = a [M, K] w [N, K]^T (+ bias [N]); silu: w is
// [2N, K] and out silu of the first N columns times the others
void stream_gemm(torch::Tensor out, torch::Tensor a, torch::Tensor w,
                 c10::optional<torch::Tensor> bias, int64_t mt, int64_t nf,
                 int64_t wv, bool silu) {
  check_bf16_rowstrided(a, "a");
  check_bf16_contig(w, "w");
  TORCH_CHECK(a.dim() == 2 && w.dim() == 2 && out.is_cuda() &&
              out.is_contiguous());
  check_rows_16b(a, "a");
  check_rows_16b(w, "w");
  const bool f32 = out.scalar_type() == torch::kFloat32;
  TORCH_CHECK((f32 && !silu) || out.scalar_type() == torch::kBFloat16);
  TORCH_CHECK(reinterpret_cast<uintptr_t>(out.data_ptr()) % 16 == 0);
  const int64_t M = a.size(0), K = a.size(1);
  const int64_t N = silu ? w.size(0) / 2 : w.size(0);
  TORCH_CHECK(w.size(1) == K && w.size(0) == (silu ? 2 * N : N) &&
              out.dim() == 2 && out.size(0) == M && out.size(1) == N);
  TORCH_CHECK(K % 32 == 0 && M <= 16 * 65535 && N < (1 << 30),
              "need K % 32 == 0");
  TORCH_CHECK(mt == 1 || mt == 2);
  TORCH_CHECK(silu ? nf == 2 && (wv == 8 || wv == 16)
                   : (nf == 1 && (wv == 4 || wv == 16)) ||
                         (nf == 2 && (wv == 8 || wv == 16)));
  if (bias.has_value()) {
    check_bf16_contig(*bias, "bias");
    TORCH_CHECK(bias->numel() == N && !silu);
  }
  if (M == 0 || N == 0) return;
  arks_stream_gemm(out.data_ptr(), a.data_ptr(), w.data_ptr(),
                   bias.has_value() ? bias->data_ptr() : nullptr, (int)M,
                   (int)N, (int)K, a.stride(0), (int)mt, (int)nf, (int)wv,
                   f32 ? 1 : 0, silu ? 1 : 0, current_stream());
}

// part [splits, M, N] fp32: the sums of a [M, K] w [N, K]^T over runs of K,
// even ones (per 0) or of per columns, the last of what is left
void stream_split(torch::Tensor part, torch::Tensor a, torch::Tensor w,
                  int64_t per) {
  check_bf16_rowstrided(a, "a");
  check_bf16_contig(w, "w");
  TORCH_CHECK(a.dim() == 2 && w.dim() == 2 && part.dim() == 3);
  check_rows_16b(a, "a");
  check_rows_16b(w, "w");
  check_parts(part);
  const int64_t M = a.size(0), N = w.size(0), K = a.size(1);
  const int64_t splits = part.size(0);
  TORCH_CHECK(w.size(1) == K && part.size(1) == M && part.size(2) == N);
  TORCH_CHECK(M >= 1 && M <= 64 && N < (1 << 30) && K < (1 << 30),
              "need at most 64 rows");
  TORCH_CHECK(per == 0 ? K % 64 == 0 && splits <= K / 64
                       : per > 0 && per % 32 == 0 && K % 32 == 0 &&
                             (splits - 1) * per < K && K <= splits * per,
              "splits do not fit the columns");
  arks_stream_split(part.data_ptr(), a.data_ptr(), w.data_ptr(), (int)M, (int)N,
                    (int)K, a.stride(0), (int)splits, (int)per,
                    current_stream());
}

void stream_sum(torch::Tensor out, torch::Tensor part,
                c10::optional<torch::Tensor> bias) {
  check_bf16_contig(out, "out");
  check_parts(part);
  const int64_t M = part.size(1), N = part.size(2);
  TORCH_CHECK(out.dim() == 2 && out.size(0) == M && out.size(1) == N);
  if (bias.has_value()) {
    check_bf16_contig(*bias, "bias");
    TORCH_CHECK(bias->numel() == N);
  }
  arks_stream_sum(out.data_ptr(), part.data_ptr(),
                  bias.has_value() ? bias->data_ptr() : nullptr, M, (int)N,
                  (int)part.size(0), current_stream());
}

// out [M, N] = silu(a w_gate^T) * (a w_up^T), w [2N, K] (tile_gemm.hip)
void tile_silu(torch::Tensor out, torch::Tensor a, torch::Tensor w) {
  check_bf16_contig(out, "out");
  check_bf16_rowstrided(a, "a");
  check_bf16_contig(w, "w");
  TORCH_CHECK(out.dim() == 2 && a.dim() == 2 && w.dim() == 2);
  check_rows_16b(out, "out");
  check_rows_16b(a, "a");
  check_rows_16b(w, "w");
  const int64_t M = a.size(0), K = a.size(1), N = w.size(0) / 2;
  TORCH_CHECK(w.size(1) == K && w.size(0) == 2 * N && out.size(0) == M &&
              out.size(1) == N);
  TORCH_CHECK(K >= 64 && K % 64 == 0 && N % 8 == 0 && M < (1 << 30) &&
                  N < (1 << 29) && K < (1 << 22) &&
                  a.stride(0) < (1 << 22),
              "need K % 64 == 0, N % 8 == 0");
  if (M == 0 || N == 0) return;
  arks_tile_silu(out.data_ptr(), a.data_ptr(), w.data_ptr(), (int)M, (int)N,
                 (int)K, a.stride(0), current_stream());
}

// out [M, N] = a w^T (+ bias), bf16, or fp32 [splits, M, N] its sums over runs of
// K; silu: silu(gate) * up of w [2N, K]; tiles of tm rows of a x tw of w
// (wide_gemm.hip)
void wide_gemm(torch::Tensor out, torch::Tensor a, torch::Tensor w,
               c10::optional<torch::Tensor> bias, int64_t tm, int64_t tw,
               bool silu) {
  const bool parts = out.dim() == 3;
  check_bf16_rowstrided(a, "a");
  check_bf16_contig(w, "w");
  if (parts) check_parts(out);
  else check_bf16_contig(out, "out");
  TORCH_CHECK((parts || out.dim() == 2) && a.dim() == 2 && w.dim() == 2);
  check_rows_16b(out, "out");
  check_rows_16b(a, "a");
  check_rows_16b(w, "w");
  const int64_t M = a.size(0), K = a.size(1), splits = parts ? out.size(0) : 1;
  const int64_t N = silu ? w.size(0) / 2 : w.size(0);
  TORCH_CHECK(w.size(1) == K && w.size(0) == (silu ? 2 * N : N) &&
              out.size(out.dim() - 2) == M && out.size(out.dim() - 1) == N);
  TORCH_CHECK(K >= 64 && K % 64 == 0 && N % 8 == 0 && M < (1 << 24) &&
                  N < (1 << 24) && K < (1 << 22) && a.stride(0) < (1 << 22) &&
                  (!silu || (N + 320) * K < ((int64_t)1 << 31)),
              "need K % 64 == 0, N % 8 == 0");
  TORCH_CHECK(splits >= 1 && splits <= K / 64 && splits <= 64 && !(parts && silu));
  if (bias.has_value()) {
    check_bf16_contig(*bias, "bias");
    TORCH_CHECK(bias->numel() == N && !silu && !parts);
  }
  if (M == 0 || N == 0) return;
  TORCH_CHECK(arks_wide_gemm(out.data_ptr(), a.data_ptr(), w.data_ptr(),
                             bias.has_value() ? bias->data_ptr() : nullptr,
                             (int)M, (int)N, (int)K, a.stride(0), (int)tm,
                             (int)tw, (int)splits, parts ? 1 : silu ? 2 : 0,
                             current_stream()),
              "no tile of this size");
}

// out [M, N] = a w^T (+ bias), bf16, or fp32 [splits, M, N] its sums over runs
// of K; silu: silu(gate) * up of w [2N, K] (mid_gemm.hip)
void mid_gemm(torch::Tensor out, torch::Tensor a, torch::Tensor w,
              c10::optional<torch::Tensor> bias, int64_t qt, bool silu) {
  const bool parts = out.dim() == 3;
  check_bf16_rowstrided(a, "a");
  check_bf16_contig(w, "w");
  if (parts) {
    TORCH_CHECK(out.is_cuda() && out.scalar_type() == torch::kFloat32 &&
                    out.is_contiguous() && !silu && !bias.has_value(),
                "sums are contiguous fp32 on the GPU, without a bias");
  } else {
    check_bf16_contig(out, "out");
  }
  TORCH_CHECK((parts || out.dim() == 2) && a.dim() == 2 && w.dim() == 2);
  TORCH_CHECK(reinterpret_cast<uintptr_t>(out.data_ptr()) % 16 == 0);
  check_rows_16b(a, "a");
  check_rows_16b(w, "w");
  const int64_t M = a.size(0), K = a.size(1);
  const int64_t N = silu ? w.size(0) / 2 : w.size(0);
  const int64_t splits = parts ? out.size(0) : 1;
  TORCH_CHECK(w.size(1) == K && w.size(0) == (silu ? 2 * N : N) &&
              out.size(parts ? 1 : 0) == M && out.size(parts ? 2 : 1) == N);
  TORCH_CHECK(qt == 2 || qt == 4 || qt == 5);
  TORCH_CHECK(M <= 256 && K % 64 == 0 && N % 8 == 0 && splits >= 1 &&
                  splits <= K / 64 && K < (1 << 22) && N < (1 << 24) &&
                  a.stride(0) < (1 << 22) &&
                  (!silu || 2 * N * K < (1ll << 31)),
              "need M <= 256, K % 64 == 0, N % 8 == 0");
  if (bias.has_value()) {
    check_bf16_contig(*bias, "bias");
    TORCH_CHECK(bias->numel() == N);
  }
  if (M == 0 || N == 0) return;
  arks_mid_gemm(out.data_ptr(), a.data_ptr(), w.data_ptr(),
                bias.has_value() ? bias->data_ptr() : nullptr, (int)M, (int)N,
                (int)K, a.stride(0), (int)qt, (int)splits, parts, silu,
                current_stream());
}

// out [splits + splits2, M, N]: the sums of a . w^T in `splits` runs of K, then
// those of a2 . w2^T (mid_gemm.hip)
void mid_pair(torch::Tensor out, torch::Tensor a, torch::Tensor w,
              torch::Tensor a2, torch::Tensor w2, int64_t qt, int64_t splits) {
  TORCH_CHECK(out.is_cuda() && out.dim() == 3 && out.is_contiguous() &&
                  out.scalar_type() == torch::kFloat32 &&
                  reinterpret_cast<uintptr_t>(out.data_ptr()) % 16 == 0,
              "sums are contiguous fp32 on the GPU");
  const int64_t M = out.size(1), N = out.size(2), splits2 = out.size(0) - splits;
  TORCH_CHECK(M <= 64 && N % 8 == 0 && N < (1 << 24) && splits >= 1 &&
                  splits2 >= 1 && (qt == 2 || qt == 4 || qt == 5),
              "need M <= 64, N % 8 == 0");
  auto check = [&](const torch::Tensor& x, const torch::Tensor& weight,
                   int64_t runs) {
    check_bf16_rowstrided(x, "a");
    check_bf16_contig(weight, "w");
    TORCH_CHECK(x.dim() == 2 && weight.dim() == 2);
    check_rows_16b(x, "a");
    check_rows_16b(weight, "w");
    const int64_t K = x.size(1);
    TORCH_CHECK(x.size(0) == M && weight.size(0) == N && weight.size(1) == K &&
                    x.device() == out.device() && weight.device() == out.device() &&
                    K % 64 == 0 && runs <= K / 64 && K < (1 << 22) &&
                    x.stride(0) < (1 << 22),
                "need rows of K % 64 == 0 columns, a run of 64 at least");
  };
  check(a, w, splits);
  check(a2, w2, splits2);
  if (M == 0 || N == 0) return;
  arks_mid_pair(out.data_ptr(), a.data_ptr(), w.data_ptr(), (int)a.size(1),
                a.stride(0), (int)splits, a2.data_ptr(), w2.data_ptr(),
                (int)a2.size(1), a2.stride(0), (int)splits2, (int)M, (int)N,
                (int)qt, current_stream());
}

// What a step's rows read, into host tensors: sequence i's tokens (prompt, then
// output) from starts[i] on, counts[i] of them (none given: its last one), their
// positions and cache slots, packed; its length behind them into lens[i], its
// page numbers into row i of block_tables (what stands behind them stays). Lists
// are walked here because a step waits for it: 200 requests with 8700 pages take
// 400 us in Python, 30 here. rows (one token each): those behind the sequences' are
// padding up to there, without a cache slot, of length 1.
void stage_rows(pybind11::list prompts, pybind11::list outputs,
                pybind11::list tables, pybind11::object starts,
                pybind11::object counts, torch::Tensor ids, torch::Tensor pos,
                torch::Tensor slots, torch::Tensor lens,
                torch::Tensor block_tables, int64_t block_size, int64_t rows) {
  const Py_ssize_t n = PyList_GET_SIZE(prompts.ptr());
  auto host = [](const torch::Tensor& t, torch::ScalarType type, int64_t least) {
    TORCH_CHECK(!t.is_cuda() && t.scalar_type() == type && t.is_contiguous() &&
                    t.numel() >= least,
                "stage_rows: a host tensor is missing or too small");
  };
  const bool last = starts.is_none();
  TORCH_CHECK(counts.is_none() == last && block_size > 0);
  pybind11::list from, many;
  if (!last) from = starts, many = counts;
  TORCH_CHECK(PyList_GET_SIZE(outputs.ptr()) == n &&
              PyList_GET_SIZE(tables.ptr()) == n &&
              (last || (PyList_GET_SIZE(from.ptr()) == n &&
                        PyList_GET_SIZE(many.ptr()) == n)));
  TORCH_CHECK(rows <= n || last, "stage_rows: padding is of rows of one token");
  const int64_t most = std::max<int64_t>(n, rows);
  host(lens, torch::kInt32, most);
  host(block_tables, torch::kInt32, 0);
  TORCH_CHECK(block_tables.dim() == 2 && block_tables.size(0) >= most &&
              (rows <= n || block_tables.size(1) >= 1));
  host(ids, torch::kInt64, last ? most : 0);
  host(pos, torch::kInt64, last ? most : 0);
  host(slots, torch::kInt64, last ? most : 0);
  const int64_t room =
      std::min({ids.numel(), pos.numel(), slots.numel()});
  const int64_t width = block_tables.size(1);
  auto* to_ids = ids.data_ptr<int64_t>();
  auto* to_pos = pos.data_ptr<int64_t>();
  auto* to_slots = slots.data_ptr<int64_t>();
  auto* to_lens = lens.data_ptr<int32_t>();
  auto* to_table = block_tables.data_ptr<int32_t>();
  auto whole = [](PyObject* o) {
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw pybind11::error_already_set();
    return (int64_t)v;
  };
  auto list_of = [](PyObject* o) {
    TORCH_CHECK(PyList_Check(o), "stage_rows: lists of lists");
    return o;
  };
  int64_t at = 0;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* p = list_of(PyList_GET_ITEM(prompts.ptr(), i));
    PyObject* o = list_of(PyList_GET_ITEM(outputs.ptr(), i));
    PyObject* t = list_of(PyList_GET_ITEM(tables.ptr(), i));
    const int64_t np = PyList_GET_SIZE(p), all = np + PyList_GET_SIZE(o);
    const int64_t pages = PyList_GET_SIZE(t);
    const int64_t s = last ? all - 1 : whole(PyList_GET_ITEM(from.ptr(), i));
    const int64_t c = last ? 1 : whole(PyList_GET_ITEM(many.ptr(), i));
    TORCH_CHECK(s >= 0 && c >= 0 && s + c <= all && at + c <= room &&
                    pages <= width && s + c <= pages * block_size,
                "stage_rows: tokens, pages or room missing");
    int32_t* row = to_table + i * width;
    for (int64_t j = 0; j < pages; ++j)
      row[j] = (int32_t)whole(PyList_GET_ITEM(t, j));
    for (int64_t j = s; j < s + c; ++j, ++at) {
      to_ids[at] = whole(j < np ? PyList_GET_ITEM(p, j)
                                : PyList_GET_ITEM(o, j - np));
      to_pos[at] = j;
      to_slots[at] = (int64_t)row[j / block_size] * block_size + j % block_size;
    }
    to_lens[i] = (int32_t)(s + c);
  }
  for (int64_t i = n; i < rows; ++i) {
    to_ids[i] = to_pos[i] = 0;
    to_slots[i] = -1;
    to_lens[i] = 1;
    to_table[i * width] = 0;
  }
}

// Tiles of weight rows and steps of 64 columns of an expert's products in
// moe_gemm.hip's engine: gate and up of 2I x H, then H x I.
static std::array<int, 4> engine_rounds(int64_t H, int64_t I) {
  return {(int)((I + 127) / 128), (int)((H + 255) / 256), (int)(H / 64),
          (int)(I / 64)};
}

// The experts' rows of x [T, H] and their mix: (y [T * k, H], weights and rows
// [T, k]); w13 [El, 2I, H], w2 [El, H, I], pairs beyond this rank's El experts
// from expert_base on weigh zero. tile: pairs of a work item; mid: of 32, 64 or
// 128 pairs in mid_gemm.hip (32: qt_up and qt_down, weight rows a wave / 16, may
// be 2), else in moe_gemm.hip (16, 128 or, 256, its engine's up to 320). logits
// [T, experts]: the plan finds ids and weights (only their sizes count then).
// experts: the number on all ranks (at least El).
std::tuple<torch::Tensor, torch::Tensor, torch::Tensor> moe_expert_rows(
    torch::Tensor x, torch::Tensor w13, torch::Tensor w2, torch::Tensor weights,
    torch::Tensor ids, int64_t expert_base, int64_t tile, bool mid,
    int64_t qt_up, int64_t qt_down,
    c10::optional<torch::Tensor> logits = c10::nullopt, bool renorm = false,
    int64_t experts = 0) {
  check_bf16_rowstrided(x, "x");
  check_bf16_contig(w13, "w13");
  check_bf16_contig(w2, "w2");
  check_rows_16b(x, "x");
  check_rows_16b(w13, "w13");
  check_rows_16b(w2, "w2");
  const int64_t T = x.size(0), H = x.size(1), El = w13.size(0);
  const int64_t I = w2.size(2), k = weights.size(1), P = T * k;
  TORCH_CHECK(x.dim() == 2);
  TORCH_CHECK(w13.size(1) == 2 * I && w13.size(2) == H && w2.size(0) == El &&
                  w2.size(1) == H,
              "expert weights do not fit");
  for (const int64_t qt : {qt_up, qt_down})
    TORCH_CHECK(qt == 4 || (qt == 2 && tile == 32 && mid), "4, or 2 in items of 32");
  TORCH_CHECK(mid ? tile == 32 || tile == 64 || tile == 128
                  : tile == 16 || tile == 128 || tile == 256);
  TORCH_CHECK((H | I) % (mid ? 64 : tile == 16 ? 32 : tile == 128 ? 8 : 64) == 0 &&
                  El <= 1024 && k <= 16,
              "need H and I % 8 == 0 (tile 16: % 32, 256 and mid: % 64), at "
              "most 1024 experts, k <= 16");
  // row offsets are 32 bits wide, the engine's items of one expert 15
  TORCH_CHECK(!(mid || tile == 256) ||
                  (T * x.stride(0) < (1ll << 31) && 2 * I * H < (1ll << 31) &&
                   P < (1 << 23) - 255),
              "too large for this tile");
  TORCH_CHECK(weights.is_cuda() && ids.is_cuda() &&
              weights.scalar_type() == torch::kFloat32 &&
              weights.is_contiguous() && ids.scalar_type() == torch::kInt32 &&
              ids.is_contiguous() && ids.size(0) == T && ids.size(1) == k &&
              weights.size(0) == T);
  if (logits.has_value())
    TORCH_CHECK(logits->is_cuda() && logits->is_contiguous() &&
                    logits->scalar_type() == torch::kFloat32 &&
                    logits->dim() == 2 && logits->size(0) == T &&
                    logits->size(1) <= 128 && logits->size(1) >= k && k >= 1 &&
                    P <= 512,
                "the plan takes fp32 logits of 128 experts, 512 pairs");
  if (T == 0) return {torch::empty({0, H}, x.options()), weights, ids};
  const int64_t max_items = std::min(P, El) + P / (tile == 256 ? 192 : tile);
  TORCH_CHECK(max_items <= 65535 || tile != 16, "too many rows for this tile");
  auto ints = x.options().dtype(torch::kInt32);
  // one workgroup plans 8192 pairs in 9 us and 16384 in 20; two launches of a
  // workgroup per 2048 pairs take 8 and 10 (128 experts)
  const int64_t groups = P <= 8192 ? 1 : std::min<int64_t>(64, (P + 2047) / 2048);
  // [items | perm | rows | count | claims | counts of the groups], the items
  // on 16-byte places
  torch::Tensor plan = torch::empty(
      {4 * max_items + 2 * P + 17 + (groups > 1 ? groups * El : 0)}, ints);
  int* items = plan.data_ptr<int>();
  int* perm = items + 4 * max_items;
  int* rows = perm + P;
  int* n_items = rows + P;
  torch::Tensor w_pair = torch::empty_like(weights);
  torch::Tensor h = torch::empty({P, I}, x.options());
  torch::Tensor y = torch::empty({P, H}, x.options());
  auto stream = current_stream();
  int* claims = n_items + 1;
  const int places = tile == 256 ? 320 : (int)tile;
  const auto rounds = engine_rounds(H, I);
  if (logits.has_value())
    arks_moe_plan_topk(perm, rows, w_pair.data_ptr(), items, n_items, claims,
                       logits->data_ptr(), (int)logits->size(1), (int)k, renorm,
                       (int)P, (int)expert_base, (int)El, places, (int)max_items,
                       rounds.data(), stream);
  else
    arks_moe_plan(perm, rows, w_pair.data_ptr(), items, n_items, claims,
                  claims + 16, ids.data_ptr(), weights.data_ptr(), (int)P,
                  (int)expert_base, (int)El, places, (int)max_items, (int)groups,
                  rounds.data(), stream);
  if (mid) {
    const int ft = (int)tile / 32;
    arks_mid_items(h.data_ptr(), x.data_ptr(), w13.data_ptr(), perm, items,
                   n_items, x.stride(0), 2 * I * H, (int)I, (int)H, (int)k,
                   (int)expert_base, (int)max_items, ft, (int)qt_up, 1, stream);
    arks_mid_items(y.data_ptr(), h.data_ptr(), w2.data_ptr(), nullptr, items,
                   n_items, I, H * I, (int)H, (int)I, (int)k,
                   (int)expert_base, (int)max_items, ft, (int)qt_down, 0, stream);
  } else {
    // (moe_gemm.hip: experts that mostly have one item)
    const int once = P <= 160 * std::max(experts, El) ? 2 : 0;
    arks_moe_gemm(h.data_ptr(), x.data_ptr(), w13.data_ptr(), perm, items,
                  n_items, claims, nullptr, x.stride(0), 2 * I * H, H, (int)I, (int)H,
                  (int)k, (int)max_items, (int)tile, 1, once, (int)expert_base,
                  stream);
    arks_moe_gemm(y.data_ptr(), h.data_ptr(), w2.data_ptr(), perm, items,
                  n_items, claims, nullptr, I, H * I, I, (int)H, (int)I, (int)k,
                  (int)max_items, (int)tile, 0, once, (int)expert_base, stream);
  }
  return {y, w_pair, plan.narrow(0, 4 * max_items + P, P).view({T, k})};
}

// The experts' rows of x [T, W] in whole tiles: (y [T * k, W], rows [T, k]).
// w_gu: from its first row on each expert's ff gate rows, then its up rows;
// w_down [W, ..]: from its first column on ff columns an expert. All pairs are
// of these experts; scaled: a pair's weight is a factor of its gate and up.
std::tuple<torch::Tensor, torch::Tensor> moe_wide_rows(
    torch::Tensor x, torch::Tensor w_gu, torch::Tensor w_down,
    torch::Tensor weights, torch::Tensor ids, int64_t experts, int64_t ff,
    bool scaled) {
  check_bf16_rowstrided(x, "x");
  check_bf16_contig(w_gu, "w_gu");
  check_bf16_contig(w_down, "w_down");
  check_rows_16b(x, "x");
  check_rows_16b(w_gu, "w_gu");
  check_rows_16b(w_down, "w_down");
  TORCH_CHECK(x.dim() == 2 && w_gu.dim() == 2 && w_down.dim() == 2 &&
              weights.dim() == 2);
  const int64_t T = x.size(0), W = x.size(1), k = weights.size(1), P = T * k;
  const int64_t down = w_down.size(1);
  TORCH_CHECK(w_gu.size(1) == W && w_down.size(0) == W && experts >= 1 &&
                  ff >= 64 && w_gu.size(0) >= experts * 2 * ff &&
                  down >= experts * ff,
              "expert weights do not fit");
  TORCH_CHECK((W | ff) % 64 == 0 && W >= 64 && experts <= 1024 && k >= 1 &&
                  k <= 16 && T * x.stride(0) < (1ll << 31) &&
                  2 * ff * W < (1ll << 31) && W * down < (1ll << 31) &&
                  P < (1 << 23) - 255,
              "sizes that tiles of 256 do not take");
  TORCH_CHECK(weights.is_cuda() && ids.is_cuda() &&
              weights.scalar_type() == torch::kFloat32 &&
              weights.is_contiguous() && ids.scalar_type() == torch::kInt32 &&
              ids.is_contiguous() && ids.sizes() == weights.sizes() &&
              weights.size(0) == T);
  torch::Tensor y = torch::empty({P, W}, x.options());
  if (T == 0) return {y, ids};
  const int64_t max_items = std::min(P, experts) + P / 192;
  const int64_t groups = P <= 8192 ? 1 : std::min<int64_t>(64, (P + 2047) / 2048);
  // as in moe_expert_rows
  torch::Tensor plan = torch::empty(
      {4 * max_items + 2 * P + 17 + (groups > 1 ? groups * experts : 0)},
      x.options().dtype(torch::kInt32));
  int* items = plan.data_ptr<int>();
  int* perm = items + 4 * max_items;
  int* rows = perm + P;
  int* n_items = rows + P;
  int* claims = n_items + 1;
  torch::Tensor w_pair = torch::empty_like(weights);
  torch::Tensor h = torch::empty({P, ff}, x.options());
  auto stream = current_stream();
  arks_moe_plan(perm, rows, w_pair.data_ptr(), items, n_items, claims,
                claims + 16, ids.data_ptr(), weights.data_ptr(), (int)P, 0,
                (int)experts, 320, (int)max_items, (int)groups,
                engine_rounds(W, ff).data(), stream);
  // not rotated: an expert's row adds up in the same order at any number of rows
  const int once = P <= 160 * experts ? 1 : 0;
  arks_moe_gemm(h.data_ptr(), x.data_ptr(), w_gu.data_ptr(), perm, items,
                n_items, claims, scaled ? w_pair.data_ptr() : nullptr,
                x.stride(0), 2 * ff * W, W, (int)ff, (int)W, (int)k,
                (int)max_items, 256, 2, once, 0, stream);
  arks_moe_gemm(y.data_ptr(), h.data_ptr(), w_down.data_ptr(), perm, items,
                n_items, claims, nullptr, ff, ff, down, (int)W, (int)ff, (int)k,
                (int)max_items, 256, 0, once, 0, stream);
  return {y, plan.narrow(0, 4 * max_items + P, P).view({T, k})};
}

// The routed experts of x: the mix of moe_expert_rows
void moe_experts(torch::Tensor out, torch::Tensor x, torch::Tensor w13,
                 torch::Tensor w2, torch::Tensor weights, torch::Tensor ids,
                 int64_t expert_base, int64_t tile, bool mid, int64_t qt_up,
                 int64_t qt_down, int64_t experts) {
  check_bf16_contig(out, "out");
  TORCH_CHECK(x.dim() == 2 && out.size(0) == x.size(0) &&
              out.size(1) == x.size(1));
  const auto [y, w, rows] = moe_expert_rows(x, w13, w2, weights, ids,
                                            expert_base, tile, mid, qt_up, qt_down,
                                            c10::nullopt, false, experts);
  if (x.size(0) == 0) return;
  arks_moe_mix_rows(out.data_ptr(), y.data_ptr(), w.data_ptr(), rows.data_ptr(),
                    (int)x.size(0), (int)x.size(1), (int)weights.size(1),
                    current_stream());
}

void mfma_probe(torch::Tensor d, torch::Tensor a, torch::Tensor b) {
  check_bf16_contig(a, "a");
  check_bf16_contig(b, "b");
  TORCH_CHECK(d.scalar_type() == torch::kFloat32 && d.is_contiguous());
  TORCH_CHECK(a.size(0) == 16 && a.size(1) == 32);
  TORCH_CHECK(b.size(0) == 32 && b.size(1) == 16);
  arks_mfma_probe(d.data_ptr(), a.data_ptr(), b.data_ptr(), current_stream());
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  def_paged_attention(m);
  m.def("rmsnorm", &rmsnorm);
  m.def("fused_add_rmsnorm", &fused_add_rmsnorm);
  m.def("silu_mul", &silu_mul);
  m.def("rope_inplace", &rope_inplace);
  m.def("reshape_and_cache", &reshape_and_cache);
  m.def("rope_and_cache", &rope_and_cache, pybind11::arg("positions"),
        pybind11::arg("q"), pybind11::arg("k"), pybind11::arg("v"),
        pybind11::arg("k_cache"), pybind11::arg("v_cache"),
        pybind11::arg("slot_mapping"), pybind11::arg("cos_sin"),
        pybind11::arg("head_dim"), pybind11::arg("q_norm") = pybind11::none(),
        pybind11::arg("k_norm") = pybind11::none(), pybind11::arg("eps") = 0.0);
  m.def("attention_prefill_varlen", &attention_prefill_varlen);
  m.def("quant_fp8_rows", &quant_fp8_rows);
  m.def("rmsnorm_fp8", &rmsnorm_fp8);
  m.def("silu_mul_fp8", &silu_mul_fp8);
  m.def("greedy_sample", &greedy_sample);
  m.def("gumbel_sample", &gumbel_sample);
  m.def("ipc_alloc", &ipc_alloc);
  m.def("arm_flags", &arm_flags);
  m.def("ipc_alloc_free", &ipc_alloc_free);
  m.def("ipc_handle", &ipc_handle);
  m.def("ipc_open", &ipc_open);
  m.def("ipc_close", &ipc_close);
  m.def("one_shot_allreduce", &one_shot_allreduce);
  m.def("moe_topk", &moe_topk);
  m.def("moe_mix_rows", &moe_mix_rows);
  m.def("fused_add_rmsnorm_parts", &fused_add_rmsnorm_parts);
  m.def("rope_and_cache_parts", &rope_and_cache_parts);
  m.def("stream_gemm", &stream_gemm);
  m.def("stream_split", &stream_split, pybind11::arg("part"),
        pybind11::arg("a"), pybind11::arg("w"), pybind11::arg("per") = 0);
  m.def("stream_sum", &stream_sum);
  m.def("tile_silu", &tile_silu);
  m.def("wide_gemm", &wide_gemm);
  m.def("mid_gemm", &mid_gemm);
  m.def("mid_pair", &mid_pair);
  m.def("stage_rows", &stage_rows);
  m.def("moe_expert_rows", &moe_expert_rows, pybind11::arg("x"),
        pybind11::arg("w13"), pybind11::arg("w2"), pybind11::arg("weights"),
        pybind11::arg("ids"), pybind11::arg("expert_base"),
        pybind11::arg("tile"), pybind11::arg("mid"), pybind11::arg("qt_up"),
        pybind11::arg("qt_down"), pybind11::arg("logits"), pybind11::arg("renorm"),
        pybind11::arg("experts") = 0);
  m.def("moe_wide_rows", &moe_wide_rows);
  m.def("fused_add_rmsnorm_mix", &fused_add_rmsnorm_mix);
  m.def("moe_experts", &moe_experts, pybind11::arg("out"), pybind11::arg("x"),
        pybind11::arg("w13"), pybind11::arg("w2"), pybind11::arg("weights"),
        pybind11::arg("ids"), pybind11::arg("expert_base"),
        pybind11::arg("tile"), pybind11::arg("mid"), pybind11::arg("qt_up") = 4,
        pybind11::arg("qt_down") = 4, pybind11::arg("experts") = 0);
  m.def("mfma_probe", &mfma_probe);
  m.def("mfma_probe32", &mfma_probe32);
  m.def("tr16_probe", &tr16_probe);
}
