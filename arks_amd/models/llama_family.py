"""Qwen2 / Llama decoder family for the arks_amd engine.

One implementation covers both architectures (Qwen2 = Llama + QKV bias +
different rope_theta/vocab). HF-config-driven (arks_amd.config.ModelConfig);
weight names follow the HF checkpoint layout so safetensors load directly.

Compute path: arks_amd.ops HIP kernels for the products of up to 256 rows, the
gate and up products of many and experts of any number, RMSNorm / RoPE / paged
attention / SwiGLU; F.linear (hipBLASLt) for the other products; TP via
column/row-parallel shards with one RCCL all-reduce per attention and per MLP
block.
"""

from __future__ import annotations

import math

import torch
import torch.nn as nn

from .. import ops
from ..config import ModelConfig
from ..engine.forward_batch import ForwardBatch
from ..parallel.comm import get_tp_rank, get_tp_world_size
from ..parallel.layers import (
    ColumnParallelLinear,
    MergedColumnParallelLinear,
    ParallelLMHead,
    QKVParallelLinear,
    RowParallelLinear,
    passable,
)


class RMSNorm(nn.Module):
    fp8_out = False  # emit (fp8, scales) for a W8A8 consumer GEMM

    def __init__(self, hidden: int, eps: float, dtype=torch.bfloat16):
        super().__init__()
        self.weight = nn.Parameter(torch.ones(hidden, dtype=dtype), requires_grad=False)
        self.eps = eps

    def forward(self, x, residual=None):
        if self.fp8_out:
            x = ops.parts_sum(x)
            if residual is None:
                return ops.rmsnorm_fp8(x, self.weight, self.eps)
            q, s, res = ops.fused_add_rmsnorm_fp8(x, residual, self.weight, self.eps)
            return (q, s), res
        if residual is None:
            return ops.rmsnorm(x, self.weight, self.eps)
        return ops.fused_add_rmsnorm(x, residual, self.weight, self.eps)


class Attention(nn.Module):
    def __init__(self, cfg: ModelConfig, dtype=torch.bfloat16,
                 layer_idx: int = 0):
        super().__init__()
        tp = get_tp_world_size()
        self.head_dim = cfg.head_dim
        self.nq_local = cfg.num_attention_heads // tp
        self.nkv_local = cfg.num_key_value_heads // tp
        self.scale = 1.0 / math.sqrt(cfg.head_dim)
        # per-layer sliding window (HF Qwen2 max_window_layers/layer_types
        # semantics; Mistral = every layer; 0 = full attention). Masking
        # happens inside the kernels.
        self.window = cfg.layer_window(layer_idx)
        # SmolLM3 NoPE layers attend without positional encoding: k/v are
        # cached unrotated (HF modeling_smollm3.py:200-226 semantics)
        self.use_rope = cfg.layer_uses_rope(layer_idx)
        self.qkv_proj = QKVParallelLinear(
            cfg.hidden_size, cfg.head_dim, cfg.num_attention_heads,
            cfg.num_key_value_heads, bias=cfg.attention_bias, dtype=dtype,
        )
        self.o_proj = RowParallelLinear(
            cfg.num_attention_heads * cfg.head_dim, cfg.hidden_size, bias=False,
            dtype=dtype,
        )
        # Qwen3: per-head RMSNorm on q and k before RoPE
        self.q_norm = (
            RMSNorm(cfg.head_dim, cfg.rms_norm_eps, dtype) if cfg.qk_norm else None
        )
        self.k_norm = (
            RMSNorm(cfg.head_dim, cfg.rms_norm_eps, dtype) if cfg.qk_norm else None
        )

    def forward(self, x, batch: ForwardBatch, kv_cache, parts: bool = False):
        """parts: the caller takes ops.Parts too."""
        T = (x[0] if isinstance(x, tuple) else x).shape[0]
        # the rotation kernel can norm the heads of q and k
        rope_norms = (self.use_rope and self.q_norm is not None
                      and self.head_dim in ops.HEAD_NORM_DIMS
                      and passable(self.q_norm, RMSNorm)
                      and passable(self.k_norm, RMSNorm))
        # in decode steps k and v are read from the cache alone
        if (not batch.is_prefill and self.use_rope and not isinstance(x, tuple)
                and not self.qkv_proj.fp8
                and (self.q_norm is None or rope_norms)
                and self.head_dim % 8 == 0
                and passable(self.qkv_proj, ColumnParallelLinear)):
            qkv = ops.linear_parts(x, self.qkv_proj.weight, self.qkv_proj.bias)
        else:
            qkv = self.qkv_proj(x)
        if isinstance(qkv, ops.Parts):
            norms = {} if self.q_norm is None else dict(
                q_norm=self.q_norm.weight, k_norm=self.k_norm.weight,
                eps=self.q_norm.eps)
            q = ops.rope_and_cache_parts(
                batch.positions, qkv, kv_cache[0], kv_cache[1],
                batch.slot_mapping, self._cos_sin, self.head_dim, **norms)
            return self._out(self._decode(q, batch, kv_cache).view(T, -1), batch,
                             parts)
        # Strided views into the fused QKV buffer — RoPE/cache/attention
        # kernels take row strides, so no .contiguous() copies on the hot path.
        q, k, v = self.qkv_proj.split_qkv(qkv)
        k_cache, v_cache = kv_cache
        norms = {}
        if self.q_norm is not None and not rope_norms:
            hd = self.head_dim
            q = self.q_norm(
                q.contiguous().view(-1, hd)).view(T, self.nq_local * hd)
            k = self.k_norm(
                k.contiguous().view(-1, hd)).view(T, self.nkv_local * hd)
            # reshape_and_cache wants one shared kv stride (also of one row)
            v = v.reshape(-1).view(T, -1)
        elif self.q_norm is not None:
            norms = dict(q_norm=self.q_norm.weight, k_norm=self.k_norm.weight,
                         eps=self.q_norm.eps)
        if self.use_rope:
            q, k = ops.rope_and_cache(
                batch.positions, q, k, v, k_cache, v_cache,
                batch.slot_mapping, self._cos_sin, self.head_dim, **norms,
            )
        else:
            # NoPE layer: cache k/v as-is, q unrotated
            ops.reshape_and_cache(
                k.unflatten(-1, (self.nkv_local, self.head_dim)),
                v.unflatten(-1, (self.nkv_local, self.head_dim)),
                k_cache, v_cache, batch.slot_mapping,
            )
        k = k.unflatten(-1, (self.nkv_local, self.head_dim))
        v = v.unflatten(-1, (self.nkv_local, self.head_dim))
        q = q.unflatten(-1, (self.nq_local, self.head_dim))
        if batch.is_prefill:
            if batch.block_tables is not None:
                # Prefix-cache hit in the batch: new tokens attend over the
                # full paged KV (cached prefix + the rows just written above).
                out = ops.attention_extend_paged(
                    q, k_cache, v_cache, batch.block_tables, batch.seq_lens,
                    batch.cu_seqlens, batch.seq_lens_list, self.scale,
                    window=self.window, tiles=batch.ext_tiles,
                    step_cache=batch.step_cache,
                )
            else:
                out = ops.attention_prefill_varlen(
                    q, k, v, batch.cu_seqlens, batch.seq_lens_list, self.scale,
                    window=self.window,
                )
        else:
            out = self._decode(q, batch, kv_cache)
        return self._out(out.view(T, -1), batch, parts)

    def _out(self, x, batch: ForwardBatch, parts: bool):
        if not parts:
            return self.o_proj(x)
        return self.o_proj(x, parts=True, own_cut=not batch.is_prefill)

    def _decode(self, q, batch: ForwardBatch, kv_cache):
        k_cache, v_cache = kv_cache
        return ops.attention_decode_paged(
            q.view(q.shape[0], self.nq_local, self.head_dim), k_cache, v_cache,
            batch.block_tables, batch.seq_lens,
            self.scale, window=self.window, plan=ops.step_decode_plan(
                batch.seq_lens, self.nkv_local, self.window,
                k_cache.dtype != torch.bfloat16, None, batch.step_cache),
        )


class MLP(nn.Module):
    def __init__(self, cfg: ModelConfig, dtype=torch.bfloat16):
        super().__init__()
        self.gate_up_proj = MergedColumnParallelLinear(
            cfg.hidden_size, cfg.intermediate_size, bias=False, dtype=dtype
        )
        self.down_proj = RowParallelLinear(
            cfg.intermediate_size, cfg.hidden_size, bias=False, dtype=dtype
        )

    fp8 = False

    def forward(self, x, parts: bool = False, own_cut: bool = True):
        """parts: the caller takes ops.Parts too (own_cut as ops.linear_parts)."""
        if self.fp8:
            return self.down_proj(ops.silu_mul_fp8(self.gate_up_proj(x)))
        if (isinstance(x, tuple) or self.gate_up_proj.fp8
                or not passable(self.gate_up_proj, ColumnParallelLinear)):
            h = ops.silu_mul(self.gate_up_proj(x))
        else:
            h = ops.linear_silu_mul(x, self.gate_up_proj.weight)
        if not parts:
            return self.down_proj(h)
        return self.down_proj(h, parts=True, own_cut=own_cut)


class MoEMLP(nn.Module):
    """Mixtral-style sparse MoE block, expert-parallel over the TP group:
    each rank owns num_local_experts/tp whole experts (an expert's FFN is
    never split), computes its experts' contributions for the tokens routed
    to them, and one all-reduce sums the partial outputs — the same single
    collective per block as the dense RowParallel MLP. The router (gate) is
    replicated so every rank routes identically."""

    fp8 = False  # MoE experts stay bf16 (v1)

    def __init__(self, cfg: ModelConfig, dtype=torch.bfloat16):
        super().__init__()
        tp = get_tp_world_size()
        E = cfg.num_local_experts
        assert E % tp == 0, (E, tp)
        self.num_experts = E
        self.top_k = cfg.num_experts_per_tok
        self.local_experts = E // tp
        self.expert_base = get_tp_rank() * self.local_experts
        self.hidden = cfg.hidden_size
        self.inter = cfg.moe_intermediate_size or cfg.intermediate_size
        self.norm_topk = cfg.norm_topk_prob
        self.gate = nn.Parameter(
            torch.empty(E, cfg.hidden_size, dtype=dtype), requires_grad=False
        )
        # [gate rows | up rows] and down per local expert, in the
        # checkpoint's own [out, in] layout: the expert kernels read weight
        # rows along their input
        self.w_up = nn.Parameter(
            torch.empty(self.local_experts, 2 * self.inter, self.hidden,
                        dtype=dtype), requires_grad=False,
        )
        self.w_down = nn.Parameter(
            torch.empty(self.local_experts, self.hidden, self.inter,
                        dtype=dtype), requires_grad=False,
        )
        # Qwen2-MoE shared expert (dense, TP-sharded like a normal MLP) with
        # a sigmoid scalar gate
        self.shared = None
        self.shared_gate = None
        if cfg.shared_expert_intermediate_size:
            import dataclasses

            dense_cfg = dataclasses.replace(
                cfg, intermediate_size=cfg.shared_expert_intermediate_size
            )
            self.shared = MLP(dense_cfg, dtype)
            self.shared_gate = nn.Parameter(
                torch.zeros(1, cfg.hidden_size, dtype=dtype),
                requires_grad=False,
            )

    @property
    def w13(self) -> torch.Tensor:
        """w_up as the right operand of a product, [expert, in, 2 * inter]."""
        return self.w_up.transpose(1, 2)

    @property
    def w2(self) -> torch.Tensor:
        """w_down as the right operand of a product, [expert, inter, out]."""
        return self.w_down.transpose(1, 2)

    # rows up to which decode steps are captured as graphs (the expert kernels
    # need no host read of the routing at any size)
    DENSE_TOKENS = 256

    def forward(self, x, parts: bool = False):
        """parts: the caller takes ops.Mixed too (one rank, no shared expert)."""
        from ..parallel.comm import tp_all_reduce

        mixed = parts and self.shared is None and get_tp_world_size() == 1
        if mixed:
            out = ops.moe_routed_parts(x, self.gate, self.top_k, self.norm_topk,
                                       self.w_up, self.w_down, self.expert_base)
            if out is not None:
                return out
        weights, selected = ops.moe_route(x, self.gate, self.top_k,
                                          self.norm_topk)
        if mixed:
            return ops.moe_experts_parts(
                x, self.w_up, self.w_down, weights, selected, self.expert_base,
                self.num_experts)
        out = ops.moe_experts(x, self.w_up, self.w_down, weights, selected,
                              self.expert_base, self.num_experts)
        out = tp_all_reduce(out)
        if self.shared is not None:
            gate = torch.sigmoid(
                torch.nn.functional.linear(x, self.shared_gate).float()
            ).to(x.dtype)
            out = out + gate * self.shared(x)
        return out


class DecoderLayer(nn.Module):
    def __init__(self, cfg: ModelConfig, dtype=torch.bfloat16,
                 layer_idx: int = 0):
        super().__init__()
        self.input_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps, dtype)
        self.self_attn = Attention(cfg, dtype, layer_idx=layer_idx)
        self.post_attention_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps, dtype)
        self.mlp = (
            MoEMLP(cfg, dtype) if cfg.num_local_experts > 0 else MLP(cfg, dtype)
        )

    def forward(self, x, residual, batch: ForwardBatch, kv_cache,
                parts: bool = False):
        """parts: the caller takes ops.Parts and ops.Mixed too."""
        if residual is None:
            residual = x
            x = self.input_layernorm(x)
        else:
            x, residual = self.input_layernorm(x, residual)
        # the norm behind a row-parallel product can add its split sums; what a
        # hook may look at stays a tensor
        if (passable(self.self_attn, Attention)
                and passable(self.self_attn.o_proj, RowParallelLinear)
                and passable(self.post_attention_layernorm, RMSNorm)):
            x = self.self_attn(x, batch, kv_cache, parts=True)
        else:
            x = self.self_attn(x, batch, kv_cache)
        x, residual = self.post_attention_layernorm(x, residual)
        if parts and passable(self.mlp, MoEMLP):
            return self.mlp(x, parts=True), residual
        if (parts and passable(self.mlp, MLP)
                and passable(self.mlp.down_proj, RowParallelLinear)):
            return (self.mlp(x, parts=True, own_cut=not batch.is_prefill),
                    residual)
        return self.mlp(x), residual


class LlamaFamilyForCausalLM(nn.Module):
    """Covers Qwen2ForCausalLM and LlamaForCausalLM."""

    def __init__(self, cfg: ModelConfig, dtype=torch.bfloat16):
        super().__init__()
        self.cfg = cfg
        self.dtype = dtype
        self.embed_tokens = nn.Embedding(
            cfg.vocab_size, cfg.hidden_size, dtype=dtype
        )
        self.embed_tokens.weight.requires_grad_(False)
        self.layers = nn.ModuleList(
            DecoderLayer(cfg, dtype, layer_idx=i)
            for i in range(cfg.num_hidden_layers)
        )
        self.norm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps, dtype)
        self.lm_head = ParallelLMHead(cfg.hidden_size, cfg.vocab_size, dtype)
        cos_sin = self._build_cos_sin()
        self.register_buffer("rope_cos_sin", cos_sin, persistent=False)
        for layer in self.layers:
            layer.self_attn._cos_sin = cos_sin

    def quantize_fp8(self) -> None:
        """W8A8 fp8 for the weight-bandwidth-bound GEMMs (profiles/r01_p2:
        gate_up/down/lm_head dominate the decode step; o_proj is left bf16 —
        no gain at its size and its input is the attention output, which
        has no producing kernel to fuse a quant into)."""
        from ..parallel.layers import quantize_module_fp8

        for layer in self.layers:
            quantize_module_fp8(layer.self_attn.qkv_proj)
            layer.input_layernorm.fp8_out = True
            if isinstance(layer.mlp, MoEMLP):
                continue  # MoE experts stay bf16 (v1)
            quantize_module_fp8(layer.mlp.gate_up_proj)
            quantize_module_fp8(layer.mlp.down_proj)
            # producing kernels emit fp8 directly (fused activation quant)
            layer.post_attention_layernorm.fp8_out = True
            layer.mlp.fp8 = True
        quantize_module_fp8(self.lm_head)
        self.norm.fp8_out = True

    def _build_cos_sin(self, min_len: int | None = None):
        from ..ops import ref

        return ref.rope_cos_sin_cache(
            self.cfg.head_dim,
            max(self.cfg.max_position_embeddings, min_len or 0),
            self.cfg.rope_theta, rope_scaling=self.cfg.rope_scaling,
        )

    def extend_rope_table(self, min_len: int) -> None:
        """Grow the RoPE cos/sin table to at least `min_len` positions
        (serving past max_position_embeddings would otherwise read out of
        bounds in the rope kernel; plain RoPE extrapolates)."""
        if self.rope_cos_sin.shape[0] >= min_len:
            return
        cache = self._build_cos_sin(min_len).to(
            device=self.rope_cos_sin.device, dtype=self.rope_cos_sin.dtype
        )
        self.register_buffer("rope_cos_sin", cache, persistent=False)
        for layer in self.layers:
            layer.self_attn._cos_sin = cache

    def _apply(self, fn, recurse=True):  # keep the shared cos_sin in sync
        out = super()._apply(fn, recurse)
        for layer in self.layers:
            layer.self_attn._cos_sin = self.rope_cos_sin
        return out

    def forward(self, batch: ForwardBatch, kv_caches: list) -> torch.Tensor:
        """Returns logits for batch.logits_indices rows."""
        batch.step_cache = {}
        x = self.embed_tokens(batch.input_ids)
        residual = None
        last = len(self.layers) - 1
        for i, layer in enumerate(self.layers):
            parts = passable(layer, DecoderLayer)
            if parts and i < last:
                after = self.layers[i + 1]
                parts = (passable(after, DecoderLayer)
                         and passable(after.input_layernorm, RMSNorm))
            elif parts:
                parts = passable(self.norm, RMSNorm)
            x, residual = (layer(x, residual, batch, kv_caches[i], parts=True)
                           if parts else
                           layer(x, residual, batch, kv_caches[i]))
        x, _ = self.norm(x, residual)
        if isinstance(x, tuple):  # fp8: (values, per-token scales)
            q8, sc = x
            if batch.logits_indices is not None:
                q8 = q8[batch.logits_indices]
                sc = sc[batch.logits_indices]
            return self.lm_head((q8, sc))
        if batch.logits_indices is not None:
            x = x[batch.logits_indices]
        return self.lm_head(x)

    # ------------------------- weight loading -------------------------
    def load_hf_state_dict(self, tensors: dict[str, torch.Tensor]) -> None:
        """Load an HF-layout state dict (full tensors; sharded here)."""
        pending_qkv: dict[int, dict] = {}
        pending_mlp: dict[int, dict] = {}
        own = dict(self.named_parameters())

        def put(name, value):
            p = own[name]
            assert p.shape == value.shape, (name, p.shape, value.shape)
            p.data.copy_(value.to(p.dtype))

        def put_cat(name, parts):
            # fused params load piecewise: each (pinned) slice goes straight
            # into its span of the parameter — no host-side torch.cat copy
            p = own[name]
            off = 0
            for part in parts:
                n = part.shape[0]
                p.data[off:off + n].copy_(part.to(p.dtype))
                off += n
            assert off == p.shape[0], (name, off, p.shape)

        for name, w in tensors.items():
            name = name.removeprefix("model.")
            if name == "embed_tokens.weight":
                put("embed_tokens.weight", w)
                if self.cfg.tie_word_embeddings:
                    put("lm_head.weight", self.lm_head.shard(w))
            elif name in ("lm_head.weight",):
                put("lm_head.weight", self.lm_head.shard(w))
            elif name == "norm.weight":
                put("norm.weight", w)
            elif name.startswith("layers."):
                parts = name.split(".")
                li = int(parts[1])
                sub = ".".join(parts[2:])
                layer = self.layers[li]
                if sub in ("input_layernorm.weight", "post_attention_layernorm.weight"):
                    put(f"layers.{li}.{sub}", w)
                elif sub in ("self_attn.q_norm.weight", "self_attn.k_norm.weight"):
                    put(f"layers.{li}.{sub}", w)
                elif sub.startswith("self_attn.") and sub.split(".")[1] in (
                    "q_proj", "k_proj", "v_proj",
                ):
                    proj, param = sub.split(".")[1], sub.split(".")[2]
                    pending_qkv.setdefault(li, {})[f"{proj}.{param}"] = w
                    d = pending_qkv[li]
                    keys_w = {"q_proj.weight", "k_proj.weight", "v_proj.weight"}
                    keys_b = {"q_proj.bias", "k_proj.bias", "v_proj.bias"}
                    if keys_w <= d.keys():
                        parts = layer.self_attn.qkv_proj.shard_qkv_parts(
                            d["q_proj.weight"], d["k_proj.weight"], d["v_proj.weight"]
                        )
                        put_cat(f"layers.{li}.self_attn.qkv_proj.weight", parts)
                        for kk in keys_w:
                            del d[kk]
                    if layer.self_attn.qkv_proj.bias is not None and keys_b <= d.keys():
                        parts = layer.self_attn.qkv_proj.shard_qkv_parts(
                            d["q_proj.bias"], d["k_proj.bias"], d["v_proj.bias"]
                        )
                        put_cat(f"layers.{li}.self_attn.qkv_proj.bias", parts)
                        for kk in keys_b:
                            del d[kk]
                elif sub == "self_attn.o_proj.weight":
                    put(
                        f"layers.{li}.self_attn.o_proj.weight",
                        layer.self_attn.o_proj.shard(w),
                    )
                elif sub in ("mlp.gate_proj.weight", "mlp.up_proj.weight"):
                    pending_mlp.setdefault(li, {})[sub] = w
                    d = pending_mlp[li]
                    if {"mlp.gate_proj.weight", "mlp.up_proj.weight"} <= d.keys():
                        parts = layer.mlp.gate_up_proj.shard_merged_parts(
                            d["mlp.gate_proj.weight"], d["mlp.up_proj.weight"]
                        )
                        put_cat(f"layers.{li}.mlp.gate_up_proj.weight", parts)
                        d.clear()
                elif sub == "mlp.down_proj.weight":
                    put(f"layers.{li}.mlp.down_proj.weight", layer.mlp.down_proj.shard(w))
                elif sub == "mlp.shared_expert_gate.weight":
                    layer.mlp.shared_gate.data.copy_(
                        w.to(layer.mlp.shared_gate.dtype))
                elif sub in ("mlp.shared_expert.gate_proj.weight",
                             "mlp.shared_expert.up_proj.weight"):
                    pending_mlp.setdefault((li, "se"), {})[sub] = w
                    d = pending_mlp[(li, "se")]
                    if len(d) == 2:
                        fused = layer.mlp.shared.gate_up_proj.shard_merged(
                            d["mlp.shared_expert.gate_proj.weight"],
                            d["mlp.shared_expert.up_proj.weight"],
                        )
                        layer.mlp.shared.gate_up_proj.weight.data.copy_(
                            fused.to(layer.mlp.shared.gate_up_proj.weight.dtype))
                        d.clear()
                elif sub == "mlp.shared_expert.down_proj.weight":
                    layer.mlp.shared.down_proj.weight.data.copy_(
                        layer.mlp.shared.down_proj.shard(w).to(
                            layer.mlp.shared.down_proj.weight.dtype))
                elif sub in ("block_sparse_moe.gate.weight", "mlp.gate.weight"):
                    layer.mlp.gate.data.copy_(w.to(layer.mlp.gate.dtype))
                elif sub.startswith("mlp.experts."):
                    # Qwen3-MoE naming: experts.N.{gate,up,down}_proj.weight
                    moe = layer.mlp
                    e = int(sub.split(".")[2])
                    which = sub.split(".")[3]
                    le = e - moe.expert_base
                    if 0 <= le < moe.local_experts:
                        I = moe.inter
                        if which == "gate_proj":
                            moe.w_up.data[le, :I].copy_(w.to(moe.w_up.dtype))
                        elif which == "up_proj":
                            moe.w_up.data[le, I:].copy_(w.to(moe.w_up.dtype))
                        elif which == "down_proj":
                            moe.w_down.data[le].copy_(w.to(moe.w_down.dtype))
                elif sub.startswith("block_sparse_moe.experts."):
                    # Mixtral expert naming: w1=gate, w3=up, w2=down.
                    # EP-sharded: only this rank's experts are kept.
                    moe = layer.mlp
                    e = int(sub.split(".")[2])
                    which = sub.split(".")[3]
                    le = e - moe.expert_base
                    if 0 <= le < moe.local_experts:
                        I = moe.inter
                        if which == "w1":
                            moe.w_up.data[le, :I].copy_(w.to(moe.w_up.dtype))
                        elif which == "w3":
                            moe.w_up.data[le, I:].copy_(w.to(moe.w_up.dtype))
                        elif which == "w2":
                            moe.w_down.data[le].copy_(w.to(moe.w_down.dtype))
                # rotary_emb.inv_freq etc. are ignored (recomputed)

    @torch.no_grad()
    def random_init(self, seed: int = 0) -> None:
        """Random-init with TP-consistent semantics: full HF-layout tensors
        are generated deterministically per name (so every TP rank sees
        slices of the SAME logical weights) and routed through the normal
        shard-aware loader. Generates on the model's device when possible."""
        import zlib

        cfg = self.cfg
        dev = self.embed_tokens.weight.device

        def gen(name: str, *shape, std: float = 0.02) -> torch.Tensor:
            s = (seed * 1000003 + zlib.crc32(name.encode())) % (2**63 - 1)
            if dev.type == "cuda":
                g = torch.Generator(device=dev).manual_seed(s)
                t = torch.randn(shape, generator=g, dtype=torch.float32, device=dev)
            else:
                g = torch.Generator().manual_seed(s)
                t = torch.randn(shape, generator=g, dtype=torch.float32)
            return t.mul_(std)

        H, I, hd = cfg.hidden_size, cfg.intermediate_size, cfg.head_dim
        nq, nkv = cfg.num_attention_heads, cfg.num_key_value_heads
        glob: dict[str, torch.Tensor] = {
            "model.embed_tokens.weight": gen("embed", cfg.vocab_size, H),
            "model.norm.weight": torch.ones(H),
        }
        if not cfg.tie_word_embeddings:
            glob["lm_head.weight"] = gen("lm_head", cfg.vocab_size, H)
        self.load_hf_state_dict(glob)
        del glob
        for i in range(cfg.num_hidden_layers):
            pre = f"model.layers.{i}"
            tensors = {
                f"{pre}.self_attn.q_proj.weight": gen(f"{pre}.q", nq * hd, H),
                f"{pre}.self_attn.k_proj.weight": gen(f"{pre}.k", nkv * hd, H),
                f"{pre}.self_attn.v_proj.weight": gen(f"{pre}.v", nkv * hd, H),
                f"{pre}.self_attn.o_proj.weight": gen(f"{pre}.o", H, nq * hd),
                f"{pre}.input_layernorm.weight": torch.ones(H),
                f"{pre}.post_attention_layernorm.weight": torch.ones(H),
            }
            if cfg.num_local_experts > 0:
                Ie = cfg.moe_intermediate_size or I
                if cfg.shared_expert_intermediate_size:
                    Is = cfg.shared_expert_intermediate_size
                    sp = f"{pre}.mlp.shared_expert"
                    tensors[f"{sp}.gate_proj.weight"] = gen(f"{sp}.g", Is, H)
                    tensors[f"{sp}.up_proj.weight"] = gen(f"{sp}.u", Is, H)
                    tensors[f"{sp}.down_proj.weight"] = gen(f"{sp}.d", H, Is)
                    tensors[f"{pre}.mlp.shared_expert_gate.weight"] = gen(
                        f"{sp}.sg", 1, H
                    )
                qstyle = not cfg.architecture.startswith("MixtralFor")
                gname = "mlp.gate" if qstyle else "block_sparse_moe.gate"
                tensors[f"{pre}.{gname}.weight"] = gen(
                    f"{pre}.moe.gate", cfg.num_local_experts, H
                )
                for e in range(cfg.num_local_experts):
                    if qstyle:
                        ep = f"{pre}.mlp.experts.{e}"
                        tensors[f"{ep}.gate_proj.weight"] = gen(f"{ep}.w1", Ie, H)
                        tensors[f"{ep}.up_proj.weight"] = gen(f"{ep}.w3", Ie, H)
                        tensors[f"{ep}.down_proj.weight"] = gen(f"{ep}.w2", H, Ie)
                    else:
                        ep = f"{pre}.block_sparse_moe.experts.{e}"
                        tensors[f"{ep}.w1.weight"] = gen(f"{ep}.w1", Ie, H)
                        tensors[f"{ep}.w3.weight"] = gen(f"{ep}.w3", Ie, H)
                        tensors[f"{ep}.w2.weight"] = gen(f"{ep}.w2", H, Ie)
            else:
                tensors[f"{pre}.mlp.gate_proj.weight"] = gen(f"{pre}.gate", I, H)
                tensors[f"{pre}.mlp.up_proj.weight"] = gen(f"{pre}.up", I, H)
                tensors[f"{pre}.mlp.down_proj.weight"] = gen(f"{pre}.down", H, I)
            if cfg.qk_norm:
                tensors[f"{pre}.self_attn.q_norm.weight"] = torch.ones(hd)
                tensors[f"{pre}.self_attn.k_norm.weight"] = torch.ones(hd)
            if cfg.attention_bias:
                tensors[f"{pre}.self_attn.q_proj.bias"] = torch.zeros(nq * hd)
                tensors[f"{pre}.self_attn.k_proj.bias"] = torch.zeros(nkv * hd)
                tensors[f"{pre}.self_attn.v_proj.bias"] = torch.zeros(nkv * hd)
            # load layer-by-layer to bound peak memory
            self.load_hf_state_dict(tensors)
