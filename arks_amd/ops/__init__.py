"""Op dispatch for arks_amd.

On GPU tensors every op runs the in-tree gfx950 HIP extension
(``arks_amd._C``) — there is no eager fallback: if the extension is missing
on a CUDA/ROCm device we raise immediately so a silently-slow PyTorch path
can never masquerade as the native one. On CPU tensors ops run the plain
PyTorch reference (arks_amd/ops/ref.py) so the engine/scheduler/model layers
are unit-testable without a GPU.
"""

from __future__ import annotations

import functools
import math
import os

import torch

from . import ref

_C = None
_C_ERR: str | None = None


def _load_extension():
    global _C, _C_ERR
    if _C is not None or _C_ERR is not None:
        return _C
    try:
        from . import _load

        _C = _load.load("arks_amd_C")  # the built .so in-tree
    except Exception as e:  # pragma: no cover - exercised only when unbuilt
        _C_ERR = f"{type(e).__name__}: {e}"
    return _C


def native_available() -> bool:
    return _load_extension() is not None


def _native():
    c = _load_extension()
    if c is None:
        raise RuntimeError(
            "arks_amd HIP extension (arks_amd._C) is not built but a GPU op was "
            "requested. Build it with `python -m arks_amd.ops.build` "
            f"(import error: {_C_ERR})"
        )
    return c


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float = 1e-6) -> torch.Tensor:
    if x.is_cuda:
        out = torch.empty_like(x)
        _native().rmsnorm(out, x, weight, eps)
        return out
    return ref.rmsnorm(x, weight, eps)


def fused_add_rmsnorm(x, residual, weight, eps: float = 1e-6):
    """In-place on GPU: residual += x (written to residual), out = norm(residual)."""
    if isinstance(x, Mixed):
        out = torch.empty_like(residual)
        _native().fused_add_rmsnorm_mix(out, x.y, x.weights, x.rows, residual,
                                        weight, eps)
        return out, residual
    if isinstance(x, Parts):
        assert x.bias is None
        out = torch.empty_like(residual)
        _native().fused_add_rmsnorm_parts(out, x.sums, residual, weight, eps)
        return out, residual
    if x.is_cuda:
        out = torch.empty_like(x)
        _native().fused_add_rmsnorm(out, x, residual, weight, eps)
        return out, residual
    return ref.fused_add_rmsnorm(x, residual, weight, eps)


def silu_mul(gate_up: torch.Tensor) -> torch.Tensor:
    if gate_up.is_cuda:
        shape = list(gate_up.shape)
        shape[-1] //= 2
        out = gate_up.new_empty(shape)
        _native().silu_mul(out, gate_up)
        return out
    return ref.silu_mul(gate_up)


def rope_apply_inplace(positions, q, k, cos_sin, head_dim: int):
    """Rotates q and k in place (GPU). CPU path returns new tensors."""
    if q.is_cuda:
        _native().rope_inplace(positions, q, k, cos_sin, head_dim)
        return q, k
    return ref.rope_apply(positions, q, k, cos_sin, head_dim)


HEAD_NORM_DIMS = (32, 64, 128, 256)  # head sizes rope_and_cache norms


def rope_and_cache(positions, q, k, v, k_cache, v_cache, slot_mapping,
                   cos_sin, head_dim: int, q_norm=None, k_norm=None,
                   eps: float = 0.0):
    """Fused RoPE + paged-cache write (GPU): rotates q/k in place and
    scatters rotated k + v into the cache in one launch. CPU path runs the
    reference steps. q_norm, k_norm [head_dim]: every head of q and k is
    RMS-normed first (GPU: head_dim in HEAD_NORM_DIMS)."""
    if q.is_cuda:
        _native().rope_and_cache(positions, q, k, v, k_cache, v_cache,
                                 slot_mapping, cos_sin, head_dim, q_norm,
                                 k_norm, eps)
        return q, k
    T = q.shape[0]
    if q_norm is not None:
        q, k = (ref.rmsnorm(t.reshape(T, -1, head_dim), w, eps).view(T, -1)
                for t, w in ((q, q_norm), (k, k_norm)))
    q2, k2 = ref.rope_apply(positions, q, k, cos_sin, head_dim)
    nkv = k.numel() // max(T, 1) // head_dim
    ref.reshape_and_cache(
        k2.reshape(T, nkv, head_dim), v.reshape(T, nkv, head_dim),
        k_cache, v_cache, slot_mapping,
    )
    return q2, k2


def rope_and_cache_parts(positions, qkv, k_cache, v_cache, slot_mapping,
                         cos_sin, head_dim: int, q_norm=None, k_norm=None,
                         eps: float = 0.0):
    """rope_and_cache of a projection [q | k | v] that is still Parts: returns
    q, and writes k and v to the cache alone."""
    _, T, width = qkv.sums.shape
    q = torch.empty((T, width - 2 * k_cache.shape[1] * head_dim),
                    dtype=torch.bfloat16, device=qkv.sums.device)
    _native().rope_and_cache_parts(positions, q, qkv.sums, qkv.bias, k_cache,
                                   v_cache, slot_mapping, cos_sin, head_dim,
                                   q_norm, k_norm, eps)
    return q


def reshape_and_cache(k, v, k_cache, v_cache, slot_mapping):
    if k.is_cuda:
        _native().reshape_and_cache(k, v, k_cache, v_cache, slot_mapping)
        return
    ref.reshape_and_cache(k, v, k_cache, v_cache, slot_mapping)


PREFILL_QTILE = 64  # q rows per workgroup in the prefill kernel


def build_prefill_tiles(seq_lens: list[int], device) -> torch.Tensor:
    """int32 [ntiles, 2] of (seq_idx, q0) covering every sequence in 64-row
    tiles — the prefill kernel's grid."""
    tiles = []
    for i, n in enumerate(seq_lens):
        for q0 in range(0, n, PREFILL_QTILE):
            tiles.append((i, q0))
    return torch.tensor(tiles, dtype=torch.int32, device=device).reshape(-1, 2)


def attention_prefill_varlen(q, k, v, cu_seqlens, seq_lens: list[int],
                             scale: float, window: int = 0):
    """Causal varlen prefill attention. seq_lens is the host-side list of
    per-sequence lengths (used to build the q-tile grid without a D2H sync).
    window > 0 = sliding-window attention."""
    if q.is_cuda:
        out = torch.empty_like(q)
        tile_info = build_prefill_tiles(seq_lens, q.device)
        _native().attention_prefill_varlen(out, q, k, v, cu_seqlens, tile_info,
                                           scale, window)
        return out
    return ref.attention_prefill_varlen(q, k, v, cu_seqlens, scale, window)


def stage_rows(prompts: list, outputs: list, tables: list, starts, counts, ids,
               pos, slots, lens, block_tables, block_size: int,
               rows: int = 0) -> None:
    """What a step's rows read, into host tensors (see bindings.cpp)."""
    _native().stage_rows(prompts, outputs, tables, starts, counts, ids, pos,
                         slots, lens, block_tables, block_size, rows)


def upload(tensors: list, device) -> list:
    """Host tensors (or what stays on the host) on a device: moved as one, since
    a step waits for every copy of its own (a dozen took 300 us)."""
    device = torch.device(device)
    held = [isinstance(t, torch.Tensor) for t in tensors]
    if device.type != "cuda":
        return [t.to(device) if h else t for t, h in zip(tensors, held)]
    at, total = [], 0
    for t, h in zip(tensors, held):
        at.append(total)
        total += -(-t.numel() * t.element_size() // 16) * 16 if h else 0
    host = torch.empty(total, dtype=torch.uint8, pin_memory=True)
    whole = lambda buf, t, o: buf[o:o + t.numel() * t.element_size()].view(
        t.dtype).view(t.shape)
    for t, o, h in zip(tensors, at, held):
        if h:
            whole(host, t, o).copy_(t)
    moved = host.to(device, non_blocking=True)
    return [whole(moved, t, o) if h else t
            for t, o, h in zip(tensors, at, held)]


EXTEND2_QTILE = 256  # q rows per workgroup in the 8-wave ladder kernel
E2_KVBLK = 64        # keys per LDS tile in the ladder kernel
# Sequences with at least this many new q tokens go to the 256-row ladder
# kernel; shorter ones (decode-adjacent chunks, prefix-cache hits) stay on
# the 64-row kernel where a mostly-empty 256-row tile would waste waves.
EXTEND2_MIN_QLEN = 97
EXTEND2_SHORT_KEYS = 256  # shorter portions with this many keys go there too


def build_extend_tiles(q_lens: list[int], kv_lens: list[int] | None,
                       kv_fp8: bool, device, num_q_heads: int = 32,
                       ladder: bool = True, flash_decode: bool = True,
                       min_ladder: int = EXTEND2_MIN_QLEN):
    """Per-seq routing for the extend dispatcher:
    (tiles64, tiles256 [n,4], decode_rows, combine_table, ws_rows).

    q_len == 1 sequences (decode steps mixed into a prefill batch) go to
    the flash-decode kernel — an extend q-tile for one query scans the
    full KV with 255 masked rows (~6x slower than the decode kernel's
    partitioned scan). Remaining sequences split between the 64-row and
    256-row extend kernels; tiles are sorted by DESCENDING key depth
    (causal q-tiles differ up to 4x in KV work and the dispatcher issues
    blocks in order — deep tiles first removes the straggler tail). When
    the batch is too small to fill the chip, deep 256-row tiles are
    additionally SPLIT over their KV range flash-decode-style (part rows
    + a combine pass over f32 partials); split parts sort first so the
    partial workspace only covers them. min_ladder: the shortest portion
    that goes to the 256-row kernel. Build once per batch and reuse across
    all layers."""
    t64, t256, dec = [], [], []
    kvl = kv_lens if kv_lens is not None else q_lens
    # Few short portions behind a context leave the 64-row kernel a few
    # workgroups that walk all keys alone; the 256-row kernel splits them.
    # 28/4 heads, us, 64-row and split: 65 rows at 256 keys 18.4 and 17.0, at
    # 512 keys 33 and 20, at 6113 keys 414 and 48; 4 x 33 rows at 1024 keys 76
    # and 39, 8 x 33 rows 77 and 71, 16 x 33 rows (more than one workgroup per
    # CU) 83 and 107.
    short = [i for i, n in enumerate(q_lens)
             if 0 < n < min_ladder and not (n == 1 and flash_decode)]
    few = (ladder and not kv_fp8
           and sum(-(-q_lens[i] // PREFILL_QTILE) for i in short) * num_q_heads
           <= 256)
    deep = {i for i in short if few and kvl[i] >= EXTEND2_SHORT_KEYS}
    for i, n in enumerate(q_lens):
        off = kvl[i] - n
        if n == 1 and flash_decode:
            dec.append(i)
        elif kv_fp8 or (n < min_ladder and i not in deep) or not ladder:
            for q0 in range(0, n, PREFILL_QTILE):
                t64.append((i, q0, min(kvl[i], off + q0 + PREFILL_QTILE)))
        else:
            for q0 in range(0, n, EXTEND2_QTILE):
                t256.append((i, q0, min(kvl[i], off + q0 + EXTEND2_QTILE)))
    t64.sort(key=lambda t: -t[2])
    t256.sort(key=lambda t: -t[2])
    t64_t = torch.tensor([x[:2] for x in t64], dtype=torch.int32).reshape(-1, 2)

    # KV-split policy for the 256-row kernel: when the long portions' tiles x
    # heads cannot fill ~2 workgroups per CU, split the deepest tiles' key
    # ranges. Short portions are here to be split also beside enough others,
    # unless those walk as many keys. 28/4 heads: 2560 rows beside 65 at 6113 keys 156 us
    # (unsplit 364, in the 64-row kernel 530), beside 33 at 1000 keys 125 (117).
    def parts(tiles: int) -> int:
        # truly starved launches only (256 CUs, 1 block/CU kernel): the
        # partial slabs + combine cost ~2x slab traffic, so marginal
        # shortfalls are better left unsplit
        wgs = tiles * max(num_q_heads, 1)
        return min(8, -(-512 // wgs)) if 0 < wgs < 256 else 1

    long = [k for i, _, k in t256 if i not in deep]
    factor = parts(len(long))
    deep_factor = max(2, parts(len(t256) - len(long)))
    longest = max(long, default=0)
    rows, combine = [], []
    ws_rows = 0
    if factor > 1 or deep:
        split, plain = [], []
        for (i, q0, kmax) in t256:
            span = (kmax + E2_KVBLK - 1) // E2_KVBLK
            most = (deep_factor if i in deep and (factor > 1 or kmax > longest)
                    else factor)
            p = min(most, max(1, span // 4))
            (split if p > 1 else plain).append((i, q0, p))
        # cap the f32 partial workspace at ~512 MB
        slab = num_q_heads * EXTEND2_QTILE * 130 * 4
        if sum(p for _, _, p in split) * slab > 512 * 1024 * 1024:
            split, plain = [], split + plain
        for (i, q0, p) in split:
            combine.append((len(rows), p, i, q0))
            for part in range(p):
                rows.append((i, q0, part, p))
        ws_rows = len(rows)
        for (i, q0, p) in plain:
            rows.append((i, q0, 0, 1))
    else:
        rows = [(i, q0, 0, 1) for (i, q0, _) in t256]
    t256_t = torch.tensor(rows, dtype=torch.int32).reshape(-1, 4)
    ctab = torch.tensor(combine, dtype=torch.int32).reshape(-1, 4)

    drows = dseqs = None
    if dec:
        # the single q row of each decode seq sits at cu_seqlens_q[i]; seq-level
        # metadata indexes with `dec` itself. Rows side by side (a scheduler
        # puts running sequences together) are a slice, which needs no gather
        # and no scatter: two launches, 10 us a layer.
        cu = [0]
        for n in q_lens:
            cu.append(cu[-1] + n)
        at = [cu[i] for i in dec]
        drows = (slice(at[0], at[0] + len(at))
                 if at[-1] - at[0] == len(at) - 1
                 else torch.tensor(at, dtype=torch.long))
        dseqs = torch.tensor(dec, dtype=torch.long)
    t64_t, t256_t, ctab, drows, dseqs = upload(
        [t64_t, t256_t, ctab, drows, dseqs], device)
    return t64_t, t256_t, (drows, dseqs), ctab, ws_rows


def attention_extend_paged(
    q, k_cache, v_cache, block_tables, kv_lens, cu_seqlens_q,
    q_lens: list[int], scale: float, window: int = 0, tiles=None,
    sink: bool = False, native=None, maps: int = 1, sink_w=None, slopes=None,
    out=None, step_cache: dict | None = None,
):
    """Causal attention of packed NEW tokens over each sequence's full paged
    KV history (cached prefix + new tokens already written by
    reshape_and_cache). The prefix-caching / chunked-prefill attention path.
    q_lens is the host-side per-seq new-token count (tile grid without a
    D2H sync); kv_lens is the device int32 total kv length per seq.
    window > 0 = sliding-window attention. sink: every softmax also holds a
    value-less key of score 0. native: the extension whose build of these
    kernels runs (default: arks_amd_C). maps M > 1: a key row of the cache
    holds M keys side by side that share the row's value (k_cache [pages, G,
    16, M*D]); q has G*M groups of heads, group g*M + m reads key m of head
    g (tiles built without the flash-decode rows). sink_w, slopes [Hq] fp32:
    a sink's score per head, a distance bias slope[h] (i - j) off the scores
    (256-row tiles and single rows only: build_extend_tiles(min_ladder=1);
    the extension must be the layer-list models'). out: a contiguous
    [Tq, Hq, D] tensor to write. step_cache: a dict of the calls of one
    forward pass, which shares what they would each derive from the lengths
    and tables of the single rows.

    Dispatch: big chunks, and a few small ones behind a context, run the
    8-wave 32x32-MFMA ladder kernel (attn_extend2.hip, 256-row q tiles); other
    small chunks and fp8-KV runs use the 4-wave 64-row kernel."""
    if q.is_cuda:
        C = native if native is not None else _native()
        sink = 1 if sink else 0
        if out is None:
            out = torch.empty(
                (q.shape[0], q.shape[1], q.shape[2]), dtype=q.dtype,
                device=q.device)
        kv_fp8 = k_cache.dtype != torch.bfloat16
        t64, t256, (drows, dseqs), ctab, ws_rows = (
            tiles if tiles is not None
            else build_extend_tiles(q_lens, None, kv_fp8, q.device,
                                    num_q_heads=q.shape[1])
        )
        if t256.numel():
            if ws_rows:
                ws = _extend_ws(
                    ws_rows * q.shape[1] * EXTEND2_QTILE * (q.shape[2] + 2),
                    q.device,
                )
            else:
                ws = q.new_empty(0, dtype=torch.float32)
            C.attention_extend_paged2(
                out, q, k_cache, v_cache, block_tables, kv_lens, cu_seqlens_q,
                t256, ws, scale, window, sink, maps, sink_w, slopes,
            )
            if ctab.numel():
                C.attention_extend2_combine(
                    out, ws, ctab, cu_seqlens_q, scale, k_cache.shape[1] * maps,
                )
        if t64.numel():
            assert sink_w is None and slopes is None
            C.attention_extend_paged(
                out, q, k_cache, v_cache, block_tables, kv_lens, cu_seqlens_q,
                t64, scale, window, sink, maps,
            )
        if drows is not None:
            assert maps == 1, "single rows of a two-map cache: no flash-decode"
            dq = q[drows]
            biased = sink_w is not None or slopes is not None
            # attention_sink_paged takes contiguous rows, the other one gaps
            if (dq.stride()[1:] != (dq.shape[2], 1) or dq.stride(0) % 8
                    or dq.data_ptr() % 16
                    or (biased and not dq.is_contiguous())):
                dq = dq.clone(memory_format=torch.contiguous_format)
            dtab, dlens, plan = _single_rows(
                block_tables, kv_lens, dseqs, k_cache.shape[1], window, kv_fp8,
                not biased, C, step_cache)
            if biased:
                each = torch.arange(dq.shape[0] + 1, dtype=torch.int32,
                                    device=q.device)
                dout = attention_sink_paged(
                    dq, k_cache, v_cache, dtab, dlens, each, each[:-1], scale,
                    bool(sink), max_q_len=1, sink_w=sink_w, window=window,
                    slopes=slopes)
            else:
                dout = attention_decode_paged(
                    dq, k_cache, v_cache, dtab, dlens, scale, window=window,
                    sink=bool(sink), native=C, plan=plan,
                    out=out[drows] if isinstance(drows, slice) else None,
                )
                if isinstance(drows, slice):
                    return out
            out[drows] = dout
        return out
    return ref.attention_extend_paged(
        q, k_cache, v_cache, block_tables, kv_lens, cu_seqlens_q, scale,
        window,
    )


def _of_step(step_cache: dict, key, inputs: tuple, make):
    """What make() gives for these tensors: made once per forward pass
    (step_cache), and again for other ones or after they were written."""
    state = [0 if t.is_inference() else t._version for t in inputs]
    held = step_cache.get(key)
    if (held is None or held[1] != state
            or any(a is not b for a, b in zip(held[0], inputs))):
        held = step_cache[key] = (inputs, state, make())
    return held[2]


def _single_rows(block_tables, kv_lens, dseqs, num_kv_heads: int, window: int,
                 kv_fp8: bool, planned: bool, native,
                 step_cache: dict | None):
    """(block tables, lengths, decode plan) of the single rows of a mixed
    batch: shared by the layers of a forward pass (step_cache)."""
    cache = {} if step_cache is None else step_cache
    dtab, dlens = _of_step(
        cache, "single_rows", (block_tables, kv_lens, dseqs),
        lambda: (block_tables[dseqs].contiguous(), kv_lens[dseqs].contiguous()))
    plan = (step_decode_plan(dlens, num_kv_heads, window, kv_fp8, native, cache)
            if planned else None)
    return dtab, dlens, plan


def step_decode_plan(seq_lens, num_kv_heads: int, window: int, kv_fp8: bool,
                     native, step_cache: dict | None):
    """attention_decode_plan, shared by the layers of a forward pass
    (step_cache)."""
    if step_cache is None:
        return None
    return _of_step(
        step_cache, ("decode_plan", num_kv_heads, window, kv_fp8), (seq_lens,),
        lambda: attention_decode_plan(seq_lens, num_kv_heads, window, kv_fp8,
                                      native=native))


def decode_waves(num_seqs: int, num_kv_heads: int, kv_fp8: bool = False,
                 num_partitions: int | None = None) -> int:
    """Runs per key/value head that the decode kernel cuts all sequences'
    pages into (attn_decode.hip). One workgroup of 4 waves per CU, two where the
    rows are half as long (fp8) or where there are more sequences than runs, so
    that a run would hold several short ones. us, kernel and merge, one workgroup
    per CU (two), lengths even over the logarithm unless said:
    - up to 1024 (sequence, head) pairs: 28/4 heads x 128: 64 of 1024 30.5 (31.2),
      200 of 20..4000 60.8 (63.9), 256 of 100 17.0 (20.0); 14/2 x 64: 128 of
      20..4000 18.4 (20.5), 256 of 1..4000, even, 52.0 (52.4); 32/8 x 64: 100 of
      20..4000 36.1 (34.2), 128 of 100 11.3 (12.7);
    - more of them: 32/8 x 128: 256 of 100 31.1 (27.5), 256 of 20..4000 141.5
      (145.9); 32/8 x 64: 200 of 20..4000 62.1 (59.7), 256 of 20..500 24.6 (21.8);
      16/16 x 64: 256 of 100 33.1 (27.3);
    - fp8, 28/4 x 128: 200 of 20..4000 45.9 (42.9), 256 of 1..4000, even, 121.5
      (108.1).
    Counts between are 6 to 25 % slower. num_partitions: that many runs per
    sequence on average instead."""
    if num_partitions is not None:
        return max(1, num_partitions * num_seqs)
    many = kv_fp8 or num_seqs * num_kv_heads > 1024
    waves = 2048 if many else 1024
    return max(1, waves // num_kv_heads)


def attention_decode_plan(seq_lens, num_kv_heads: int, window: int = 0,
                          kv_fp8: bool = False,
                          num_partitions: int | None = None, native=None):
    """What every wave of attention_decode_paged reads, for layers of this
    window, number of key/value heads and kind of pages: made once per step
    and handed to each of them (plan=). None on CPU tensors."""
    if not seq_lens.is_cuda:
        return None
    C = native if native is not None else _native()
    waves = decode_waves(seq_lens.shape[0], num_kv_heads, kv_fp8,
                         num_partitions)
    plan = torch.empty(4 * waves + 2 * seq_lens.shape[0], dtype=torch.int32,
                       device=seq_lens.device)
    C.attention_decode_plan(plan, seq_lens, waves, window)
    return plan


def attention_decode_paged(
    q, k_cache, v_cache, block_tables, seq_lens, scale: float,
    num_partitions: int | None = None, part_out=None, window: int = 0,
    sink: bool = False, native=None, plan=None, out=None,
):
    """plan: attention_decode_plan's for these lengths, heads, window and
    num_partitions (None: made here). out: a contiguous tensor to write."""
    if q.is_cuda:
        C = native if native is not None else _native()
        S, hq, hd = q.shape
        hkv = k_cache.shape[1]
        if out is None:
            out = torch.empty((S, hq, hd), dtype=q.dtype, device=q.device)
        kv_fp8 = k_cache.dtype != torch.bfloat16
        if plan is None:
            plan = attention_decode_plan(seq_lens, hkv, window, kv_fp8,
                                         num_partitions, C)
        waves = decode_waves(S, hkv, kv_fp8, num_partitions)
        need = (waves + S) * (hq * hd + 16 * hkv)
        if part_out is None or part_out.numel() < need:
            part_out = torch.empty(need, dtype=torch.float32, device=q.device)
        C.attention_decode_paged(
            out, q, k_cache, v_cache, block_tables, seq_lens, scale,
            part_out, plan, waves, window, 1 if sink else 0,
        )
        return out
    return ref.attention_decode_paged(
        q, k_cache, v_cache, block_tables, seq_lens, scale, window
    )


_EXTEND_WS: dict = {}


def _extend_ws(need: int, device):
    key = (device.index,)
    ws = _EXTEND_WS.get(key)
    if ws is None or ws.numel() < need:
        ws = torch.empty(need, dtype=torch.float32, device=device)
        _EXTEND_WS[key] = ws
    return ws


def skinny_gemm(x, weight, bias=None):
    """x weight^T (+ bias) for decode-sized M (<= 64) with K split over
    workgroups where it can be (stream_gemm.hip; fixed order of the sums, no
    atomics)."""
    M, K = x.shape
    if K % 64 or weight.shape[0] % 4:
        return _stream_gemm(x, weight, bias)
    return parts_sum(Parts(_stream_parts(x, weight), bias))


# 0: products take the library's kernels (up to 256 rows, and gate and up
# products of any number), experts the kernels of moe_gemm.hip without the
# engine: for comparisons
_USE_SKINNY = os.environ.get("ARKS_SKINNY_GEMM", "1") == "1"
# weights up to this many elements take the framework's kernels at any number
# of rows up to 64, larger ones where the rules below say so
_SKINNY_MAX_ELEMS = 34_000_000


# weights of two products that go in one launch, together
_PAIR_ELEMS = 100_000_000


def _rows_16b(x):
    """x, or a copy whose rows start on 16 bytes."""
    if x.stride(-1) == 1 and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0:
        return x
    return x.clone(memory_format=torch.contiguous_format)


def _stream_split(M: int, N: int):
    """(row tiles, groups of 16 weight rows, waves) of a streamed product
    (stream_gemm.hip). Up to 256 groups of weight rows one per workgroup, so
    that most CUs have one, and up to 512 two: 3584 x 3584, 8 rows, us: 8.4
    (two 11.6); 4608 x 3584: 11.9 (13.0). Waves that split K help while few
    rows of x come with each weight. Beyond, one group of 4 waves for up to 4
    rows (28672 x 4096, 4 rows: 47.7, two groups of 16 waves 51.7), two for
    more (16384 x 4096, 8 rows: 30.1, one group 31.4)."""
    mt = 1 if M <= 16 else 2
    tiles = -(-N // 16)
    if tiles <= 256:
        return mt, 1, 16 if M <= 8 else 4
    if tiles <= 512 or M > 16:
        return mt, 2, 16
    if tiles > 2048:
        return mt, 2, 8
    return (mt, 1, 4) if M <= 4 else (mt, 2, 16)


def _plain(*tensors) -> bool:
    """Whether kernels may take these past autograd: no gradient, tangent or
    transform (vmap) of theirs is followed."""
    if torch.autograd.forward_ad._current_level >= 0:
        return False
    grad = torch.is_grad_enabled()
    return not any(
        type(t) not in (torch.Tensor, torch.nn.Parameter)
        or torch._C._functorch.is_functorch_wrapped_tensor(t)
        or (grad and t.requires_grad) for t in tensors if t is not None)


def _few_rows(x, weight, bias=None) -> bool:
    """Whether the kernels of stream_gemm.hip can take x weight^T (+ bias)."""
    return (_USE_SKINNY and x.is_cuda and x.dim() == 2
            and 1 <= x.shape[0] <= 64
            and x.dtype == weight.dtype == torch.bfloat16
            and weight.shape[1] % 32 == 0
            and _plain(x, weight, bias)
            and weight.is_contiguous() and weight.data_ptr() % 16 == 0
            and (bias is None or (bias.dtype == x.dtype
                                  and bias.is_contiguous()))
            and native_available())


def _streams(x, weight, silu: bool = False, bias=None) -> bool:
    """Whether x weight^T takes stream_gemm (larger weights: if _mid does not
    take them)."""
    return (_few_rows(x, weight, bias)
            and _stream_sizes(x.shape[0], *weight.shape, silu))


def _stream_sizes(M: int, N: int, K: int, silu: bool = False) -> bool:
    """_streams, by the sizes. A workgroup reads all of x's rows beside its 16
    or 32 weight rows, so the line lies where that traffic (rows x K), and the
    waves' tails, meet what the other path loses: us, here (other), the other being the split product with its sums up to
    _SKINNY_MAX_ELEMS and the library beyond. 3584 x 3584: 1 row 7.4 (10.9),
    16 rows 9.5 (11.3), 32 rows 12.5 (13.0). 5120 x 2048, 32 rows 10.4 (12.4);
    6144 x 4096, 32 rows 20.1 (17.7); 544 x 8192, 8 rows 13.8 (10.4). Library:
    18432 x 4096, 16 rows 42.6 (80.1); 32000 x 4096, 8 rows 54.5 (67.4), 16
    rows 62.0 (62.5); 151936 x 2048, 16 rows 134 (206), 32 rows 167 (149);
    37888 x 3584, 1 row 52.9 (53.2), 8 rows 58.7 (53.1), with the activation
    57.8 (59); 3584 x 18944, 1 row 30.3 (32.5), 4 rows 33.4 (32.6)."""
    if M > 64 or K % 32:
        return False
    if N * K <= _SKINNY_MAX_ELEMS:
        return M * K <= 98304 and (K <= 4096 or N >= 2048) or K % 64 != 0
    if M <= 2 or (silu and M <= 8 and K <= 4096):
        return True
    return M <= 16 and (K <= 2048 or (K <= 4096 and N * K <= 1 << 27))


def _splits(x, weight, bias=None) -> bool:
    """Whether x weight^T splits K over workgroups of stream_gemm.hip (asked
    after _mid, which takes N % 8 == 0, and _streams): weights up to
    _SKINNY_MAX_ELEMS, and larger ones that are tall. us with the sums
    (library): 3584 x 18944, 4 rows 30.7 (32.6), 32 rows 31.7 (43.9), 64 rows
    36.8 (49.6); 8192 x 28672, 8 rows 88.5 (91.8), 64 rows 108 (154); wide
    ones, as 16384 x 4096 at 32 rows, 36 (34)."""
    N, K = weight.shape
    return (_few_rows(x, weight, bias) and K % 64 == 0 and N % 4 == 0
            and (N * K <= _SKINNY_MAX_ELEMS or K >= 2 * N))


def _mid_cut(M: int, N: int, K: int, silu: bool, summed: bool,
             whole: bool = False):
    """(qt, splits) of a mid_gemm: weight rows of a tile (32 * qt) and runs
    of K that finish first, by a fit of what 52 sizes took at 1 to 256 rows with
    all of their cuts (the chosen ones are 0.7 % from the best on average): a
    step of 64 columns takes what its loads and matrix operations do, or the
    weights' stream where all CUs share it; the fp32 sums of the runs are written
    and read at 5 TB/s, and added by a launch of their own unless the consumer
    does (summed). At most 8 runs, as the consumer's time grows with them. Beyond
    64 rows a run is one chain of sums, whose error grows with it: where K is cut,
    of the cuts within 4 % of the least time the one with the most runs (error
    against 64 bits and us, so, and with the least time by the fit: 2048 x 2048, 96
    rows, 1.02e-7 in 8 runs, 11.3, and 1.32e-7 in 4, 10.8; 5120 x 27648 3.64e-7 in
    8, 58.8, and 4.24e-7 in 6, 59.7; 288 sizes and numbers of rows take 1.0009 of
    the time).
    whole: one run."""
    steps, groups = K // 64, -(-M // 32)
    cuts = []
    for qt in (4, 5, 2):
        tiles = -(-N // ((16 if silu else 32) * qt))
        most = 1 if silu or whole or tiles > 256 else min(8, steps)
        for splits in range(1, most + 1):
            rounds, last = divmod(tiles * splits, 256)
            alone = 0.02 + 0.095 * qt + 0.06 * groups
            run = -(-steps // splits)
            us = rounds * (0.6 + run * max(alone, 0.15 * qt))
            if last:
                us += 0.6 + run * max(alone, 0.15 * qt * last / 256)
            if splits > 1:
                us += splits * (0.1 + M * N * 1.6e-6) + (0.0 if summed else 4.0)
            cuts.append((us, qt, splits))
    best = min(cuts, key=lambda c: c[0])
    if M > 64 and best[2] > 1:
        best = min((c for c in cuts if c[0] <= 1.04 * best[0]),
                   key=lambda c: (-c[2], c[0]))
    return best[1:]


def _mid_takes(x, weight, bias=None) -> bool:
    """Whether mid_gemm can take these tensors, at sizes that it has."""
    return (_USE_SKINNY and x.is_cuda and x.dim() == 2
            and 1 <= x.shape[0] <= 256
            and x.dtype == weight.dtype == torch.bfloat16
            and _plain(x, weight, bias)
            and x.stride(0) < 1 << 22
            and weight.is_contiguous() and weight.data_ptr() % 16 == 0
            and (bias is None or (bias.dtype == x.dtype
                                  and bias.shape == weight.shape[:1]
                                  and bias.is_contiguous()))
            and native_available())


def _mid(x, weight, bias=None, silu: bool = False, summed: bool = False):
    """(qt, splits) if x weight^T (or silu(gate) * up of it) takes mid_gemm,
    else None. summed: the consumer adds the sums of splits. It takes up to 256
    rows, but for what the streamed product (few rows of small weights, which
    has no sums to add) or the library does as fast (_mid_sizes). us, here
    (other): 37888 x 3584 with the activation, 1 row 44.6 (48.1), 32 rows 45.1
    (57.6), 128 rows 53.1 (71.2), 200 rows 59.8 (85); 152064 x 3584, 1 row 168
    (182), 64 rows 188 (209), 200 rows 247 (325); 3584 x 18944 with a launch for
    the sums, 1 row 26.3 (27.4), 100 rows 36.1 (96.5)."""
    if not _mid_takes(x, weight, bias):
        return None
    N, K = weight.shape
    return _mid_sizes(x.shape[0], N // 2 if silu else N, K, silu, summed)


@functools.lru_cache(maxsize=4096)
def _mid_sizes(M: int, N: int, K: int, silu: bool, summed: bool):
    """_mid, by the sizes (N columns of the result). The others' side of the
    lines, us, here (other), sums with their consumer:
    - streamed, which has no sums to add: 1536 x 1536, 1 row 7.9 (7.3); 4096 x
      4096, 4 rows 11.7 (11.2); 3584 x 3584, 1 row the same, 8 rows 0.89 of it;
      5120 x 2048, 8 rows 0.88; without a consumer 4096 x 4096, 8 rows 1.18, 32
      rows 0.82, 8192 x 2048, 16 rows 1.11, 48 rows 0.71; with the activation
      1920 x 1088 (60 tiles), 5 rows 6.0 (5.6), 4096 x 5120 (half of the CUs)
      the same;
    - library, sums: 4096 x 2048, 208 rows 1.13 of it; 193 to 224 rows of
      3072..3840 x 3072..4096 0.55 to 1.00 (3584 x 3584, 224 rows 22.4 (23.7)), 256
      rows 0.87 to 1.03, 4096 x 3072, 193 to 224 rows 1.02 to 1.03; 1152 x 896, 208
      rows 1.07; without a consumer 8192 x 2048, 96 rows 1.07, 208 rows 1.29, 64 rows
      0.85, 4096 x 4096, 208 rows 1.02, 2192 x 896 (35 tiles), 100 rows 9.4 (8.3);
      with the activation 2256 x 2048 (71 tiles), 250 rows 24.5 (19.4);
    - library, whole: 50304 x 2560, whose tiles fill the second round of CUs by
      a quarter, 96 rows 1.15, 64 rows 1.04; 55296 x 5120, 0.84 full, 160 to 224
      rows 1.10 to 1.14, 50304 x 4096, 0.77 full, 1.06 to 1.10, 128 rows 0.96, 102400
      x 4096, three rounds 0.83 full, 0.90 to 0.94; gate and up 55296 x 5120, 0.84 full,
      96 rows 1.06, 57344 x 8192, 0.875 full, 0.86."""
    if (K % 64 or N % 8 or not 64 <= K < 1 << 22 or not 0 < N < 1 << 24
            or (silu and 2 * N * K >= 1 << 31)):
        return None
    small = N * K <= _SKINNY_MAX_ELEMS
    qt, splits = _mid_cut(M, N, K, silu, summed)
    tiles = -(-N // ((16 if silu else 32) * qt))
    fill = tiles * splits / (256 * -(-tiles * splits // 256))
    if summed:
        if small and (M * K <= 32768 and (
                          1024 < K <= 2048 or (K <= 4096 and 3072 <= N <= 4096))
                      or M * K <= 24576 and 1024 < K <= 3072
                      or K <= 1024 and M <= (64 if N <= 8192 else 8)):
            return None
        if N * K < 13_000_000 and K <= 4096 and M > (
                128 if K <= 1024 or (K <= 2048 and M % 32)
                else 224 if K >= 3072 and 3072 <= N < 4096 else 192):
            return None
    elif silu:
        if (fill < 0.6 and K >= 4096 and M <= 64
                or fill < 0.3 and (M <= 32 or M > 192)
                or qt == 2 and fill > 0.9 and M <= 8 and K <= 4096
                or N * K > 1 << 27 and fill < 0.86 and 64 < M <= 160
                or N * K > 1 << 27 and fill < 0.9 and M > 128 and K >= 8192):
            return None
    else:
        few = splits > 1 or fill <= 0.5
        # (the streamed product takes K beyond 4096 from 2048 columns on; below,
        # its splits are slower: 896 x 4864, 4 rows 7.3 us here, 8.5, 1536 x 8192
        # 9.2 and 11.8)
        if (small and few and N <= 8192 and _stream_sizes(M, N, K)
                and M <= (16 if K <= 256 and N > 2048 else 64)
                and (K <= 1536 or M * K <= (65536 if N > 2048 else 32768))):
            return None
        if few and M > 64 and (
                K <= 1024 or (M > 160 and N * K < 16_000_000)
                or (N > 2048 and (K <= 2048 or N * K < 16_000_000))
                or (splits > 1 and M > 96 and K <= 3072)):
            return None
        if M > 192 and M % 32 and 2048 < K <= 4096 and N * K <= 1 << 26:
            return None
        if splits == 1 and tiles > 256 and (
                (fill < 0.8 and M > 64 and (
                    K <= 1024 or (K <= 2048 and M > 192) or 2048 < K <= 3072))
                or (M > 128 and (K >= 8192 or (
                    tiles <= 512 and fill < 0.9 and N * K > 1 << 27)))):
            return None
    return qt, splits


def _mid_gemm(x, weight, bias, cut, silu: bool = False, summed: bool = False):
    """A product by mid_gemm: a tensor, or Parts where K is split or the
    consumer adds sums (summed; one run of K then reaches it in fp32 too)."""
    (qt, splits), M = cut, x.shape[0]
    N = weight.shape[0] // (2 if silu else 1)
    if splits > 1 or summed:
        sums = torch.empty((splits, M, N), dtype=torch.float32, device=x.device)
        _native().mid_gemm(sums, _rows_16b(x), weight, None, qt, False)
        return Parts(sums, bias)
    out = torch.empty((M, N), dtype=x.dtype, device=x.device)
    _native().mid_gemm(out, _rows_16b(x), weight, bias, qt, silu)
    return out


class Parts:
    """A product whose sums over runs of K are not added yet: sums [splits,
    M, N] fp32, and a bias [N] that belongs to their sum."""

    def __init__(self, sums, bias=None):
        self.sums, self.bias = sums, bias

    def columns(self, first: int, end: int):
        """Those of columns [first, end)."""
        return Parts(self.sums[:, :, first:end],
                     None if self.bias is None else self.bias[first:end])


class Mixed:
    """Experts' rows y [pairs, H] that are not mixed yet: row t of the result
    is the sum over j of weights[t, j] * y[rows[t, j]]."""

    def __init__(self, y, weights, rows):
        self.y, self.weights, self.rows = y, weights, rows


def _stream_parts(x, weight):
    """Split sums; as many splits as give every CU a workgroup of 128 weight
    rows (3584 x 3584, 64 rows, us without the sums: 4 splits 14.9, 8 11.4, 12
    13.2), at most 16 and, where many rows make the sums long, 8."""
    M, (N, K) = x.shape[0], weight.shape
    splits = max(1, min(256 // -(-N // 128), 16 if M <= 32 else 8,
                        K // (128 if K % 128 == 0 else 64)))
    sums = torch.empty((splits, M, N), dtype=torch.float32, device=x.device)
    _native().stream_split(sums, _rows_16b(x), weight)
    return sums


def parts_sum(x):
    """The bf16 tensor that x, a Parts, a Mixed or already a tensor, stands
    for."""
    if isinstance(x, Mixed):
        return moe_mix_rows(x.y, x.weights, x.rows)
    if not isinstance(x, Parts):
        return x
    out = torch.empty(x.sums.shape[1:], dtype=torch.bfloat16,
                      device=x.sums.device)
    _native().stream_sum(out, x.sums.contiguous(), x.bias)
    return out


def _stream_gemm(x, weight, bias=None, dtype=None, silu: bool = False):
    M, N = x.shape[0], weight.shape[0] // (2 if silu else 1)
    out = torch.empty((M, N), dtype=dtype or x.dtype, device=x.device)
    mt, nf, wv = _stream_split(M, weight.shape[0])
    if silu:  # a group of gate rows with their up rows
        nf, wv = 2, 16 if weight.shape[0] <= 8192 else 8
    _native().stream_gemm(out, _rows_16b(x), weight, bias, mt, nf, wv, silu)
    return out


# Tiles of wide_gemm.hip (rows of a x rows of w): us of a step of 64 columns
# where all CUs are busy. Other combinations of 128, 192, 256 and 320 give less
# than 0.1 % over 1500 sizes.
_WIDE_STEP = {(128, 256): 0.92, (192, 256): 1.16, (256, 128): 0.89,
              (256, 192): 1.11, (256, 256): 1.33, (256, 320): 1.59,
              (320, 128): 1.03, (320, 256): 1.56}


@functools.lru_cache(maxsize=4096)
def _wide_fit(M: int, N: int, K: int, split: bool, summed: bool):
    """(us, rows of a, rows of w, runs of K, workgroups) of a wide_gemm, w [N, K]:
    the tiles and runs that finish first by a fit of what 15 sizes took at 257 to
    8192 rows with every tile and cut (the chosen ones are 0.7 % from the best on
    average). A round over the CUs takes its steps and the end of a tile; the
    last, when fewer CUs run, somewhat less. fp32 sums are written (0.12 us / MB)
    and read again (0.15), by a launch of their own unless the consumer adds them
    (summed). split: K may be cut."""
    best, steps = None, K // 64
    for (tm, tw), step in _WIDE_STEP.items():
        tiles = -(-M // tm) * -(-N // tw)
        for splits in range(1, max(1, min(16, steps // 4) if split else 1) + 1):
            jobs = tiles * splits
            if splits > 1 and splits * M * N > 1 << 25:
                break  # 128 MB of sums
            most = max(jobs * (x + 1) // 8 - jobs * x // 8 for x in range(8))
            rounds, last = -(-most // 32), ((most - 1) % 32 + 1) / 32
            one = -(-steps // splits) * step + 6.0 * tm * tw / 65536
            us = 3.2 + one * (rounds - 0.22 * (1.0 - last))
            if splits > 1:
                us += splits * M * N * 1.08e-6 + (0.0 if summed else 4.0)
            if best is None or us < best[0]:
                best = us, tm, tw, splits, jobs
    return best


def _wide_cut(M: int, N: int, K: int, split: bool, summed: bool):
    """_wide_fit without its time."""
    return _wide_fit(M, N, K, split, summed)[1:]


def _wide_takes(x, weight, bias=None) -> bool:
    """Whether wide_gemm can take these tensors, of more rows than mid_gemm."""
    return (_USE_SKINNY and x.is_cuda and x.dim() == 2
            and not getattr(weight, "plain_prompts", False)
            and 256 < x.shape[0] < 1 << 24
            and x.dtype == weight.dtype == torch.bfloat16
            and weight.shape[1] % 64 == 0 and weight.shape[0] % 16 == 0
            and 64 <= weight.shape[1] < 1 << 22
            and 0 < weight.shape[0] < 1 << 24
            and x.stride(0) < 1 << 22 and _plain(x, weight, bias)
            and weight.is_contiguous() and weight.data_ptr() % 16 == 0
            and (bias is None or (bias.dtype == x.dtype
                                  and bias.shape == weight.shape[:1]
                                  and bias.is_contiguous()))
            and native_available())


def _wide(x, weight, bias=None, summed: bool = False):
    """(rows of a, rows of w, runs of K) if x weight^T takes wide_gemm, else
    None: more than 256 rows of long weights, where that is expected to finish in
    front of the library. At its best a library kernel of 256 x 256 tiles does a step
    of 64 columns in 1.06 us in whole rounds over the CUs, here it is 1.33: so the
    library keeps what fills its rounds, and sums that have a launch of their own
    (not summed) count 2e-6 us each beyond the fit. Of a few hundred rows it often
    has slower kernels, which turn with the row count. us in front of a norm
    (library), 3584 x 18944: 300 rows 64 (108), 450 rows 77 (207), 700 rows 101 (176),
    1309 rows 175 (267), 2314 rows 275 (499), 4666 rows 479 (908), left to it 3344 rows
    412 (357), 8192 rows 873 (807); 4096 x 14336: 300 rows 57 (84), 1536 rows 174
    (188), left 3344 rows 336 (314); 4096 x 8192: 300 rows 42 (53), 5000 rows 268 (295),
    left 3344 rows 214 (194). Over 18 weights of 13 to 235 million
    elements (N 1024 to 12288, K 8192 to 28672) at 37 numbers of rows 0.825 of the
    library's time, the better of the two 0.804, 11 sizes more than 3 % slower, the
    worst 1.12 (3072 x 24576, 3344 rows); with a launch for the sums 0.840 (0.816), 25
    and 1.12. With K up to 4096 a run has few steps: 4096 x 4096, 491 rows 32 (30),
    1159 rows 51 (44)."""
    if not _wide_takes(x, weight, bias):
        return None
    M, (N, K) = x.shape[0], weight.shape
    if K < 8192 or N < 1024:
        return None
    us, *cut, _ = _wide_fit(M, N, K, True, summed)
    if cut[2] > 1 and not summed:
        us += 2e-6 * cut[2] * M * N
    rounds = -(-(-(-M // 256) * -(-N // 256)) // 256)
    return cut if us < 3.0 + rounds * (5.0 + 1.06 * K / 64) else None


def _wide_silu(x, weight):
    """(rows of a, rows of w) if silu_mul(x weight^T) takes wide_gemm, the
    activation inside, else None: more than 256 rows, where at least half of the
    CUs get a tile (fewer: 4096 x 2048, 600 rows 31 us, library and activation
    23). us, here (library and activation; tiles of 256 alone): 37888 x 3584, 300
    rows 97 (121; 131), 400 rows 104 (144; 157), 600 rows 154 (168; 162), 1000
    rows 194 (316; 236), 2048 rows 384 (416; 396), 3150 rows 607 (809; 677), 8192
    rows 1520 (1663; 1599); 28672 x 4096, 600 rows 109 (136; 151); 12288 x 2048,
    1280 rows 50 (61; 60). Tiles of 256 alone have the shorter loop, and keep what fills
    0.98 of their rounds: 28672 x 4096, 4096 rows 713 (tiles of 256 670), 8192 rows 1381
    (1303); 55296 x 5120, 8192 rows 3290 (3142); 36864 x 6144, 8192 rows 2602 (2502)."""
    if not _wide_takes(x, weight):
        return None
    N, K = weight.shape
    if x.shape[0] > 512 and _tile_fill(x.shape[0], N // 2) >= 0.98:
        return None
    if (N // 2 + 320) * K >= 1 << 31:  # a tile's rows lie 4 GiB apart
        return None
    tm, tw, _, jobs = _wide_cut(x.shape[0], N, K, False, False)
    return (tm, tw) if jobs >= 128 else None


def _wide_gemm(x, weight, bias, cut, summed: bool = False):
    """A product by wide_gemm: a tensor, or Parts where K is cut or the consumer
    adds sums (summed)."""
    (tm, tw, splits), M, N = cut, x.shape[0], weight.shape[0]
    if splits > 1:
        sums = torch.empty((splits, M, N), dtype=torch.float32, device=x.device)
        _native().wide_gemm(sums, _rows_16b(x), weight, None, tm, tw, False)
        parts = Parts(sums, bias)
        return parts if summed else parts_sum(parts)
    out = torch.empty((M, N), dtype=x.dtype, device=x.device)
    _native().wide_gemm(out, _rows_16b(x), weight, bias, tm, tw, False)
    return out


def plain_prompts(weights) -> None:
    """Products of more than 256 rows of these weights stay out of wide_gemm, and those
    of prompts are rounded to bf16 in front of a norm, as without one that adds sums: the
    weights of a model whose pages are e4m3. A value next to a border between two of
    its values goes to the other side with the last bit of a sum, a step of 1/8 of it,
    and the rows that follow read it from its page: two orders of the same sums, 8
    layers of 3584 columns deep, give logits 0.015 to 0.022 of their norm apart (with
    bf16 pages 0.012). Neither is nearer to 64 bits: prompts of 400 rows, of 3 x 300 to
    700 and of 2 x 900 to 1500 are 0.0355, 0.0352 and 0.0234 off so, 0.0365, 0.0338 and
    0.0228 without; this one is kept for the answers that such a server gave before.
    Not covered are experts: their rows go to the engine as beside bf16 pages (4 layers
    of 128 experts: 0.013 to 0.016 from what items gave, 0.033 to 0.054 off 64 bits
    either way)."""
    for w in weights:
        w.plain_prompts = True


def linear_parts(x, weight, bias=None, own_cut: bool = True):
    """linear_bf16 for a consumer that takes Parts. own_cut: up to 256 rows K is
    cut with that in mind; else as linear_bf16 does, so that a prompt's rows have
    the order of sums that they have without a consumer."""
    if not own_cut and getattr(weight, "plain_prompts", False):
        return linear_bf16(x, weight, bias)
    cut = _mid(x, weight, bias, summed=own_cut)
    if cut is not None:
        return _mid_gemm(x, weight, bias, cut, summed=own_cut or cut[1] > 1)
    if own_cut and (x.dim() == 2 and not _streams(x, weight, bias=bias)
                    and _splits(x, weight, bias)):
        return Parts(_stream_parts(x, weight), bias)
    cut = _wide(x, weight, bias, summed=True)
    if cut is not None:
        return _wide_gemm(x, weight, bias, cut, summed=True)
    return linear_bf16(x, weight, bias)


@functools.lru_cache(maxsize=1024)
def _pair_cut(M: int, N: int, K: int, K2: int):
    """(qt, runs of K, runs of K2) of a pair of products of N columns, by the fit
    of _mid_cut: a workgroup's time is that of the longest run, and the sums of all
    runs are written and read. At most 8 runs of each."""
    steps, groups = (K // 64, K2 // 64), -(-M // 32)
    best = None
    for qt in (4, 5, 2):
        tiles = -(-N // (32 * qt))
        alone = 0.02 + 0.095 * qt + 0.06 * groups
        for run in range(1, max(steps) + 1):
            splits = [-(-s // run) for s in steps]
            if max(splits) > 8:
                continue
            rounds, last = divmod(tiles * sum(splits), 256)
            us = rounds * (0.6 + run * max(alone, 0.15 * qt))
            if last:
                us += 0.6 + run * max(alone, 0.15 * qt * last / 256)
            us += sum(splits) * (0.1 + M * N * 1.6e-6)
            if best is None or us < best[0]:
                best = us, qt, splits
    return best[1], *best[2]


def linear_pair(x, weight, x2, weight2):
    """(x weight^T, x2 weight2^T), both Parts, or None: one launch for up to 64
    rows of two products of as many columns, as long as the start and the end of a
    launch weigh beside the weights' stream (up to _PAIR_ELEMS). us with the norm
    behind both, cold weights (linear_parts of each; linear_bf16): 4096 x 4096 twice,
    1 row 18.3 (20.4; 20.7), 8 rows 18.7 (22.9; 22.8), 64 rows 21.4 (27.0; 31.6);
    4096 x (8192 and 4096), 8 rows 23.9 (27.9; 30.3); 1024 x 1024, 8 rows 8.6 (11.1;
    11.2); 5120 x 5120 27.1 (30.0; 40.6); 8192 x 8192 56.8 (57.3; 60.0), 6144 x (12288
    and 6144) 49.0 (49.0; 51.2)."""
    if (x.dim() == x2.dim() == 2 and 1 <= x.shape[0] == x2.shape[0] <= 64
            and weight.shape[0] == weight2.shape[0] and weight.shape[0] % 8 == 0
            and weight.shape[1] % 64 == weight2.shape[1] % 64 == 0
            and 1024 <= min(weight.shape[1], weight2.shape[1])
            and weight.numel() + weight2.numel() <= _PAIR_ELEMS
            and _mid_takes(x, weight) and _mid_takes(x2, weight2)):
        M, N = x.shape[0], weight.shape[0]
        qt, n, n2 = _pair_cut(M, N, weight.shape[1], weight2.shape[1])
        sums = torch.empty((n + n2, M, N), dtype=torch.float32, device=x.device)
        _native().mid_pair(sums, _rows_16b(x), weight, _rows_16b(x2), weight2, qt,
                           n)
        return Parts(sums[:n]), Parts(sums[n:])
    return None


def linear_bf16(x, weight, bias=None):
    """Linear dispatch: the streamed product for few rows of small weights, the
    tiles of mid_gemm.hip for up to 256 rows, K split over workgroups for sizes
    that those do not take, the tiles of wide_gemm.hip for more rows of long weights
    (_wide), hipBLASLt (F.linear) otherwise."""
    cut = _mid(x, weight, bias)
    if cut is not None:
        return parts_sum(_mid_gemm(x, weight, bias, cut))
    if x.dim() == 2 and _streams(x, weight, bias=bias):
        return _stream_gemm(x, weight, bias)
    if x.dim() == 2 and _splits(x, weight, bias):
        return parts_sum(Parts(_stream_parts(x, weight), bias))
    cut = _wide(x, weight, bias)
    if cut is not None:
        return _wide_gemm(x, weight, bias, cut)
    import torch.nn.functional as F

    return F.linear(x, weight, bias)


def _fixed_run(M: int, N: int, K: int) -> int:
    """Columns of K that one sum of a fixed product takes (0: a library
    product): 512 sums of 64 weight rows in all, of at least 256 columns;
    beyond 48 rows 448 where K > N, which takes tall weights too."""
    if N % 64 or K % 32:
        return 0
    tiles, tall = N // 64, K > N and M > 48
    if N * K > (80_000_000 if tall else _SKINNY_MAX_ELEMS):
        return 0
    if tall and tiles < 128:
        splits = -(-448 // tiles)
    else:
        splits = 1 if tiles >= 384 else -(-512 // tiles)
    splits = min(splits, -(-K // 256))
    return -(-(-(-K // splits)) // 32) * 32


def fix_sums(weights) -> None:
    """Has linear_fixed take the products of these parameters."""
    for w in weights:
        w.fixed_sums = True


def sums_fixed(M: int, *weights) -> bool:
    """Whether linear_fixed adds any of these weights up in runs of _fixed_run at M
    rows (up to 64). Larger weights, whose order there is that of _fixed_cut, do not
    count: where routed_experts takes them, up to 16 rows, theirs is its own."""
    return any(_fixed_run(M, *w.shape) for w in weights)


@functools.lru_cache(maxsize=1024)
def _fixed_cut(N: int, K: int, f32: bool):
    """(qt, splits) of a fixed product of more than _SKINNY_MAX_ELEMS weights
    (f32: with an fp32 result, one run), or None: mid_gemm's sums of up to 64 rows
    are the same for a cut, as long as tiles begin at the same steps (K up to 16384,
    arks_mid_gemm), and the cut is that of 16 rows at any number of them. us, 1 to
    16 rows (library): 12608 x 4096 18.5 (26), 16640 x 4096 27 (67), 10240 x 5120
    21.5 (24), 20480 x 2560 23.5 (48), 114688 x 4096 148 (160 to 198); in fp32 32000
    x 4096 45 (59), 64 rows 46 (51)."""
    if (N * K <= _SKINNY_MAX_ELEMS or K % 64 or N % 8
            or not 2048 <= K <= 16384 or N >= 1 << 24):
        return None
    return _mid_cut(16, N, K, False, False, whole=f32)


def _fixed_mid(x, weight, bias=None, f32: bool = False):
    """The cut, if x weight^T takes a fixed product of mid_gemm: up to 64 rows, with
    K below 4096 32 (50304 x 2560, 48 rows 57 us, library 53)."""
    N, K = weight.shape
    if not _mid_takes(x, weight, bias) or x.shape[0] > (64 if K >= 4096 else 32):
        return None
    return _fixed_cut(N, K, f32)


def linear_fixed(x, weight, bias=None):
    """x weight^T (+ bias) whose order of sums follows from the weight alone up
    to 48 rows (large weights with K below 4096: 32), for models that choose
    experts. Near a tie between two of them the last bits of a row decide, and with
    the expert its logits move (up to 0.2 of their norm in 3 layers of 16 experts):
    the choice must not turn with the number of rows that share a step. linear_bf16
    picks its kernel, and so the order, by the rows."""
    M, (N, K) = x.shape[0], weight.shape
    per = _fixed_run(M, N, K) if _few_rows(x, weight, bias) else 0
    if per:
        sums = torch.empty((-(-K // per), M, N), dtype=torch.float32,
                           device=x.device)
        _native().stream_split(sums, _rows_16b(x), weight, per)
        return parts_sum(Parts(sums, bias))
    cut = _fixed_mid(x, weight, bias)
    if cut is not None:
        return parts_sum(_mid_gemm(x, weight, bias, cut))
    import torch.nn.functional as F

    return F.linear(x, weight, bias)


def linear_f32_fixed(x, weight):
    """x weight^T in fp32, as linear_fixed, where mid_gemm has a fixed product
    with an fp32 result, else None."""
    cut = _fixed_mid(x, weight, f32=True)
    if cut is None:
        return None
    return _mid_gemm(x, weight, None, cut, summed=True).sums[0]


def _mid_f32_tile(M: int, N: int, K: int):
    """qt of a whole mid_gemm with an fp32 result, or None where another product
    takes x weight^T: weights above _SKINNY_MAX_ELEMS at up to 64 rows, whose sums
    are short chains, of K from 2560 on: 32000 x 4096 errs by 1.15e-7 at any
    number of rows, streamed by 1.9e-7 up to 4 rows and 1.15e-7 up to 16, a
    library product by 3.9e-7 (K 2048 1.02e-7, streamed 0.97e-7). us, here
    (streamed to 16 rows, then library): 32000 x 4096, 1 row 43.6 (49.5), 8 rows
    43.1 (55.0), 32 rows 44.1 (60.1), 64 rows 46.0 (61.9); 128256 x 4096, 64
    rows 188 (223); 50304 x 2560, whose tiles fill their rounds to 0.77, 16 rows
    50.0 (67.8), 48 rows 58.0 (54.3)."""
    if (M > 64 or N * K <= _SKINNY_MAX_ELEMS or K < 2560 or K % 64 or N % 8
            or K >= 1 << 22 or N >= 1 << 24):
        return None
    qt, _ = _mid_cut(M, N, K, False, False, whole=True)
    tiles = -(-N // (32 * qt))
    if tiles < (0.6 if M <= 16 else 0.8) * 256 * -(-tiles // 256):
        return None
    return qt


def linear_f32_rows(x, weight):
    """x weight^T in fp32 (bf16 operands) where the tiles of mid_gemm or the
    streamed product take it, else None."""
    if x.dim() == 2 and _mid_takes(x, weight):
        qt = _mid_f32_tile(x.shape[0], *weight.shape)
        if qt is not None:
            return _mid_gemm(x, weight, None, (qt, 1), summed=True).sums[0]
    if x.dim() == 2 and _streams(x, weight):
        return _stream_gemm(x, weight, dtype=torch.float32)
    return None


_MM_OUT_DTYPE = {}  # device type -> torch.mm(..., out_dtype=) available


def _mm_out_dtype(x) -> bool:
    ok = _MM_OUT_DTYPE.get(x.device.type)
    if ok is None:
        try:
            one = x.new_zeros(16, 16)
            torch.mm(one, one, out_dtype=torch.float32)
            ok = True
        except (TypeError, RuntimeError):
            ok = False
        _MM_OUT_DTYPE[x.device.type] = ok
    return ok


def linear_f32_lib(x, weight):
    """x weight^T in fp32 as a library product: 16-bit operands, fp32 sums, no
    rounding of the result where torch.mm has such a product."""
    import torch.nn.functional as F

    if x.dtype != torch.float32 and _mm_out_dtype(x):
        return torch.mm(x, weight.t(), out_dtype=torch.float32)
    return F.linear(x, weight).float()


@functools.lru_cache(maxsize=4096)
def _tile_fill(M: int, N: int) -> float:
    """Share of the chip that tiles of 256 (the last of 128) rows x 128 columns
    keep busy with rows that are there: workgroups of an XCD take its tiles in
    turn, those of the last rows, 0.55 of a whole one's time, behind the others
    (tile_gemm.hip). 600 rows x 96 columns of tiles are 24 and 12 on each of 8
    XCDs of 32 workgroups, so that some have one of each."""
    rows, left = divmod(M, 256)
    rows, tail = rows + (left > 128), 0 < left <= 128
    cols = -(-N // 128)
    slots = min(256, -(-(rows + tail) * cols // 8) * 8) // 8
    longest = 0.0
    for xcd in range(8):
        whole = rows * cols * (xcd + 1) // 8 - rows * cols * xcd // 8
        every = whole + tail * (cols * (xcd + 1) // 8 - cols * xcd // 8)
        for at in (0, whole % slots, every % slots):  # where the counts drop
            n = -(-max(0, whole - at) // slots)
            longest = max(longest, n + 0.55 * (-(-max(0, every - at) // slots) - n))
    return M * N / (256 * 128 * 256 * longest)


def _tiles(x, weight) -> bool:
    """Whether silu_mul(x weight^T) takes the product of tile_gemm.hip, with
    its activation inside, rather than the library's and a pass behind it: many
    rows, and tiles that fill their rounds over the chip, the more so the longer
    K is, as the library's loop is faster and the activation's pass counts for
    less. us, here (library and activation): 18944 x 3584, 384 rows 130 (122),
    512 rows 158 (148), 600 rows 167 (173), 900 rows 235 (291), 1024 rows 245
    (260), 2017 rows 409 (547), 3150 rows 623 (811), 8192 rows 1540 (1636);
    12288 x 4096, 600 rows (0.57 full) 1.26 of the library's time, 900 rows
    (0.66) 1.11, 1200 rows (0.88) 0.96; 14336 x 8192, 640 rows (0.71) 1.15, 900
    rows (0.77) 0.96; 13824 x 5120, 1300 rows (0.71) 1.07, 900 rows (0.74)
    0.78: the library's kernels turn with the row count too."""
    M, (N, K) = x.shape[0], weight.shape
    least = 0.67 if K < 4096 else 0.72 if K < 8192 else 0.75
    return (_USE_SKINNY and M > 512 and x.is_cuda
            and x.dtype == weight.dtype == torch.bfloat16 and K % 64 == 0
            and 64 <= K < 1 << 22 and N % 16 == 0
            and x.stride(0) < 1 << 22 and _tile_fill(M, N // 2) >= least
            and _plain(x, weight)
            and weight.is_contiguous() and weight.data_ptr() % 16 == 0
            and native_available())


def linear_silu_mul(x, weight):
    """silu_mul(x weight^T), weight [2N, K] the gate rows, then the up rows."""
    if x.dim() == 2 and weight.shape[0] % 2 == 0:
        cut = _mid(x, weight, silu=True)
        if cut is not None:
            return _mid_gemm(x, weight, None, cut, silu=True)
        if _streams(x, weight, True):
            return _stream_gemm(x, weight, silu=True)
        tile = _wide_silu(x, weight)
        if tile is not None:
            out = x.new_empty((x.shape[0], weight.shape[0] // 2))
            _native().wide_gemm(out, _rows_16b(x), weight, None, *tile, True)
            return out
        if _tiles(x, weight):
            out = x.new_empty((x.shape[0], weight.shape[0] // 2))
            _native().tile_silu(out, _rows_16b(x), weight)
            return out
    return silu_mul(linear_bf16(x, weight))


def rmsnorm_fp8(x, weight, eps: float = 1e-6):
    """Fused RMSNorm -> per-token fp8 e4m3: (out8, inv_scale). GPU-only
    fast path (hidden <= 8192); otherwise compose the unfused ops."""
    if x.is_cuda and x.shape[-1] <= 8192:
        out = torch.empty(x.shape, dtype=torch.float8_e4m3fn, device=x.device)
        inv_scale = torch.empty(x.shape[0], dtype=torch.float32, device=x.device)
        _native().rmsnorm_fp8(out, inv_scale, x, None, weight, eps)
        return out, inv_scale
    return quant_fp8_rows(rmsnorm(x, weight, eps))


def fused_add_rmsnorm_fp8(x, residual, weight, eps: float = 1e-6):
    """Fused residual-add + RMSNorm -> fp8: (out8, inv_scale, residual)."""
    if x.is_cuda and x.shape[-1] <= 8192:
        out = torch.empty(x.shape, dtype=torch.float8_e4m3fn, device=x.device)
        inv_scale = torch.empty(x.shape[0], dtype=torch.float32, device=x.device)
        _native().rmsnorm_fp8(out, inv_scale, x, residual, weight, eps)
        return out, inv_scale, residual
    y, res = fused_add_rmsnorm(x, residual, weight, eps)
    q, s = quant_fp8_rows(y)
    return q, s, res


def silu_mul_fp8(gate_up):
    """Fused SwiGLU -> per-token fp8: (out8, inv_scale)."""
    d = gate_up.shape[-1] // 2
    # dynamic-LDS default cap is 64 KiB; stay under it (d*2 bytes staged)
    if gate_up.is_cuda and d % 8 == 0 and d * 2 <= 60 * 1024:
        out = torch.empty((gate_up.shape[0], d), dtype=torch.float8_e4m3fn,
                          device=gate_up.device)
        inv_scale = torch.empty(gate_up.shape[0], dtype=torch.float32,
                                device=gate_up.device)
        _native().silu_mul_fp8(out, inv_scale, gate_up.contiguous())
        return out, inv_scale
    return quant_fp8_rows(silu_mul(gate_up))


def quant_fp8_rows(x):
    """Dynamic per-token fp8 e4m3 quantization: [M, K] bf16 ->
    ([M, K] float8_e4m3fn, [M] fp32 dequant scales) for W8A8 GEMMs
    (torch._scaled_mm rowwise)."""
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=torch.float8_e4m3fn, device=x.device)
        inv_scale = torch.empty(x.shape[0], dtype=torch.float32, device=x.device)
        _native().quant_fp8_rows(out, inv_scale, x.contiguous())
        return out, inv_scale
    return ref.quant_fp8_rows(x)


def moe_topk(router_logits, k: int, renorm: bool):
    """softmax + top-k + optional renorm in one kernel:
    (weights [T,k] f32, ids [T,k] i32). torch.topk tie-breaking (lower
    expert id wins)."""
    if router_logits.is_cuda:
        T = router_logits.shape[0]
        weights = torch.empty(T, k, dtype=torch.float32,
                              device=router_logits.device)
        ids = torch.empty(T, k, dtype=torch.int32,
                          device=router_logits.device)
        _native().moe_topk(weights, ids, router_logits.contiguous(), k,
                           1 if renorm else 0)
        return weights, ids
    return ref.moe_topk(router_logits, k, renorm)


# Rows up to which the router's logits come from the streamed product, which
# reads 16 rows of the gate a workgroup; beyond, the library's is faster.
MOE_ROUTE_ROWS = 256


def moe_route(x, gate, k: int, renorm: bool):
    """moe_topk of the router product x gate^T, its logits fp32 at any number
    of rows: rounded ones tie, and the choice of a row must not turn with the
    step that it runs in."""
    if _route_streams(x, gate):
        return moe_topk(_route_logits(x, gate), k, renorm)
    return moe_topk(linear_f32_lib(x, gate), k, renorm)


def _route_streams(x, gate) -> bool:
    return (x.is_cuda and x.dtype == torch.bfloat16 and x.shape[0] <= MOE_ROUTE_ROWS
            and x.shape[1] % 32 == 0 and gate.is_contiguous()
            and gate.data_ptr() % 16 == 0)


def _route_logits(x, gate):
    logits = torch.empty((x.shape[0], gate.shape[0]), dtype=torch.float32,
                         device=x.device)
    _native().stream_gemm(logits, _rows_16b(x), gate, None, 1, 1, 16, False)
    return logits


def moe_tile(rows: int, top_k: int, experts: int, whole: bool = False) -> int:
    """Pairs of one work item: 16 where few experts have several (weights
    streamed, moe_gemm.hip), 64 where they have 1 to 64 on the mean and the
    sizes are whole steps (mid_gemm.hip, whose items of 128 take over at 32 on
    the mean, as some experts have twice the mean), 128 or more beyond
    (moe_experts). Other sizes are streamed up to 8 on the mean. us, 16 (64;
    128 of mid_gemm; 256): 128 experts of 2048 x 768, 8 per row: 7 rows 91 (91),
    16 rows 147 (139), 64 rows 208 (190; 207), 200 rows 254 (208; 223; 238), 600
    rows (226; 245; 254), 1000 rows (346; 265; 269), 1300 rows (461; 280; 281);
    8 experts of 4096 x 14336, 2 per row: 1 row 133 (162), 16 rows 505 (437;
    446), 200 rows (474; 478; 566), 600 rows (1384; 1099; 726). Up to 32 rows
    items of 32 may take their place (_moe_few). experts: those that the rows
    choose from, of all ranks."""
    if whole and experts <= rows * top_k <= 64 * experts:
        return 64
    return 16 if rows * top_k <= 8 * experts else 128


def _moe_whole(x, H: int, I: int, pairs: int) -> bool:
    """Whether experts can run in items of 64 and more pairs that load rows
    straight into LDS (mid_gemm.hip, wide_engine.h): whole steps of 64 columns,
    and what their 32-bit row offsets reach. Tiles of 128 take the rest, and
    were never the faster ones: 128 experts of 2048 x 768, 8 per row, us, engine
    (128): 5012 rows 452 (742); 8 of 4096 x 14336, 2 per row, 8192 rows 4550
    (9434)."""
    return (_USE_SKINNY and (H | I) % 64 == 0
            and x.shape[0] * x.stride(0) < 1 << 31
            and 2 * I * H < 1 << 31 and pairs < (1 << 23) - 255)


def _moe_way(rows: int, top_k: int, El: int, experts: int, H: int, I: int,
             whole: bool):
    """(pairs of an item, whether in mid_gemm.hip) for El experts here of
    `experts` in all: moe_tile's, and 256 (the engine, wide_engine.h, whose items
    have up to 320) in place of 128 where whole. Experts whose columns leave most CUs without a tile keep the kernels
    with more of them, us, 16 (64 of mid_gemm), 128 (256): 4 experts of 512 x
    256, 2 per row, 16 rows 13 (21), 64 rows 24 (21) in tiles of 128, 1000 rows
    29 (36), 5000 rows 47 (45); 16 experts of 4096 x 1024, 4 per row, 256 tiles
    of 64 columns, 16 rows 88 (86), 400 rows 132 (131)."""
    pairs = rows * top_k
    few = El * -(-I // 64) < 64 and pairs <= 8 * experts
    # the streamed kernel takes whole matrix operands of 32 columns only (16
    # experts of 2056 x 1416, 4 per row, 7 rows, with routing: 95 us in tiles,
    # 120 us as batched products)
    tile = (moe_tile(rows, top_k, experts, whole and not few)
            if (H | I) % 32 == 0 else 128)
    if tile == 64:
        return (128 if pairs > 32 * experts else 64), True
    # (the engine's items are of 192 to 320 pairs: about this many)
    if (tile == 128 and whole
            and (El + pairs // 256) * -(-I // 128) >= 64):
        tile = 256
    return tile, False


@functools.lru_cache(maxsize=4096)
def _moe_few(rows: int, top_k: int, El: int, experts: int, H: int, I: int,
             streamed: bool):
    """Up to 32 rows: (weight rows a wave / 16 of the gate and up tiles, of the
    down tiles) for items of 32 pairs in mid_gemm.hip, or None where the streamed
    kernel is expected to take less (streamed: it is the other choice, else items
    of 64 are). Counted are the tiles of the experts that so many rows touch if
    they choose evenly, in rounds over 256 CUs, a step as in _mid_cut, 1.5 us a
    round; the streamed kernel at 1.5 us and 5.2 TB/s. us with plan and mix, items of
    32 as cut here (streamed; items of 64): 128 experts of 2048 x 768, 8 per row: 1
    row 23.2 (25.7; 30.7), 7 rows 86 (92; 93), 16 rows 142 (146; 146); 8 of 4096 x
    14336, 2 per row: 1 row 132 (132; 164), 4 rows 285 (333; 303), 8 rows 381
    (435; 383); 16 of 4096 x 2048, 2 per row: 1 row 34.6 (30.9; 49), 8 rows 106
    (100; 112); 32 of 1536 x 512, 4 per row, 6 rows 27.0 (23.9; 28.8), 16 rows 36.8
    (36.6; 38.6). Over 21 sizes at 1 to 32 rows this choice takes 0.94 of the time
    without items of 32 and 1.5 % more than the best; 5 of 294 are more than 2 %
    slower than without (16 of 4096 x 2048, 5 rows 105 (97))."""
    n = max(1, round(El * (1 - (1 - top_k / experts) ** rows)))
    best = [1.5 + 6 * H * I * n / 5.2e6] if streamed else [math.inf]
    best.append(None)
    cost = {}
    for up in (True, False):
        N, K = (I, H) if up else (H, I)
        for qt in (2, 4):
            jobs = n * -(-N // ((16 if up else 32) * qt))
            rounds, last = divmod(jobs, 256)
            alone = 0.08 + 0.095 * qt
            us = rounds * (1.5 + K // 64 * max(alone, 0.15 * qt))
            if last:
                us += 1.5 + K // 64 * max(alone, 0.15 * qt * last / 256)
            cost[up, qt] = us
    for cut in ((4, 4), (2, 4), (4, 2), (2, 2)):
        us = cost[True, cut[0]] + cost[False, cut[1]]
        if us < best[0]:
            best = [us, cut]
    return best[1]


def moe_experts(x, w13, w2, weights, ids, expert_base: int = 0,
                experts: int | None = None):
    """sum_j weights[t, j] * expert(ids[t, j])(x[t]) over the silu-GLU experts
    w13 [El, 2I, H] (gate rows, then up rows), w2 [El, H, I]; experts outside
    [expert_base, expert_base + El) contribute nothing (another rank's).
    experts: the number on all ranks (None: El)."""
    if _moe_native(x, w13, w2, ids):
        x, way = _moe_cut(x, w13, w2, ids, experts)
        out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        _native().moe_experts(out, x, w13, w2, weights, ids, expert_base, *way,
                              experts=experts or 0)
        return out
    return ref.moe_experts(x, w13, w2, weights, ids, expert_base)


def moe_experts_parts(x, w13, w2, weights, ids, expert_base: int = 0,
                      experts: int | None = None):
    """moe_experts for a consumer that takes Mixed."""
    if not (_moe_native(x, w13, w2, ids) and x.shape[0]):
        return moe_experts(x, w13, w2, weights, ids, expert_base, experts)
    x, way = _moe_cut(x, w13, w2, ids, experts)
    return Mixed(*_native().moe_expert_rows(
        x, w13, w2, weights, ids, expert_base, *(*way, 4, 4)[:4], None, False,
        experts or 0))


# Rows whose choice of experts the plan makes (moe_gemm.hip), a wave a row: beyond,
# its one workgroup takes longer than the launch that it saves. us with small experts,
# so (apart): 128 experts, 8 per row, 1 row 14.3 (15.4), 8 rows 16.8 (17.8), 16 rows
# 24.6 (24.0), 32 rows 29.6 (24.8); 64, 6 per row, 8 rows 15.6 (16.6), 16 rows 20.7
# (20.8); 8, 2 per row, 8 rows 12.5 (13.8), 24 rows 14.0 (14.3).
_PLAN_ROWS = 8


def moe_routed_parts(x, gate, k: int, renorm: bool, w13, w2, expert_base: int = 0):
    """moe_experts_parts of what moe_route chooses among gate's experts, the choice
    made by the kernel that plans the experts' rows, or None where that takes no such
    rows: few, whose launches count."""
    T, E = x.shape[0], gate.shape[0]
    if not (1 <= T <= _PLAN_ROWS and E <= 128 and 1 <= k <= min(16, E) and T * k <= 512
            and _route_streams(x, gate)):
        return None
    weights = torch.empty((T, k), dtype=torch.float32, device=x.device)
    ids = torch.empty((T, k), dtype=torch.int32, device=x.device)
    if not _moe_native(x, w13, w2, ids):
        return None
    x, way = _moe_cut(x, w13, w2, ids, E)
    return Mixed(*_native().moe_expert_rows(
        x, w13, w2, weights, ids, expert_base, *(*way, 4, 4)[:4],
        _route_logits(x, gate), bool(renorm), E))


def _moe_native(x, w13, w2, ids) -> bool:
    return (x.is_cuda and x.dtype == torch.bfloat16 and w13.shape[2] % 8 == 0
            and w2.shape[2] % 8 == 0 and w13.shape[0] <= 1024
            and ids.shape[1] <= 16)


def _moe_engine(pairs: int, El: int, experts: int, H: int, I: int, way) -> bool:
    """Whether the engine takes over from items in mid_gemm.hip: from 32 pairs an
    expert on, where both products have a tile for every CU. us with plan, engine
    (the better of items of 64 and 128): 128 experts of 2048 x 768, 8 per row, 144
    rows 203 (202), 528 rows 222 (246), 1008 rows 253 (297); 64 of 2048 x 1408, 6
    per row, 352 rows 203 (218), 672 rows 227 (259); 16 of 4096 x 2048, 2 per row,
    264 rows 139 (152), 504 rows 160 (197); with fewer tiles, 8 of 4096 x 14336, 2
    per row, 252 rows 583 (526), 32 of 1536 x 512, 4 per row, 416 rows 60 (58). With
    20 to 30 pairs it is the choice of experts that decides: a prompt of 400 rows
    through 4 layers of the first 1608 us (1584)."""
    return (way[1] and pairs >= 32 * experts
            and El * min(-(-H // 256), -(-I // 128)) >= 256)


def _moe_cut(x, w13, w2, ids, experts):
    """x with rows on 16 bytes, and (pairs of an item, whether mid_gemm.hip
    takes them[, tiles of items of 32])."""
    El, H, I = w13.shape[0], w13.shape[2], w2.shape[2]
    rows, k = ids.shape
    x = _rows_16b(x)
    whole = _moe_whole(x, H, I, rows * k)
    way = _moe_way(rows, k, El, experts or El, H, I, whole)
    if _moe_engine(rows * k, El, experts or El, H, I, way):
        way = (256, False)
    # matrices of 2^19 weights and more: below, launches are what counts
    if (rows <= 32 and whole and way in ((16, False), (64, True))
            and H * I >= 1 << 19):
        cut = _moe_few(rows, k, El, experts or El, H, I, way[0] == 16)
        if cut is not None:
            way = (32, True, *cut)
    return x, way


def moe_mix(y, weights, ids, expert_base: int = 0):
    """out[t] = sum_i weights[t,i] * y[ids[t,i]-expert_base, t] with
    out-of-slice experts contributing 0 (TP expert parallelism)."""
    if y.is_cuda:
        El, T, H = y.shape
        assert ids.shape == weights.shape and ids.shape[0] == T
        le = ids - expert_base
        mine = (le >= 0) & (le < El)
        rows = le * T + torch.arange(T, dtype=torch.int32, device=y.device)[:, None]
        return moe_mix_rows(y.reshape(El * T, H), weights.where(mine, 0.0),
                            rows.where(mine, 0))
    return ref.moe_mix(y, weights, ids, expert_base)


def moe_mix_rows(y, weights, rows):
    """out[t] = sum_j weights[t,j] * y[rows[t,j]] — the gather-side mix
    over a flat per-pair expert-output buffer (zero-weight slots point at
    row 0)."""
    if y.is_cuda:
        T, k = weights.shape
        out = torch.empty(T, y.shape[1], dtype=y.dtype, device=y.device)
        _native().moe_mix_rows(out, y.contiguous(), weights, rows)
        return out
    return ref.moe_mix_rows(y, weights, rows)


def sample_tokens(logits, temperatures, uniform):
    """Gumbel-max categorical sampling; rows with temperature 0 are greedy."""
    if logits.is_cuda:
        out = torch.empty(logits.shape[0], dtype=torch.int64, device=logits.device)
        _native().gumbel_sample(out, logits, temperatures, uniform)
        return out
    return ref.gumbel_sample(logits, temperatures, uniform)


def greedy_sample(logits):
    if logits.is_cuda:
        out = torch.empty(logits.shape[0], dtype=torch.int64, device=logits.device)
        _native().greedy_sample(out, logits)
        return out
    return ref.greedy_sample(logits)


# ----------------------------------------------------------------------
# Sequence-state ops (arks_amd_seq_C): the kernels of the layer-list
# decoders — token shift, gated output norm into an fp32 residual, sink
# attention with rotated values, lightning linear attention, mamba1 conv
# and selective scan. Same dispatch rule as above: CUDA tensors run the HIP
# extension or fail loudly, CPU tensors run ops/ref.py.
# ----------------------------------------------------------------------
_S = None
_S_ERR: str | None = None


def _native_seq():
    global _S, _S_ERR
    if _S is None and _S_ERR is None:
        try:
            from . import _load

            _S = _load.load("arks_amd_seq_C")
        except Exception as e:
            _S_ERR = f"{type(e).__name__}: {e}"
    if _S is None:
        raise RuntimeError(
            "arks_amd sequence-state HIP extension (arks_amd_seq_C) is not "
            "built but a GPU op was requested. Build it with `python -m "
            f"arks_amd.ops.build arks_amd_seq_C` (import error: {_S_ERR})"
        )
    return _S


def seq_native_available() -> bool:
    try:
        _native_seq()
        return True
    except RuntimeError:
        return False


def ensure_built(name: str) -> None:
    """Compile one in-tree extension if its library is not there yet (a
    fresh checkout on a GPU box); a no-op once built."""
    global _S_ERR, _C_ERR
    from .build import build, built_so_path

    if built_so_path(name) is None:
        build(name=name)
        _S_ERR = _C_ERR = None


def token_shift(x, shift_w, prev_state, cu_seqlens, seq_lens, state_slots,
                token_seq, out_dtype):
    """(xs, xa): the shifted mixer input and the plain row, both cast to
    out_dtype; prev_state takes each sequence's last row."""
    if x.is_cuda:
        xs = torch.empty(x.shape, dtype=out_dtype, device=x.device)
        xa = xs if out_dtype == torch.float32 else torch.empty_like(xs)
        _native_seq().token_shift(xs, xa, x, shift_w, prev_state, cu_seqlens,
                                  seq_lens, state_slots, token_seq)
        return xs, (x if out_dtype == torch.float32 else xa)
    return ref.token_shift(x, shift_w, prev_state, cu_seqlens, seq_lens,
                           state_slots, out_dtype)


def gated_norm_residual(x, y, gate, gate_bias, weight, eps, out_dtype=None):
    """x (fp32, in place) += rmsnorm(y * sigmoid(gate + bias)) * weight.
    Returns the new x cast to out_dtype when one is asked for. y and gate may
    be Parts."""
    if isinstance(y, Parts) or isinstance(gate, Parts):
        W = x.shape[1]
        if (out_dtype in (None, torch.bfloat16) and W % 8 == 0 and W <= 8192
                and all(not isinstance(p, Parts) or p.bias is None
                        for p in (y, gate))):
            xa = (torch.empty(x.shape, dtype=out_dtype, device=x.device)
                  if out_dtype is not None else None)
            _native_seq().gated_norm_sums(
                x, xa, *map(_sums_or_rows, (y, gate)), gate_bias, weight, eps,
                None, None, None, None, None)
            return xa
        y, gate = parts_sum(y), parts_sum(gate)
    if x.is_cuda:
        if out_dtype == torch.float32:
            out_dtype = None  # x itself is the fp32 copy
            ret_x = True
        else:
            ret_x = False
        xa = (torch.empty(x.shape, dtype=out_dtype, device=x.device)
              if out_dtype is not None else None)
        _native_seq().gated_norm_residual(x, xa, y, gate, gate_bias, weight, eps)
        return x if ret_x else xa
    return ref.gated_norm_residual(x, y, gate, gate_bias, weight, eps, out_dtype)


def _sums_or_rows(p):
    return p.sums if isinstance(p, Parts) else p if p is None else _rows_16b(p)


def norm_shift_takes(x, batch, out_dtype) -> bool:
    """Whether gated_norm_shift takes a step's residual rows: one a sequence."""
    return (x.is_cuda and out_dtype == torch.bfloat16 and batch.max_q_len == 1
            and batch.seq_lens.shape[0] == x.shape[0] and x.shape[1] % 8 == 0
            and x.shape[1] <= 8192)


def gated_norm_shift(x, y, gate, gate_bias, weight, eps, shift_w, prev_state,
                     seq_lens, state_slots):
    """gated_norm_residual, then token_shift of its rows (in bf16, one a sequence:
    norm_shift_takes) for the layer behind, from one launch."""
    xs, xa = (torch.empty(x.shape, dtype=torch.bfloat16, device=x.device)
              for _ in range(2))
    _native_seq().gated_norm_sums(
        x, xa, *map(_sums_or_rows, (y, gate)), gate_bias, weight, eps, xs, shift_w,
        prev_state, seq_lens, state_slots)
    return xs, xa


def rms_norm_f32(x, weight, eps, out_dtype):
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=out_dtype, device=x.device)
        _native_seq().rms_norm_f32(out, x, weight, eps)
        return out
    return ref.rms_norm_f32(x, weight, eps, out_dtype)


def qk_norm_rope_cache(q, k, v, q_norm_w, k_norm_w, eps, positions,
                       inv_freq_qk, inv_freq_v, k_cache, v_cache,
                       slot_mapping, interleaved=True, rot_mag=1.0,
                       unit_norm_after=False):
    """rot_mag: factor on cos and sin; unit_norm_after: q and k are divided
    by their root mean square over the head after the rotation (no weight)."""
    if q.is_cuda:
        T, H, D = q.shape
        qo = torch.empty((T, H, D), dtype=q.dtype, device=q.device)
        _native_seq().qk_norm_rope_cache(
            qo, q, k, v, q_norm_w, k_norm_w, eps, positions, inv_freq_qk,
            inv_freq_v, k_cache, v_cache, slot_mapping, interleaved,
            float(rot_mag), bool(unit_norm_after))
        return qo
    return ref.qk_norm_rope_cache(q, k, v, q_norm_w, k_norm_w, eps, positions,
                                  inv_freq_qk, inv_freq_v, k_cache, v_cache,
                                  slot_mapping, interleaved, rot_mag,
                                  unit_norm_after)


# head sizes the MFMA kernels are built for (q/k size == value size)
_MFMA_HEAD_DIMS = (32, 64, 96, 128, 256)
_MFMA_LADDER_DIMS = (64, 128)  # 256-row ladder + flash-decode kernels


def sink_attention_tiles(q_lens, kv_lens, num_q_heads, num_kv_heads,
                         head_dim, device):
    """Work lists of the MFMA attention kernels for one step and one head
    layout (build once per step, reuse in every layer of that layout)."""
    big = head_dim in _MFMA_LADDER_DIMS
    return build_extend_tiles(
        q_lens, kv_lens, False, device, num_q_heads=num_q_heads, ladder=big,
        flash_decode=big and num_q_heads // num_kv_heads <= 8)


def attention_sink_paged(q, k_cache, v_cache, block_tables, seq_lens,
                         cu_seqlens, token_seq, scale, sink=True,
                         inv_freq_v=None, interleaved=True, max_q_len=0,
                         positions=None, tiles=None, sink_w=None,
                         softcap=0.0, window=0, keep_first=0, out=None,
                         out_scale=1.0, maps=1, slopes=None,
                         step_cache: dict | None = None):
    """Causal attention of packed rows over paged keys with an optional
    sink (score 0, or sink_w per head), tanh-capped scores, a distance bias
    (slopes [H]: slope[h] (i - j) off the scores), a sliding
    window that keeps the first keep_first keys, and position-turned values
    (see ref.attention_sink_paged). bf16 rows with equal q/k and value head
    sizes the MFMA kernels are built for run those (then a pass that turns
    each row's output back); capped, windowed or per-head-sink attention
    runs the masked matrix-core kernels where they are built; anything else
    — float32 rows, other sizes — runs the general kernel. out: a [T, H, V]
    view (rows may be strided) to write, times out_scale. maps M > 1: a key
    row holds M keys side by side that share the row's value, and query
    head group g * M + m reads key m of key/value head g."""
    masked = (sink_w is not None or softcap > 0 or window > 0
              or slopes is not None
              or out is not None or maps > 1
              or k_cache.untyped_storage().data_ptr()
              == v_cache.untyped_storage().data_ptr())
    if q.is_cuda and masked:
        T, H, D = q.shape
        V = v_cache.shape[3]
        if out is None:
            out = torch.empty((T, H, V), dtype=q.dtype, device=q.device)
        S = _native_seq()
        if not (use_masked_mfma and q.dtype == torch.bfloat16
                and S.attention_masked_mfma(
                    out, q, k_cache, v_cache, block_tables, seq_lens,
                    cu_seqlens, token_seq, scale, sink_w, softcap, window,
                    keep_first, out_scale, max_q_len == 1, maps, slopes)):
            S.attention_sink_paged(
                out, q, k_cache, v_cache, block_tables, seq_lens, cu_seqlens,
                token_seq, scale, sink, None, interleaved, max_q_len, sink_w,
                softcap, window, keep_first, out_scale, maps, slopes)
        return out
    if q.is_cuda:
        T, H, D = q.shape
        V = v_cache.shape[3]
        G = k_cache.shape[1]
        fast = (q.dtype == torch.bfloat16 and D == V and k_cache.shape[2] == 16)
        if (fast and max_q_len == 1 and T == seq_lens.shape[0]
                and D in _MFMA_LADDER_DIMS and H // G <= 8):
            # one row per sequence: the flash-decode kernel needs no host
            # work list, so it also runs inside a captured decode graph
            out = attention_decode_paged(
                q, k_cache, v_cache, block_tables, seq_lens, scale,
                sink=sink, native=_native_seq(), plan=step_decode_plan(
                    seq_lens, G, 0, False, _native_seq(), step_cache))
            if inv_freq_v is not None:
                _native_seq().unrotate_rows(out, positions, inv_freq_v,
                                            interleaved)
            return out
        if fast and tiles is not None and D in _MFMA_HEAD_DIMS:
            out = attention_extend_paged(
                q, k_cache, v_cache, block_tables, seq_lens, cu_seqlens,
                None, scale, tiles=tiles, sink=sink, native=_native_seq(),
                step_cache=step_cache)
            if inv_freq_v is not None:
                _native_seq().unrotate_rows(out, positions, inv_freq_v,
                                            interleaved)
            return out
        out = torch.empty((T, H, V), dtype=q.dtype, device=q.device)
        _native_seq().attention_sink_paged(
            out, q, k_cache, v_cache, block_tables, seq_lens, cu_seqlens,
            token_seq, scale, sink, inv_freq_v, interleaved, max_q_len, None,
            0.0, 0, 0, 1.0, 1, None)
        return out
    res = ref.attention_sink_paged(q, k_cache, v_cache, block_tables,
                                   seq_lens, cu_seqlens, scale, sink,
                                   inv_freq_v, interleaved, sink_w, softcap,
                                   window, keep_first, maps, slopes)
    if out is None:
        return res
    out.copy_((res.float() * out_scale).to(out.dtype))
    return out


use_masked_mfma = True  # tests switch it off to compare both paths
# prompt portions over two-map key rows: the work-sorted prefill kernels
# (head sizes of the 256-row ladder kernel) instead of the masked tiles
use_ladder_maps = True
PREFILL_MAP_DIMS = (64, 128)
# prompt portions under a distance bias or per-head sinks: the same kernel
use_ladder_bias = True


def seq_extension():
    """The sequence-state extension (its build of the paged attention
    kernels serves the layer-list models)."""
    return _native_seq()


SCAN_CHUNK = 64  # rows per chunk of the chunk-parallel recurrent prefill
use_lightning_mfma = True  # tests switch it off to compare both paths


def scan_chunks(q_lens: list[int], device, chunk: int = SCAN_CHUNK) -> dict:
    """Cut every sequence's rows of this step into chunks of <= `chunk`
    rows, as metadata of 'virtual sequences' the scan kernels can run in
    parallel: pass 1 scans each chunk from zero state into a scratch slot
    of its own (lens0: chunk starts at position 0), a small combine kernel
    walks each sequence's chunks in order and leaves every chunk's START
    state in its scratch slot, pass 2 scans again from those (lens1: start
    > 0) and writes the outputs. Same arithmetic as the row-by-row scan up
    to fp32 summation order."""
    rows, off = [], [0]
    for n in q_lens:
        rows += [min(chunk, n - j) for j in range(0, n, chunk)]
        off.append(len(rows))
    cu = [0]
    for r in rows:
        cu.append(cu[-1] + r)
    cu, lens0, lens1, slots, off = upload(
        [torch.tensor(x, dtype=torch.int32) for x in (
            cu, rows, [r + 1 for r in rows], list(range(len(rows))), off)], device)
    return {"n": len(rows), "cu": cu, "lens0": lens0, "lens1": lens1,
            "rows": lens0, "slots": slots, "off": off}


# the lightning kernels' input convention without positions: rows pass
# through silu (no positions, no rotary table, pairing, key scale)
_SILU_ROWS = (None, None, False, 1.0)


def lightning_scan(q, k, v, decay, state, cu_seqlens, seq_lens, state_slots,
                   max_q_len=0, chunks=None):
    """chunks (scan_chunks of this step): run the prefill chunk-parallel."""
    if q.is_cuda:
        T, H, D = q.shape
        V = v.shape[2]
        S = _native_seq()
        out = torch.empty((T, H, V), dtype=torch.float32, device=q.device)
        if chunks is not None and max_q_len > SCAN_CHUNK:
            c = chunks
            part = torch.empty((c["n"], H, D, V), dtype=torch.float32,
                               device=q.device)
            # bf16 rows with head sizes the matrix-core kernels are built
            # for run those; the general kernel does the same two passes
            mfma = (q.dtype == torch.bfloat16 and use_lightning_mfma
                    and S.lightning_mfma(out, part, q, k, v, decay, c["cu"], 1,
                                         *_SILU_ROWS))
            if not mfma:
                S.lightning_scan(out, q, k, v, decay, part, c["cu"],
                                 c["lens0"], c["slots"], SCAN_CHUNK,
                                 *_SILU_ROWS)
            # the matrix-core passes keep their scratch states transposed
            S.lightning_combine(part, decay, state, c["off"], c["rows"],
                                cu_seqlens, seq_lens, state_slots, mfma)
            if mfma:
                S.lightning_mfma(out, part, q, k, v, decay, c["cu"], 2,
                                 *_SILU_ROWS)
            else:
                S.lightning_scan(out, q, k, v, decay, part, c["cu"],
                                 c["lens1"], c["slots"], SCAN_CHUNK,
                                 *_SILU_ROWS)
            return out
        S.lightning_scan(out, q, k, v, decay, state, cu_seqlens, seq_lens,
                         state_slots, max_q_len, *_SILU_ROWS)
        return out
    return ref.lightning_scan(q, k, v, decay, state, cu_seqlens, seq_lens,
                              state_slots)


def gated_rmsnorm(o, weight, gate, eps, out_dtype):
    if o.is_cuda:
        out = torch.empty(o.shape, dtype=out_dtype, device=o.device)
        _native_seq().gated_rmsnorm(out, o, weight, gate, eps)
        return out
    return ref.gated_rmsnorm(o, weight, gate, eps, out_dtype)


def causal_conv_silu(x, weight, bias, state, cu_seqlens, seq_lens,
                     state_slots, token_seq, weight_t=None, max_q_len=0):
    """weight_t: [taps, C] copy of the taps for the vectorised bf16 kernel;
    bias may be None; max_q_len 1 (every sequence brings one row) lets the
    kernel replace the history in the same launch."""
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        _native_seq().causal_conv_silu(out, x, weight, weight_t, bias, state,
                                       cu_seqlens, seq_lens, state_slots,
                                       token_seq, max_q_len == 1)
        return out
    return ref.causal_conv_silu(x, weight, bias, state, cu_seqlens, seq_lens,
                                state_slots)


def selective_scan(u, dbc, z, dt_w, dt_b, A, Dp, state, cu_seqlens, seq_lens,
                   state_slots, max_q_len=0, dt_pre=None, chunks=None):
    """dt_pre: fp32 [T, C] = dt_raw @ dt_w^T from a GEMM (else projected in
    the kernel); chunks (scan_chunks of this step): chunk-parallel prefill."""
    if u.is_cuda:
        S = _native_seq()
        out = torch.empty(u.shape, dtype=u.dtype, device=u.device)
        if chunks is not None and max_q_len > SCAN_CHUNK:
            c = chunks
            C, N = A.shape
            part = torch.empty((c["n"], C, N), dtype=torch.float32,
                               device=u.device)
            dsum = torch.empty((c["n"], C), dtype=torch.float32,
                               device=u.device)
            # pass 1 needs end states and dt sums only: the lane kernel
            # skips the outputs when it is given none
            light = dt_pre is not None and N <= 64
            S.selective_scan(None if light else out, u, dbc, z, dt_w, dt_b, A,
                             Dp, part, c["cu"], c["lens0"], c["slots"], dt_pre,
                             dsum)
            S.scan_combine(part, dsum, A, state, c["off"], cu_seqlens,
                           seq_lens, state_slots)
            S.selective_scan(out, u, dbc, z, dt_w, dt_b, A, Dp, part, c["cu"],
                             c["lens1"], c["slots"], dt_pre, None)
            return out
        S.selective_scan(out, u, dbc, z, dt_w, dt_b, A, Dp, state, cu_seqlens,
                         seq_lens, state_slots, dt_pre, None)
        return out
    return ref.selective_scan(u, dbc, z, dt_w, dt_b, A, Dp, state, cu_seqlens,
                              seq_lens, state_slots)


def gelu_tanh(x):
    """tanh-form GELU; x may be a column slice of a wider GEMM output, or Parts."""
    if isinstance(x, Parts):
        if x.bias is None and x.sums.shape[2] % 8 == 0:
            out = torch.empty(x.sums.shape[1:], dtype=torch.bfloat16,
                              device=x.sums.device)
            _native_seq().gelu_tanh_sums(out, x.sums)
            return out
        x = parts_sum(x)
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        _native_seq().gelu_tanh(out, x)
        return out
    return ref.gelu_tanh(x)


# ----------------------------------------------------------------------
# Stream-residual blocks, window attention with pooled blocks, rotary
# retention, clamped GLU, grouped routing (same extension, same rule).
# ----------------------------------------------------------------------
def stream_mix_norm(xs, y, y_bias, mix, out_w, in_w, norm_w, norm_b, eps):
    """Residual kept as s weighted copies xs [s, T, C] fp32. With y: every
    copy is rewritten from all old ones, new[t] = sum_s mix[s,t] old[s] +
    out_w[t] (y + y_bias). With in_w: returns layer_norm(sum_s in_w[s]
    new[s]) * norm_w + norm_b as fp32 [T, C] — the next sublayer's input,
    produced by the same pass over the rows."""
    if xs.is_cuda:
        s, T, C = xs.shape
        n = (torch.empty((T, C), dtype=torch.float32, device=xs.device)
             if in_w is not None else None)
        _native_seq().stream_mix_norm(xs, n, y, y_bias, mix, out_w, in_w,
                                      norm_w, norm_b, eps)
        return n
    return ref.stream_mix_norm(xs, y, y_bias, mix, out_w, in_w, norm_w,
                               norm_b, eps)


def short_conv_residual(h, weight, state, cu_seqlens, seq_lens, state_slots,
                        token_seq, out_dtype):
    """h + causal depthwise conv of h over time (taps = weight.shape[1],
    history of taps-1 rows per sequence in `state`), cast to out_dtype."""
    if h.is_cuda:
        out = torch.empty(h.shape, dtype=out_dtype, device=h.device)
        _native_seq().short_conv_residual(out, h, weight, state, cu_seqlens,
                                          seq_lens, state_slots, token_seq)
        return out
    return ref.short_conv_residual(h, weight, state, cu_seqlens, seq_lens,
                                   state_slots, out_dtype)


pool_slots_per_page = ref.pool_slots_per_page


def kv_write_pooled(k, v, k_cache, v_cache, kp_cache, vp_cache, slot_mapping,
                    positions, block_tables, token_seq, pool):
    """Write the step's keys/values to their pages, then the mean key and
    value of every block of `pool` positions this step completes into the
    pooled caches (see ref.kv_write_pooled for the layout)."""
    if k.is_cuda:
        _native_seq().kv_write_pooled(k, v, k_cache, v_cache, kp_cache,
                                      vp_cache, slot_mapping, positions,
                                      block_tables, token_seq, pool)
        return
    ref.kv_write_pooled(k, v, k_cache, v_cache, kp_cache, vp_cache,
                        slot_mapping, positions, block_tables, token_seq, pool)


use_window_mfma = True  # tests switch it off to compare both paths


def attention_window_pool(q, k_cache, v_cache, kp_cache, vp_cache,
                          block_tables, seq_lens, cu_seqlens, token_seq,
                          scale, window, pool, out, out_scale=1.0,
                          max_q_len=0):
    """Sliding-window softmax attention whose rows also see one pooled
    key/value per block of `pool` positions older than every key of the
    window (ref.attention_window_pool). Writes out [T, H, V] (may be a
    column slice of a wider row), scaled by out_scale."""
    if q.is_cuda:
        S = _native_seq()
        if not (use_window_mfma and q.dtype == torch.bfloat16
                and S.attention_window_pool_mfma(
                    out, q, k_cache, v_cache, kp_cache, vp_cache, block_tables,
                    seq_lens, cu_seqlens, token_seq, scale, window, pool,
                    out_scale, max_q_len == 1)):
            S.attention_window_pool(
                out, q, k_cache, v_cache, kp_cache, vp_cache, block_tables,
                seq_lens, cu_seqlens, token_seq, scale, window, pool,
                out_scale)
        return out
    return ref.attention_window_pool(q, k_cache, v_cache, kp_cache, vp_cache,
                                     block_tables, seq_lens, cu_seqlens,
                                     scale, window, pool, out, out_scale)


def retention_scan(q, k, v, decay, state, cu_seqlens, seq_lens, state_slots,
                   positions, inv_freq, interleaved, k_scale, max_q_len=0,
                   chunks=None):
    """The lightning kernels on plain rows: q and k are turned by their
    position (first 2*len(inv_freq) dims) and k scaled as they are loaded,
    nothing is activated. chunks: chunk-parallel prefill as lightning_scan."""
    if q.is_cuda:
        T, H, D = q.shape
        V = v.shape[2]
        S = _native_seq()
        out = torch.empty((T, H, V), dtype=torch.float32, device=q.device)
        rot = (positions, inv_freq, bool(interleaved), float(k_scale))
        if chunks is not None and max_q_len > SCAN_CHUNK:
            c = chunks
            part = torch.empty((c["n"], H, D, V), dtype=torch.float32,
                               device=q.device)
            mfma = (q.dtype == torch.bfloat16 and use_lightning_mfma
                    and S.lightning_mfma(out, part, q, k, v, decay, c["cu"], 1,
                                         *rot))
            if not mfma:
                S.lightning_scan(out, q, k, v, decay, part, c["cu"],
                                 c["lens0"], c["slots"], SCAN_CHUNK, *rot)
            S.lightning_combine(part, decay, state, c["off"], c["rows"],
                                cu_seqlens, seq_lens, state_slots, mfma)
            if mfma:
                S.lightning_mfma(out, part, q, k, v, decay, c["cu"], 2, *rot)
            else:
                S.lightning_scan(out, q, k, v, decay, part, c["cu"],
                                 c["lens1"], c["slots"], SCAN_CHUNK, *rot)
            return out
        S.lightning_scan(out, q, k, v, decay, state, cu_seqlens, seq_lens,
                         state_slots, max_q_len, *rot)
        return out
    return ref.retention_scan(q, k, v, decay, state, cu_seqlens, seq_lens,
                              state_slots, positions, inv_freq, interleaved,
                              k_scale)


def head_norm_gate(o, gate, eps, heads, out, out_scale=1.0):
    """Per-head unit RMS of o [T, heads*V] fp32, times silu(gate), times
    out_scale, into out (may be a column slice of a wider row)."""
    if o.is_cuda:
        _native_seq().head_norm_gate(out, o, gate, eps, heads, out_scale)
        return out
    return ref.head_norm_gate(o, gate, eps, heads, out, out_scale)


_GLU_MODES = {"swiglu": 0, "clamped": 1, "gelu_tanh": 2}


def glu_act(gu, kind, limit=0.0, alpha=1.0, out=None, row_scale=None):
    """[gate | up] rows -> activated rows (ref.glu_act); out: a [T, F]
    view (rows may be strided) to write instead of a new tensor; row_scale
    [T] fp32: a factor on each row's gate and up."""
    if gu.is_cuda:
        F_ = gu.shape[-1] // 2
        if out is None:
            out = torch.empty((gu.shape[0], F_), dtype=gu.dtype,
                              device=gu.device)
        _native_seq().glu_act(out, gu, _GLU_MODES[kind], float(limit),
                              float(alpha), row_scale)
        return out
    res = ref.glu_act(gu, kind, limit, alpha, row_scale)
    if out is None:
        return res
    out.copy_(res)
    return out


def moe_route_grouped(logits, top, groups=1, keep=1, score="softmax",
                      renorm=True, matrix=False, bias=None, correction=None,
                      group_top=1, shared_gate=False):
    """Group-limited routing: (weights [T, top] fp32, ids [T, top] int32);
    score "softmax" or "sigmoid" of the logits (+ bias [E] fp32), renorm: the
    chosen scores divided by their sum. correction [E]: added to the scores
    where experts and groups are chosen, not to the weights; group_top: how
    many of a group's largest choice scores make its own (1 or 2). matrix:
    also a [T, E] fp32 tensor holding each row's weights at the experts it
    uses and 0 elsewhere. shared_gate: the logits' last column is the shared
    expert's, and its sigmoid the matrix's."""
    if logits.is_cuda:
        T, E = logits.shape
        w = torch.empty((T, top), dtype=torch.float32, device=logits.device)
        ids = torch.empty((T, top), dtype=torch.int32, device=logits.device)
        mat = (torch.empty((T, E), dtype=torch.float32, device=logits.device)
               if matrix else None)
        _native_seq().moe_route_grouped(w, ids, logits, top, groups, keep,
                                        score == "sigmoid", bool(renorm), mat,
                                        bias, correction, group_top,
                                        bool(shared_gate))
        return (w, ids, mat) if matrix else (w, ids)
    experts = logits[:, :logits.shape[1] - bool(shared_gate)]
    w, ids = ref.moe_route_grouped(experts, top, groups, keep, score, renorm,
                                   bias, correction, group_top)
    if matrix:
        mat = ref.route_scale_matrix(w, ids, experts.shape[1])
        if shared_gate:
            mat = torch.cat([mat, torch.sigmoid(logits[:, -1:].float())], 1)
        return w, ids, mat
    return w, ids


def route_rows_takes(h, router, groups: int = 1) -> bool:
    """Whether moe_route_rows takes these rows: steps of few, whose launches count,
    and a lane an expert, no groups. us in a replayed graph, here (the library's
    product and moe_route_grouped): 16 experts of 4096 columns, 1 row 6.4 (12.0), 64
    rows 6.9 (12.8); 64 of 2048, 64 rows 10.2 (12.6), 256 rows 16.3 (12.4)."""
    T, W = h.shape
    return (_USE_SKINNY and h.is_cuda and 1 <= T <= 64 and groups == 1
            and h.dtype == router.dtype == torch.bfloat16
            and 8 <= W and W % 8 == 0 and router.shape[0] <= 64
            and _plain(h, router) and h.stride(-1) == 1 and h.stride(0) % 8 == 0
            and h.data_ptr() % 16 == 0 and router.is_contiguous()
            and router.data_ptr() % 16 == 0 and seq_native_available())


def moe_route_rows(h, router, top, score="softmax", renorm=True, matrix=False,
                   bias=None, correction=None, shared_gate=False):
    """moe_route_grouped of the fp32 logits h router^T without groups, where
    route_rows_takes."""
    T, E = h.shape[0], router.shape[0]
    w = torch.empty((T, top), dtype=torch.float32, device=h.device)
    ids = torch.empty((T, top), dtype=torch.int32, device=h.device)
    mat = (torch.empty((T, E), dtype=torch.float32, device=h.device)
           if matrix else None)
    _native_seq().moe_route_rows(w, ids, h, router, top, score == "sigmoid",
                                 bool(renorm), mat, bias, correction,
                                 bool(shared_gate))
    return (w, ids, mat) if matrix else (w, ids)


def moe_sort_pairs(ids, experts, pad=0):
    """(row, expert) pairs in expert order (ref.moe_sort_pairs) from one
    launch."""
    if ids.is_cuda:
        rows = torch.empty(ids.numel() + pad, dtype=torch.int32,
                           device=ids.device)
        place = torch.empty_like(ids)
        counts = torch.empty(experts, dtype=torch.int32, device=ids.device)
        if _native_seq().moe_sort_pairs(rows, place, counts, ids):
            return rows, place, counts
    return ref.moe_sort_pairs(ids, experts, pad)


def moe_mix_seq(y, weights, ids):
    """moe_mix for callers of the sequence-state extension (any float
    dtype of y)."""
    if y.is_cuda:
        El, T, H = y.shape
        out = torch.empty(T, H, dtype=y.dtype, device=y.device)
        _native_seq().moe_mix(out, y.contiguous(), weights, ids)
        return out
    return ref.moe_mix(y, weights, ids, 0)


def moe_mix_rows_seq(y, weights, rows, add=None):
    """out[t] = sum_j weights[t, j] y[rows[t, j]] (+ add[t])."""
    if y.is_cuda:
        T, k = weights.shape
        out = torch.empty(T, y.shape[1], dtype=y.dtype, device=y.device)
        _native_seq().moe_mix_rows(out, y.contiguous(), weights, rows, add)
        return out
    return ref.moe_mix_rows(y, weights, rows, add)


# ----------------------------------------------------------------------
# Shared-norm parallel blocks with a tanh norm, latent attention, mamba2
# (same extension, same rule).
# ----------------------------------------------------------------------
def residual_tanh_norm(x, y, mult, alpha, weight, bias, out_dtype, xa=None):
    """x (fp32 residual, in place) += mult * y when y is given; xa, a
    [T, C] view of the model's dtype (any row stride), takes the new x;
    returns tanh(alpha x) * weight + bias in out_dtype (None when weight is
    None). alpha is a one-element fp32 tensor."""
    if x.is_cuda:
        h = (torch.empty(x.shape, dtype=out_dtype, device=x.device)
             if weight is not None else None)
        _native_seq().residual_tanh_norm(x, h, xa, y, float(mult), alpha,
                                         weight, bias)
        return h
    return ref.residual_tanh_norm(x, y, mult, alpha, weight, bias, out_dtype, xa)


def latent_prepare(cq, ckv, q_norm_w, kv_norm_w, eps, positions, inv_freq,
                   cache, slot_mapping, interleaved=True, rot_mag=1.0):
    """Latent attention's row work before the up-projections
    (ref.latent_prepare): returns the normed query latent and writes the
    normed key/value latent with the turned shared key part to its page."""
    if cq.is_cuda:
        out = torch.empty(cq.shape, dtype=cq.dtype, device=cq.device)
        _native_seq().latent_prepare(out, cq, ckv, q_norm_w, kv_norm_w, eps,
                                     positions, inv_freq, cache, slot_mapping,
                                     bool(interleaved), float(rot_mag))
        return out
    return ref.latent_prepare(cq, ckv, q_norm_w, kv_norm_w, eps, positions,
                              inv_freq, cache, slot_mapping, interleaved,
                              rot_mag)


def latent_query(q, q_abs, positions, inv_freq, out, interleaved=True,
                 rot_mag=1.0):
    """out [T, H, Rk + 2P] = [q_abs ([H, T, Rk]) | turned last 2P dims of q]."""
    if q.is_cuda:
        _native_seq().latent_query(out, q, q_abs, positions, inv_freq,
                                   bool(interleaved), float(rot_mag))
        return out
    return ref.latent_query(q, q_abs, positions, inv_freq, out, interleaved,
                            rot_mag)


def latent_pages(k_up, v_up, lat, heads, rot_dim, block_size):
    """Per-head key and value pages from up-projected context rows and the
    shared key part (ref.latent_pages)."""
    if lat.is_cuda:
        pages = (lat.shape[0] // block_size, heads, block_size)
        kt = lat.new_empty(pages + (k_up.shape[1] // heads + rot_dim,))
        vt = lat.new_empty(pages + (v_up.shape[1] // heads,))
        _native_seq().latent_pages(kt, vt, k_up, v_up, lat)
        return kt, vt
    return ref.latent_pages(k_up, v_up, lat, heads, rot_dim, block_size)


# rows per chunk of mamba2's chunk-parallel prefill: a chunk's state
# (heads x state x vdim floats) is written and read four times, so chunks
# are long; the scan itself is sequential inside a chunk either way
MAMBA2_CHUNK = 256


def mamba2_scan(xbc, dt_raw, dt_bias, rate, Dp, state, cu_seqlens, seq_lens,
                state_slots, heads, vdim, nstate, groups, max_q_len=0,
                chunks=None):
    """Scalar-decay state-space recurrence (ref.mamba2_scan); chunks
    (scan_chunks of this step): chunk-parallel prefill as lightning_scan —
    every chunk's end state and summed step sizes from zero state, a
    combine pass that leaves each chunk's start state, then the outputs."""
    if xbc.is_cuda:
        S = _native_seq()
        T = xbc.shape[0]
        out = torch.empty((T, heads * vdim), dtype=torch.float32,
                          device=xbc.device)
        if chunks is not None:
            c = chunks
            part = torch.empty((c["n"], heads, nstate, vdim),
                               dtype=torch.float32, device=xbc.device)
            dsum = torch.empty((c["n"], heads), dtype=torch.float32,
                               device=xbc.device)
            S.mamba2_scan(None, xbc, dt_raw, dt_bias, rate, Dp, part, c["cu"],
                          c["lens0"], c["slots"], heads, vdim, nstate, groups,
                          dsum)
            S.mamba2_combine(part, dsum, rate, state, c["off"], cu_seqlens,
                             seq_lens, state_slots)
            S.mamba2_scan(out, xbc, dt_raw, dt_bias, rate, Dp, part, c["cu"],
                          c["lens1"], c["slots"], heads, vdim, nstate, groups,
                          None)
            return out
        S.mamba2_scan(out, xbc, dt_raw, dt_bias, rate, Dp, state, cu_seqlens,
                      seq_lens, state_slots, heads, vdim, nstate, groups, None)
        return out
    return ref.mamba2_scan(xbc, dt_raw, dt_bias, rate, Dp, state, cu_seqlens,
                           seq_lens, state_slots, heads, vdim, nstate, groups)


def gate_group_norm(y, z, weight, groups, eps, out, out_scale=1.0):
    """out = per-group unit RMS of (y * silu(z)), times weight and out_scale
    (ref.gate_group_norm); y fp32, z and out row-strided views."""
    if y.is_cuda:
        _native_seq().gate_group_norm(out, y, z, weight, groups, eps,
                                      out_scale)
        return out
    return ref.gate_group_norm(y, z, weight, groups, eps, out, out_scale)


# ----------------------------------------------------------------------
# Two-norm parallel blocks with per-channel branch scales, difference
# attention behind short convolutions, input-scaled experts (same
# extension, same rule).
# ----------------------------------------------------------------------
def residual_pair_norm(x, y1, s1, y2, s2, w1, w2, eps, out_dtype):
    """x (fp32 residual, in place) += s1 * y1 + s2 * y2 (each when given,
    s per channel); returns (h1, h2), x divided by its root mean square
    times (1 + w1) and (1 + w2), for each weight given — two norms of the
    same rows from one pass."""
    if x.is_cuda:
        h1 = (torch.empty(x.shape, dtype=out_dtype, device=x.device)
              if w1 is not None else None)
        h2 = (torch.empty(x.shape, dtype=out_dtype, device=x.device)
              if w2 is not None else None)
        _native_seq().residual_pair_norm(x, h1, h2, y1, s1, y2, s2, w1, w2,
                                         float(eps))
        return h1, h2
    return ref.residual_pair_norm(x, y1, s1, y2, s2, w1, w2, eps, out_dtype)


def conv_qkv_cache(p, n_q, n_k, n_v, weight, weight_t, state, cu_seqlens,
                   seq_lens, state_slots, token_seq, positions, temp_coef,
                   temp_every, heads, kv_heads, maps, k_cache, v_cache,
                   slot_mapping):
    """Short causal convolution over the q | k | v channels of the
    in-projection's rows, the position-dependent query factor, the query
    heads regrouped by key map, keys and values to their pages, and the
    sequences' new histories (ref.conv_qkv_cache). weight_t: [taps, C] copy
    of the taps for the vectorised bf16 kernel. Returns q [T, n_q]."""
    if p.is_cuda:
        qo = torch.empty((p.shape[0], n_q), dtype=p.dtype, device=p.device)
        _native_seq().conv_qkv_cache(
            qo, p, n_q, n_k, n_v, weight, weight_t, state, cu_seqlens,
            seq_lens, state_slots, token_seq, positions, float(temp_coef),
            int(temp_every), heads, kv_heads, maps, k_cache, v_cache,
            slot_mapping)
        return qo
    return ref.conv_qkv_cache(p, n_q, n_k, n_v, weight, state, cu_seqlens,
                              seq_lens, state_slots, positions, temp_coef,
                              temp_every, heads, kv_heads, maps, k_cache,
                              v_cache, slot_mapping)


def diff_head_norm_gate(a, gate, lam, eps, mult, heads, kv_heads, out):
    """Two attention maps per head into one gated output row
    (ref.diff_head_norm_gate): (a1 - lam a2) at unit RMS per head, times
    mult, times sigmoid(gate)."""
    if a.is_cuda:
        _native_seq().diff_head_norm_gate(out, a, gate, float(lam), float(eps),
                                          float(mult), heads, kv_heads)
        return out
    return ref.diff_head_norm_gate(a, gate, lam, eps, mult, heads, kv_heads,
                                   out)


def moe_glu_scaled(gu, scale, experts, ff, shared_ff, scale_input=True,
                   act="swiglu", limit=0.0, shared_limit=0.0, alpha=1.0,
                   shared_scale=False):
    """Activated rows of all experts side by side, each expert's gate and
    up (or, without scale_input, their activated product) scaled by the
    row's weight for it, plus the shared expert's, scaled by the last column
    of scale with shared_scale (ref.moe_glu_scaled)."""
    if gu.is_cuda:
        out = torch.empty((gu.shape[0], experts * ff + shared_ff),
                          dtype=gu.dtype, device=gu.device)
        _native_seq().moe_glu_scaled(out, gu, scale, experts, ff, shared_ff,
                                     bool(scale_input), act == "clamped",
                                     bool(shared_scale), float(limit),
                                     float(shared_limit), float(alpha))
        return out
    return ref.moe_glu_scaled(gu, scale, experts, ff, shared_ff, scale_input,
                              act, limit, shared_limit, alpha, shared_scale)


def routed_takes(h, w_gu, w_down, experts: int, ff: int) -> bool:
    """Whether routed_experts has kernels for these rows and weights: up to 16
    rows of bf16, no shared expert, sizes in whole chunks of K."""
    T, W = h.shape
    return (_USE_SKINNY and h.is_cuda and 1 <= T <= 16
            and h.dtype == w_gu.dtype == w_down.dtype == torch.bfloat16
            and experts <= 64 and ff % 256 == 0 and experts * ff % 1024 == 0
            and W % 512 == 0 and experts * ff < 1 << 22
            and 4 * ff * W < 1 << 32 and h.stride(0) < 1 << 22
            and w_gu.shape == (2 * experts * ff, W)
            and w_down.shape == (W, experts * ff)
            and all(w.is_contiguous() and w.data_ptr() % 16 == 0
                    for w in (w_gu, w_down))
            and _plain(h, w_gu, w_down) and seq_native_available())


def routed_experts(h, w_gu, w_down, scale, scale_input=True, act="swiglu",
                   limit=0.0, alpha=1.0):
    """The weighted sum of the experts that rows chose (scale [T, E] fp32: their
    weights, 0 elsewhere), for what routed_takes takes: linear, moe_glu_scaled and
    linear over all experts, without those that nobody chose, in one order of sums
    for any number of rows. us, here (those three), 16 experts of ff 3584 on 4096
    columns, 4 per row, weights cold: 1 row (4 of them chosen) 67 (244), 2 rows
    (8) 124 (287), 8 rows (11) 167 (245), 16 rows (all) 248 (308)."""
    T, E = scale.shape
    C = _native_seq()
    x = _rows_16b(h)
    a = torch.empty((T, w_down.shape[1]), dtype=h.dtype, device=h.device)
    C.routed_up(a, x, w_gu, scale, bool(scale_input), act == "clamped",
                float(limit), float(alpha))
    y = torch.empty((T, w_down.shape[0]), dtype=h.dtype, device=h.device)
    C.routed_down(y, a, w_down, scale)
    return y


def moe_wide_takes(h, w_gu, w_down, experts: int, ff: int, top: int) -> bool:
    """Whether moe_wide_rows takes these rows and weights: whole steps of 64
    columns, and what 32-bit row offsets reach; more experts than 2, whose many
    rows fill the chip one by one. For the rows of prompts. us with plan or sort and
    mix, moe_wide_rows (a library product per expert and matrix, behind a gather
    and a host read of their counts): 16 experts of 4096 x 3584, 4 per row: 257
    rows 274 (742), 1000 rows 522 (1103), 3500 rows 1098 (1736), 8000 rows 2387
    (2727); 64 of 2048 x 1408, 6 per row: 1000 rows 284 (2610), 16384 rows 1551
    (3394); 4 of 4096 x 14336, 2 per row: 257 rows 485 (703), 8192 rows 4742
    (5085); 2 of these, 2 per row: 257 rows 468 (374), 8192 rows 4583 (4157).
    An expert's row adds up in one chain, whatever rows are beside it: the library's
    products of 65 to about 4000 rows were seen to give the same bits at 5 sizes, those
    of fewer rows others in 0.01 to 0.6 % of the results; the error against 64 bits is
    the same at any number (3.50e-3 of the rows, all of it the rounding to bf16)."""
    T, W = h.shape
    return (_USE_SKINNY and h.is_cuda and T >= 1
            and h.dtype == w_gu.dtype == w_down.dtype == torch.bfloat16
            and 2 < experts <= 1024 and top <= 16 and ff > 0 and W > 0
            and (W | ff) % 64 == 0 and T * W < 1 << 31
            and T * top < (1 << 23) - 255 and 2 * ff * W < 1 << 31
            and w_gu.shape[0] >= 2 * experts * ff and w_gu.shape[1] == W
            and w_down.shape[0] == W and w_down.shape[1] >= experts * ff
            and w_down.shape[1] % 8 == 0 and w_down.numel() < 1 << 31
            and all(w.is_contiguous() and w.data_ptr() % 16 == 0
                    for w in (w_gu, w_down))
            and _plain(h, w_gu, w_down))


def moe_wide_rows(h, w_gu, w_down, weights, ids, experts: int, ff: int,
                  scale_input: bool = False):
    """The silu-GLU experts' rows of h, in any order, and each (row, choice)
    pair's place there [T, top]: w_gu [>= E * 2 ff, W], w_down [W, >= E * ff],
    ids [T, top] int32 below E. Projections, activation and result are each
    rounded to h's dtype; scale_input: the weights scale the experts' input (the
    caller adds the rows up as they are)."""
    x = h if (h.stride(-1) == 1 and h.stride(0) % 8 == 0
              and h.data_ptr() % 16 == 0
              and h.shape[0] * h.stride(0) < 1 << 31) else h.clone(
                  memory_format=torch.contiguous_format)
    return _native().moe_wide_rows(x, w_gu, w_down, weights.contiguous(),
                                   ids.contiguous(), experts, ff,
                                   bool(scale_input))


# ----------------------------------------------------------------------
# Sandwich-norm blocks, per-head output gate, capped logits, channel-decay
# delta rule (same extension, same rule).
# ----------------------------------------------------------------------
def residual_sandwich_norm(x, y, w_post, mult, w_pre, eps, out_dtype,
                           y2=None, w_post2=None):
    """x (fp32 residual, in place) += mult * (rms_norm(y) * w_post +
    rms_norm(y2) * w_post2) for the results given (one without a weight is
    added as it is); returns rms_norm(x) * w_pre in out_dtype (None without
    w_pre): the norms behind one sublayer, the sum and the norm in front of
    the next from one pass."""
    if x.is_cuda:
        h = (torch.empty(x.shape, dtype=out_dtype, device=x.device)
             if w_pre is not None else None)
        _native_seq().residual_sandwich_norm(x, h, y, w_post, float(mult),
                                             w_pre, float(eps), y2, w_post2)
        return h
    return ref.residual_sandwich_norm(x, y, w_post, mult, w_pre, eps,
                                      out_dtype, y2, w_post2)


def softcap_(x, cap):
    """x (fp32, in place) = cap * tanh(x / cap)."""
    if x.is_cuda:
        _native_seq().softcap(x, float(cap))
        return x
    return ref.softcap_(x, cap)


def head_gate(o, gate, out, out_scale=1.0):
    """out[t, h] = o[t, h] * sigmoid(gate[t, h]) * out_scale
    (ref.head_gate); o and out [T, H, V] views with dense last dims."""
    if o.is_cuda:
        _native_seq().head_gate(out, o, gate, float(out_scale))
        return out
    return ref.head_gate(o, gate, out, out_scale)


DELTA_CHUNK = 64  # rows per chunk of the matrix-core delta rule
use_delta_mfma = True  # tests switch it off to compare both paths


def channel_delta(u, decay, beta, gate, rate, dt_bias, norm_w, eps, state,
                  cu_seqlens, seq_lens, state_slots, heads, kv_heads, dim,
                  vdim, out, max_q_len=0, chunks=None, head_decay=False,
                  silu_gate=False):
    """Delta rule with a decay per key channel (head_decay: one per head) and
    its gated unit-RMS read-out (ref.channel_delta; silu_gate: silu instead
    of sigmoid) into out [T, H*V] (rows may be strided).
    chunks (scan_chunks of this step, DELTA_CHUNK rows each): bf16 rows with
    head sizes the matrix-core kernels are built for run those; anything
    else runs row by row."""
    if u.is_cuda:
        if (chunks is not None and use_delta_mfma and u.dtype == torch.bfloat16
                and _native_seq().channel_delta_chunks(
                    out, u, decay, beta, gate, rate, dt_bias, norm_w,
                    float(eps), ref.DELTA_UNIT_EPS, state, chunks["off"],
                    chunks["cu"], cu_seqlens, seq_lens, state_slots, heads,
                    kv_heads, dim, vdim, bool(head_decay), bool(silu_gate))):
            return out
        _native_seq().channel_delta_scan(
            out, u, decay, beta, gate, rate, dt_bias, norm_w, float(eps),
            ref.DELTA_UNIT_EPS, state, cu_seqlens, seq_lens, state_slots,
            heads, kv_heads, dim, vdim, max_q_len, bool(head_decay),
            bool(silu_gate))
        return out
    return ref.channel_delta(u, decay, beta, gate, rate, dt_bias, norm_w, eps,
                             state, cu_seqlens, seq_lens, state_slots, heads,
                             kv_heads, dim, vdim, out, head_decay, silu_gate)


# ----------------------------------------------------------------------
# Pre-norm two-mixer blocks: hashed embedding of token pairs, q/k norm over
# all heads at once, squared relu (same extension, same rule).
# ----------------------------------------------------------------------
def hashed_embed(ids, embed, table, prev, cu_seqlens, seq_lens, state_slots,
                 token_seq, scale, mul_prev, mul_cur, max_q_len=0):
    """fp32 rows embed[token] * scale + table[hash of (previous token,
    token)] (ref.hashed_embed). prev [slots] int32: every sequence's last
    token, replaced. max_q_len 1 (one row per sequence): one launch."""
    if embed.is_cuda:
        x = torch.empty((ids.shape[0], embed.shape[1]), dtype=torch.float32,
                        device=embed.device)
        _native_seq().hashed_embed(x, ids, embed, table, prev, cu_seqlens,
                                   seq_lens, state_slots, token_seq,
                                   float(scale), int(mul_prev), int(mul_cur),
                                   max_q_len == 1)
        return x
    return ref.hashed_embed(ids, embed, table, prev, cu_seqlens, seq_lens,
                            state_slots, scale, mul_prev, mul_cur)


def row_norm_qk_cache(q, k, v, q_norm_w, k_norm_w, eps, positions, temp_coef,
                      temp_every, k_cache, v_cache, slot_mapping):
    """q [T, H*D] and k [T, G*D] normed over all their heads at once, q times
    the position's factor, k and v to their pages (ref.row_norm_qk_cache).
    Returns q [T, H*D]."""
    if q.is_cuda:
        qo = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        _native_seq().row_norm_qk_cache(
            qo, q, k, v, q_norm_w, k_norm_w, float(eps), positions,
            float(temp_coef), int(temp_every), k_cache, v_cache, slot_mapping)
        return qo
    return ref.row_norm_qk_cache(q, k, v, q_norm_w, k_norm_w, eps, positions,
                                 temp_coef, temp_every, k_cache, v_cache,
                                 slot_mapping)


def relu_square(x):
    """max(x, 0)^2."""
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        _native_seq().relu_square(out, x)
        return out
    return ref.relu_square(x)
