"""CPU sanity tests for the reference ops (the oracle the HIP kernels are
tested against) — internal consistency checks that run without a GPU."""

import math

import pytest
import torch

from arks_amd.ops import ref


def test_rmsnorm_matches_manual():
    torch.manual_seed(0)
    x = torch.randn(4, 64)
    w = torch.randn(64)
    out = ref.rmsnorm(x, w, 1e-6)
    manual = x / (x.pow(2).mean(-1, keepdim=True) + 1e-6).sqrt() * w
    torch.testing.assert_close(out, manual, atol=1e-5, rtol=1e-5)


def test_decode_consistent_with_prefill_last_token():
    """Decoding the last token against the cache must equal the last row of
    full prefill attention."""
    torch.manual_seed(1)
    hq, hkv, hd, L, bs = 4, 2, 64, 37, 16
    q = torch.randn(L, hq, hd)
    k = torch.randn(L, hkv, hd)
    v = torch.randn(L, hkv, hd)
    cu = torch.tensor([0, L], dtype=torch.int32)
    scale = 1.0 / math.sqrt(hd)
    full = ref.attention_prefill_varlen(q, k, v, cu, scale)

    nb = (L + bs - 1) // bs
    kc = torch.zeros(nb, hkv, bs, hd)
    vc = torch.zeros(nb, hkv, bs, hd)
    slots = torch.arange(L, dtype=torch.int64)
    ref.reshape_and_cache(k, v, kc, vc, slots)
    bt = torch.arange(nb, dtype=torch.int32).unsqueeze(0)
    sl = torch.tensor([L], dtype=torch.int32)
    dec = ref.attention_decode_paged(q[-1:].clone(), kc, vc, bt, sl, scale)
    torch.testing.assert_close(dec[0], full[-1], atol=1e-4, rtol=1e-4)


def test_rope_preserves_norm():
    torch.manual_seed(2)
    hd = 64
    pos = torch.arange(10)
    q = torch.randn(10, 2 * hd)
    k = torch.randn(10, hd)
    cs = ref.rope_cos_sin_cache(hd, 32)
    q2, k2 = ref.rope_apply(pos, q, k, cs, hd)
    # Rotation preserves the norm of each head.
    torch.testing.assert_close(
        q2.view(10, 2, hd).norm(dim=-1), q.view(10, 2, hd).norm(dim=-1), atol=1e-4, rtol=1e-4
    )
    # position 0 is identity
    torch.testing.assert_close(q2[0], q[0], atol=1e-6, rtol=1e-6)


def test_gumbel_sample_greedy_when_t0():
    torch.manual_seed(3)
    logits = torch.randn(5, 100)
    temps = torch.zeros(5)
    u = torch.rand(5, 100)
    out = ref.gumbel_sample(logits, temps, u)
    torch.testing.assert_close(out, logits.argmax(-1))


def test_rope_scaling_matches_transformers():
    """llama3 + yarn rope_scaling pinned against transformers' rope_utils."""
    import torch
    from transformers import LlamaConfig
    from transformers.modeling_rope_utils import ROPE_INIT_FUNCTIONS

    from arks_amd.ops.ref import _scaled_inv_freq

    base_inv = 1.0 / (500000.0 ** (torch.arange(0, 128, 2, dtype=torch.float64) / 128))
    l3 = {"rope_type": "llama3", "factor": 8.0, "low_freq_factor": 1.0,
          "high_freq_factor": 4.0, "original_max_position_embeddings": 8192}
    cfg = LlamaConfig(rope_theta=500000.0, hidden_size=4096,
                      num_attention_heads=32,
                      max_position_embeddings=131072, rope_scaling=dict(l3))
    inv_hf, _ = ROPE_INIT_FUNCTIONS["llama3"](cfg, "cpu")
    mine, ms = _scaled_inv_freq(base_inv, l3, 500000.0, 128)
    assert ms == 1.0
    torch.testing.assert_close(mine, inv_hf.double(), rtol=1e-5, atol=0)

    yarn = {"rope_type": "yarn", "factor": 4.0,
            "original_max_position_embeddings": 4096}
    cfg2 = LlamaConfig(rope_theta=10000.0, hidden_size=4096,
                       num_attention_heads=32,
                       max_position_embeddings=16384, rope_scaling=dict(yarn))
    inv_hf2, att2 = ROPE_INIT_FUNCTIONS["yarn"](cfg2, "cpu")
    base2 = 1.0 / (10000.0 ** (torch.arange(0, 128, 2, dtype=torch.float64) / 128))
    mine2, ms2 = _scaled_inv_freq(base2, yarn, 10000.0, 128)
    torch.testing.assert_close(mine2, inv_hf2.double(), rtol=1e-5, atol=0)
    assert abs(ms2 - att2) < 1e-9


def test_step_results_follow_their_inputs(monkeypatch):
    """What the layers of a pass share belongs to the lengths, tables and rows
    that it was made from."""
    import arks_amd.ops as ops

    made = []

    def plan(lens, *a, **kw):
        made.append(lens.tolist())
        return tuple(lens.tolist())

    monkeypatch.setattr(ops, "attention_decode_plan", plan)
    cache = {}
    a, b = torch.tensor([5, 9]), torch.tensor([7, 1])
    get = lambda lens: ops.step_decode_plan(lens, 4, 0, False, None, cache)
    assert get(a) == get(a) == (5, 9) and len(made) == 1
    assert get(b) == (7, 1) and get(a) == (5, 9)
    a.add_(1)
    assert get(a) == (6, 10)
    with torch.inference_mode():
        c = torch.tensor([3])
        assert get(c) == (3,)
    tables, lens = torch.arange(12).view(3, 4), torch.tensor([10, 20, 30])
    rows = lambda pick: ops._single_rows(tables, lens, torch.tensor(pick), 4, 0,
                                         False, True, None, cache)
    for pick in ([0, 2], [1], [0, 2]):
        tab, n, p = rows(pick)
        assert torch.equal(tab, tables[pick]) and n.tolist() == list(p)
        assert p == tuple(lens[pick].tolist())
    lens.mul_(2)
    assert rows([0, 2])[2] == (20, 60)


def test_short_portions_are_split_beside_long_ones():
    """A short portion behind a deep context is cut over its keys also where
    long portions fill the chip, and leaves their own cut as it was."""
    from arks_amd.ops import build_extend_tiles

    def split(q, kv, **kw):
        t64, t256, _, combine, ws = build_extend_tiles(
            q, kv, False, "cpu", num_q_heads=28, **kw)
        rows = t256.tolist()
        assert ws == sum(r[3] > 1 for r in rows)
        for at, n, i, q0 in combine.tolist():
            assert rows[at:at + n] == [[i, q0, p, n] for p in range(n)]
        return {i: max(r[3] for r in rows if r[0] == i)
                for i in {r[0] for r in rows}}, t64.shape[0]

    assert split([2560, 65], [2560, 6113]) == ({0: 1, 1: 8}, 0)
    assert split([2560, 65], [2560, 600]) == ({0: 1, 1: 1}, 0)  # none waits
    assert split([2560, 65], [2560, 200]) == ({0: 1}, 2)  # 64-row kernel
    assert split([2560], [2560]) == ({0: 1}, 0)
    # 8 x 28 workgroups are cut in 3, also with 2 x 28 of short portions
    assert split([2048], [2048])[0] == {0: 3}
    assert split([2048, 33, 33], [2048, 3000, 3000])[0] == {0: 3, 1: 8, 2: 8}
    assert split([65], [6113])[0] == {0: 8}
    assert split([0, 65], [400, 6113], min_ladder=1)[0] == {1: 8}


def test_stage_rows():
    """What a step's rows read: spans that begin in the prompt or in the output,
    last tokens, pages; missing tokens, pages or room are refused."""
    import random

    import pytest

    import arks_amd.ops as ops

    if not ops.native_available():
        pytest.skip("needs the built extension")
    rng, bs = random.Random(5), 16
    prompts = [[rng.randrange(1 << 20) for _ in range(n)] for n in (40, 1, 16, 33)]
    outputs = [[rng.randrange(1 << 20) for _ in range(n)] for n in (0, 5, 1, 15)]
    tables = [rng.sample(range(1 << 30), n) for n in (3, 1, 2, 4)]
    starts, counts = [3, 0, 16, 30], [37, 6, 1, 17]

    def host(rows, width=5):
        return (torch.full((rows,), -7), torch.full((rows,), -7),
                torch.full((rows,), -7), torch.full((6,), -7, dtype=torch.int32),
                torch.full((6, width), -7, dtype=torch.int32))

    def check(first, many, bufs):
        ids, pos, slots, lens, bt = bufs
        at = 0
        for i, (p, o, t, c, n) in enumerate(zip(prompts, outputs, tables, first, many)):
            for j in range(c, c + n):
                assert ids[at] == (p + o)[j] and pos[at] == j
                assert slots[at] == t[j // bs] * bs + j % bs
                at += 1
            assert lens[i] == c + n
            assert bt[i].tolist() == t + [-7] * (5 - len(t))
        assert (ids[at:] == -7).all() and (pos[at:] == -7).all()
        assert (lens[4:] == -7).all() and (bt[4:] == -7).all()

    bufs = host(64)
    ops.stage_rows(prompts, outputs, tables, starts, counts, *bufs, bs)
    check(starts, counts, bufs)
    bufs = host(5)
    ops.stage_rows(prompts, outputs, tables, None, None, *bufs, bs)
    last = [len(p) + len(o) - 1 for p, o in zip(prompts, outputs)]
    check(last, [1] * 4, bufs)
    for bad in (dict(counts=[38, 6, 1, 17]), dict(starts=[-1, 0, 16, 30]),
                dict(tables=[[1, 2], *tables[1:]]), dict(bufs=host(60)),
                dict(bufs=host(64, 3)), dict(counts=[37, 6, 1]),
                dict(outputs=[()] * 4), dict(starts=None)):
        a = dict(starts=starts, counts=counts, tables=tables, outputs=outputs,
                 bufs=host(64)) | bad
        with pytest.raises((RuntimeError, TypeError)):
            ops.stage_rows(prompts, a["outputs"], a["tables"], a["starts"],
                           a["counts"], *a["bufs"], bs)


@pytest.mark.parametrize("rows", [0, 1, 2, 5])
def test_stage_rows_pads(rows):
    """Rows behind the sequences': no cache slot, length 1, page 0; nothing beyond."""
    import arks_amd.ops as ops

    if not ops.native_available():
        pytest.skip("needs the built extension")
    ids, pos, slots = torch.full((3, 6), -7).unbind()
    lens = torch.full((6,), -7, dtype=torch.int32)
    bt = torch.full((6, 3), -7, dtype=torch.int32)
    ops.stage_rows([[4, 5, 6], [7]], [[], [8]], [[2], [9]], None, None, ids, pos,
                   slots, lens, bt, 16, rows)
    pad = max(0, rows - 2)
    rest = [-7] * (4 - pad)
    assert ids.tolist() == [6, 8] + [0] * pad + rest
    assert pos.tolist() == [2, 1] + [0] * pad + rest
    assert slots.tolist() == [34, 145] + [-1] * pad + rest
    assert lens.tolist() == [3, 2] + [1] * pad + rest
    assert bt[:, 0].tolist() == [2, 9] + [0] * pad + rest
    for bad in (7, dict(starts=[0, 0], counts=[1, 1])):  # no room; not one token each
        a = dict(starts=None, counts=None) | (bad if isinstance(bad, dict) else {})
        with pytest.raises(RuntimeError):
            ops.stage_rows([[4], [7]], [[], []], [[2], [9]], a["starts"], a["counts"],
                           ids, pos, slots, lens, bt, 16,
                           bad if isinstance(bad, int) else 3)


def test_objects_older_than_a_header_are_built_again(tmp_path):
    import os

    from arks_amd.ops.build import drop_older

    src, out = tmp_path / "src", tmp_path / "out"
    for d in (src, out):
        d.mkdir()
    for path, at in ((src / "a.h", 100), (src / "b.h", 200), (src / "c.hip", 900),
                     (out / "old.o", 150), (out / "same.o", 200), (out / "new.o", 201),
                     (out / "lib.so", 150)):
        path.touch()
        os.utime(path, (at, at))
    drop_older(str(out), str(src))
    assert sorted(p.name for p in out.iterdir()) == ["lib.so", "new.o"]


def test_mid_sizes_are_whole_cuts():
    """Over a grid of sizes, what mid_gemm is given is a cut that its kernel has:
    16 * 2, 4 or 5 weight rows a wave, at least a step of 64 columns a run of K,
    one run with the activation."""
    from arks_amd import ops

    taken = set()
    for M in (1, 2, 8, 17, 64, 65, 128, 129, 192, 193, 256):
        for N in (8, 64, 328, 1024, 4608, 5752, 5760, 5768, 11520, 11528, 22976,
                  28672, 57344, 151936):
            for K in (64, 128, 192, 320, 512, 896, 2048, 3584, 8192, 18944):
                for silu, summed in ((False, False), (False, True), (True, False)):
                    cut = ops._mid_sizes(M, N, K, silu, summed)
                    if cut is None:
                        continue
                    qt, splits = cut
                    assert qt in (2, 4, 5)
                    assert 1 <= splits <= min(8, K // 64)
                    assert not silu or splits == 1
                    taken.add((qt, splits > 1, silu))
    assert taken == {(qt, many, silu) for qt in (2, 4, 5) for many in (False, True)
                     for silu in (False, True) if not (many and silu)}
    for bad in ((1, 8, 96), (1, 12, 64), (1, 8, 32), (1, 0, 64), (1, 1 << 24, 64),
                (1, 8, 1 << 22)):
        assert ops._mid_sizes(*bad, False, True) is None


def test_mid_sizes_leave_what_others_do_faster():
    """Both sides of the measured lines."""
    from arks_amd import ops

    takes = lambda *size, **kind: ops._mid_sizes(
        *size, kind.get("silu", False), kind.get("summed", False)) is not None
    summed = [  # M, N, K: streamed or the library's; beside it, taken
        ((16, 5120, 2048), (24, 5120, 2048)), ((16, 3072, 2048), (48, 3072, 2048)),
        ((64, 1152, 896), (65, 1152, 896)), ((129, 1152, 896), (128, 1152, 896)),
        ((8, 4096, 4096), (16, 4096, 4096)), ((8, 3584, 3584), (16, 3584, 3584)),
        ((8, 4096, 4096), (8, 4608, 3584)), ((8, 4096, 4096), (8, 2048, 4096)),
        ((200, 2048, 4096), (192, 2048, 4096)), ((256, 3584, 3584), (256, 4608, 3584)),
        ((8, 7680, 2560), (16, 7680, 2560)), ((176, 5120, 2048), (160, 5120, 2048)), ((250, 896, 896), (250, 896, 4864))]
    for left, taken in summed:
        assert not takes(*left, summed=True) and takes(*taken, summed=True)
    plain = [
        ((96, 8192, 2048), (64, 8192, 2048)), ((129, 64128, 8192), (128, 64128, 8192)),
        ((129, 64128, 8192), (129, 32064, 8192)), ((200, 4096, 4096), (192, 4096, 4096)),
        ((96, 50304, 1024), (96, 50304, 2048)), ((250, 50304, 2048), (192, 50304, 2048)),
        ((96, 50304, 2560), (64, 50304, 2560)), ((144, 9216, 3072), (72, 9216, 3072)),
        ((240, 12288, 4096), (256, 12288, 4096)), ((240, 12288, 4096), (240, 24576, 4096))]
    for left, taken in plain:
        assert not takes(*left) and takes(*taken)
    gated = [  # N: gate columns
        ((8, 8192, 4096), (9, 8192, 4096)), ((8, 8192, 4096), (8, 5504, 4096)),
        ((32, 4096, 5120), (32, 5120, 4096)), ((32, 3072, 4096), (64, 3072, 2048)),
        ((96, 27648, 5120), (64, 27648, 5120)), ((96, 27648, 5120), (96, 28672, 8192))]
    for left, taken in gated:
        assert not takes(*left, silu=True) and takes(*taken, silu=True)


def test_wide_cut():
    """Tiles that wide_gemm has, runs of at least four steps, at most 128 MB of
    sums, and no cut where none is asked for; a few hundred rows of long weights
    fill the CUs."""
    from arks_amd import ops

    for M in (257, 300, 511, 700, 1400, 2049, 5000, 16385):
        for N, K in ((2048, 8192), (3584, 18944), (8192, 28672), (37888, 64), (16, 64)):
            for split in (False, True):
                tm, tw, splits, jobs = ops._wide_cut(M, N, K, split, True)
                assert (tm, tw) in ops._WIDE_STEP
                assert jobs == -(-M // tm) * -(-N // tw) * splits
                assert splits == 1 or split and (
                    K // 64 // splits >= 4 and splits * M * N * 4 <= 1 << 27)
    assert all(ops._wide_cut(M, 3584, 18944, True, True)[3] >= 200
               for M in range(257, 2049, 64))


@pytest.mark.parametrize("N,K,takes,leaves", [
    (3584, 18944, (300, 1309, 2314, 4666), (3344, 4352, 8192)),
    (4096, 14336, (300, 1536, 4352), (2837, 3344, 6144, 8192)),
    (6144, 16384, (600, 1309, 2837, 6000), (1800, 2048, 3344, 4096)),
    (8192, 22016, (700, 2314, 4666), (1536, 2048, 3344, 8192)),
    (5120, 27648, (400, 1691, 3344, 7000), (2837, 4666)),
    (2048, 8192, (700, 1280), (6000, 8192)),
    (3584, 8128, (), (300, 2314)), (1008, 16384, (), (300, 2314)),
])
def test_wide_leaves_full_rounds_to_the_library(N, K, takes, leaves, monkeypatch):
    """Sizes at which the library's tiles of 256 x 256 fill their rounds over the CUs
    stay with it (measured 3 to 24 % behind here), whatever the row count is divisible
    by; those of part rounds are taken (4 % to three times as fast)."""
    from types import SimpleNamespace as S

    from arks_amd import ops

    monkeypatch.setattr(ops, "_wide_takes", lambda *a: True)
    for rows in (takes, leaves):
        for M in rows:
            for summed in (False, True):
                cut = ops._wide(S(shape=(M, K)), S(shape=(N, K)), None, summed)
                assert bool(cut) == (rows is takes), (M, summed)
                if cut:
                    assert tuple(cut) == ops._wide_cut(M, N, K, True, summed)[:3]


def test_wide_leaves_full_rounds_to_tiles_of_256(monkeypatch):
    """Gate and up products whose tiles of 256 rows fill their rounds stay in them."""
    from types import SimpleNamespace as S

    from arks_amd import ops

    monkeypatch.setattr(ops, "_wide_takes", lambda *a: True)
    wide = lambda M, N, K: ops._wide_silu(S(shape=(M, K)), S(shape=(N, K)))
    for M, N, K in ((4096, 28672, 4096), (8192, 28672, 4096), (8192, 55296, 5120),
                    (8192, 36864, 6144)):
        assert wide(M, N, K) is None and wide(M - 512 + 20, N, K)
    assert wide(512, 32768, 4096) and wide(8192, 37888, 3584)


def test_pair_cut():
    """Tiles that mid_gemm has, and 1 to 8 runs of a step or more of each product,
    whichever comes first."""
    import random

    from arks_amd import ops

    rng = random.Random(3)
    for _ in range(300):
        M, N = rng.randint(1, 64), 8 * int(2 ** rng.uniform(0, 11))
        K, K2 = (64 * int(16 * 2 ** rng.uniform(0, 5)) for _ in range(2))
        qt, *runs = ops._pair_cut(M, N, K, K2)
        assert qt in (2, 4, 5)
        for n, k in zip(runs, (K, K2)):
            assert 1 <= n <= min(8, k // 64)
        assert ops._pair_cut(M, N, K2, K) == (qt, *runs[::-1])


def test_tile_fill_is_what_the_schedule_takes():
    """The share against the schedule walked out: every workgroup's tiles of its
    XCD in turn, 1 for a whole one and 0.55 for those of the last 128 rows."""
    from arks_amd import ops

    for M in (1, 128, 129, 256, 257, 513, 600, 640, 900, 1024, 2017, 3150, 8192):
        for N in (8, 128, 1000, 4096, 9472, 12288, 14336, 18944, 28672):
            left, cols = M % 256, -(-N // 128)
            rows, tail = M // 256 + (left > 128), 0 < left <= 128
            slots = min(256, -(-(rows + tail) * cols // 8) * 8) // 8
            longest = 0
            for xcd in range(8):
                part = lambda n: n * (xcd + 1) // 8 - n * xcd // 8
                cost = [1.0] * part(rows * cols) + [0.55] * (tail * part(cols))
                longest = max([longest] + [sum(cost[s::slots]) for s in range(slots)])
            want = M * N / (256 * 128 * 256 * longest)
            assert abs(ops._tile_fill(M, N) / want - 1) < 1e-9, (M, N)


def test_moe_way():
    """Pairs of an item and their kernel: by pairs per expert, and for experts
    so small that larger items leave most of the chip idle."""
    from arks_amd import ops

    big = lambda rows, whole=True: ops._moe_way(rows, 8, 128, 128, 2048, 768, whole)
    assert [big(n) for n in (15, 16, 512, 513, 1024, 1025)] == [
        (16, False), (64, True), (64, True), (128, True), (128, True), (256, False)]
    assert [big(n, False) for n in (16, 128, 129, 5000)] == [
        (16, False), (16, False), (128, False), (128, False)]
    # a rank's 16 of 128 experts
    assert ops._moe_way(64, 8, 16, 128, 2048, 768, True) == (64, True)
    tiny = lambda rows: ops._moe_way(rows, 2, 4, 4, 512, 256, True)
    assert [tiny(n) for n in (1, 16, 17, 64, 65, 128, 129, 2000, 5000)] == [
        (16, False), (16, False), (64, True), (64, True), (128, True), (128, True),
        (128, False), (128, False), (256, False)]
    # no whole steps of 32: tiles of 128
    assert ops._moe_way(7, 4, 16, 16, 2056, 1416, False) == (128, False)


def test_moe_engine_takes_over():
    """Items of mid_gemm give way to the engine from 32 pairs an expert on, with a
    tile for every CU in both products."""
    from arks_amd import ops

    takes = lambda rows, k, E, H, I, El=None: ops._moe_engine(
        rows * k, El or E, E, H, I, ops._moe_way(rows, k, El or E, E, H, I, True))
    assert not takes(511, 8, 128, 2048, 768) and takes(512, 8, 128, 2048, 768)
    assert takes(256, 2, 16, 4096, 2048) and not takes(252, 2, 8, 4096, 14336)
    assert not takes(416, 4, 32, 1536, 512)
    assert not takes(512, 8, 128, 2048, 768, 16)  # a rank's 16 experts
    assert not ops._moe_engine(1 << 20, 128, 128, 2048, 768, (128, False))


def test_decode_waves():
    """Two workgroups per CU for fp8 rows, and where sequences outnumber runs."""
    from arks_amd import ops

    assert ops.decode_waves(64, 4) == ops.decode_waves(256, 4) == 256
    assert ops.decode_waves(257, 4) == 512
    assert ops.decode_waves(128, 8) == 128 and ops.decode_waves(256, 8) == 256
    assert ops.decode_waves(256, 2) == 512 and ops.decode_waves(80, 16) == 128
    assert ops.decode_waves(1, 4, True) == 512
    assert ops.decode_waves(3, 4, False, 5) == 15


def test_mid_cut_runs():
    """Beyond 64 rows, where a run of K is one chain of sums, the most runs that
    cost next to nothing; up to 64 rows the least time alone."""
    from arks_amd import ops

    assert ops._mid_cut(96, 2048, 2048, False, True) == (2, 8)
    assert ops._mid_cut(96, 5120, 27648, False, True) == (5, 8)
    assert ops._mid_cut(32, 3584, 18944, False, True) == (2, 4)
    # not where it costs: one run for tiles that fill the CUs
    assert ops._mid_cut(96, 32000, 4096, False, False)[1] == 1
    assert ops._mid_cut(96, 18944, 3584, True, False)[1] == 1


def test_mid_sizes_leave_to_streamed():
    """Small weights at up to 64 rows are left to the streamed product only where
    it takes them."""
    from arks_amd import ops

    left = 0
    for M in (1, 2, 4, 6, 8, 16, 32, 64):
        for N in (128, 512, 896, 1536, 2040, 2048, 4096, 8192):
            for K in (256, 896, 2048, 4096, 4160, 4864, 8192, 14336):
                if (N * K <= ops._SKINNY_MAX_ELEMS
                        and ops._mid_sizes(M, N, K, False, False) is None):
                    left += 1
                    assert ops._stream_sizes(M, N, K), (M, N, K)
    assert left > 50


def test_mid_sizes_up_to_224_rows():
    """Sums of up to 224 rows of squares from 3072 on; 4096 columns of 3072 are
    the library's beyond 192 rows."""
    from arks_amd import ops

    takes = lambda *size: ops._mid_sizes(*size, False, True) is not None
    for M in (193, 208, 224):
        for N, K in ((3072, 3072), (3584, 3584), (3840, 3328), (3072, 4096)):
            assert takes(M, N, K) and not takes(225, N, K)
        assert takes(192, 4096, 3072) and not takes(M, 4096, 3072)


def test_mid_sizes_of_a_second_round():
    """Beyond 128 rows large weights whose tiles leave much of a second round of
    CUs empty are the library's."""
    from arks_amd import ops

    takes = lambda *size: ops._mid_sizes(*size, False, False) is not None
    for M in (129, 160, 224):
        for N, K in ((55296, 5120), (50304, 4096), (43008, 5120)):
            assert not takes(M, N, K), (M, N, K)
        for N, K in ((102400, 4096), (36864, 5120), (152064, 3584), (32064, 4096)):
            assert takes(M, N, K), (M, N, K)
    assert takes(128, 50304, 4096)


def test_moe_few():
    """Items of 32 pairs where their tiles fill the rounds, streamed else."""
    from arks_amd import ops

    assert ops._moe_few(7, 8, 128, 128, 2048, 768, True) == (2, 4)
    assert ops._moe_few(1, 2, 8, 8, 4096, 14336, True) == (4, 2)
    assert ops._moe_few(1, 2, 16, 16, 4096, 2048, True) is None
    # short columns: what the items win does not pay for their rounds
    assert ops._moe_few(3, 4, 32, 32, 1536, 512, True) is None
    assert ops._moe_few(6, 4, 32, 32, 1536, 512, True) is None
    # never streamed where that is not the other choice
    for rows in range(1, 33):
        cut = ops._moe_few(rows, 2, 16, 16, 4096, 2048, False)
        assert cut is None or set(cut) <= {2, 4}
        assert cut is not None
    # a rank's 16 of 128 experts: less than one of them per row
    assert ops._moe_few(1, 8, 16, 128, 2048, 768, True) in (None, (2, 2))
    assert ops._moe_few(1, 8, 16, 128, 2048, 768, True) is None
    assert ops._moe_few(16, 8, 16, 128, 2048, 768, True) == (2, 4)
