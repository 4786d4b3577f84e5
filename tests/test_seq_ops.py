"""The sequence-state ops one by one, on inputs made so that a fault shows:
a single far key that must win the softmax, keys on both sides of a page
border, the sink deciding a row, a state slot that is reused, a decay of 1.
Each op is compared with a few lines of plain per-row arithmetic written
here (no code of arks_amd); CPU cases run the reference ops, gpu-marked
cases the HIP kernels."""

import math

import pytest
import torch

from arks_amd import ops

DEVICES = [pytest.param("cpu", torch.float32, id="cpu-f32"),
           pytest.param("cuda", torch.float32, id="gpu-f32", marks=pytest.mark.gpu),
           pytest.param("cuda", torch.bfloat16, id="gpu-bf16", marks=pytest.mark.gpu)]


def i32(x, dev):
    return torch.tensor(x, dtype=torch.int32, device=dev)


def paged_cache(K, Vv, block_size, order, nblocks, dtype, dev):
    """Scatter K [L,G,D], V [L,G,V] into pages in the given page order."""
    L, G, D = K.shape
    kc = torch.zeros(nblocks, G, block_size, D, dtype=dtype, device=dev)
    vc = torch.zeros(nblocks, G, block_size, Vv.shape[2], dtype=dtype, device=dev)
    for j in range(L):
        kc[order[j // block_size], :, j % block_size] = K[j].to(dtype)
        vc[order[j // block_size], :, j % block_size] = Vv[j].to(dtype)
    return kc, vc


@pytest.mark.parametrize("dev,dtype", DEVICES)
@pytest.mark.parametrize("D", [16, 64])
@pytest.mark.parametrize("far", [0, 15, 16, 17, 250])
def test_one_far_key_wins_the_softmax(dev, dtype, D, far):
    """The last query matches exactly one key (first token, either side of
    a page border, hundreds back): the output must be that key's value."""
    torch.manual_seed(far)
    L, G, H, bs = 300, 1, 2, 16
    K = torch.randn(L, G, D) * 0.05
    Vv = torch.randn(L, G, D)
    e = torch.zeros(D)
    e[3] = 1.0
    K[far, 0] = 6.0 * e
    order = torch.randperm(40).tolist()
    kc, vc = paged_cache(K, Vv, bs, order, 40, dtype, dev)
    for n_new in (1, 5):  # decoded alone, and as the last row of a portion
        q = torch.randn(n_new, H, D) * 0.05
        q[-1, :] = 6.0 * e
        qd = q.to(dtype).to(dev)
        tiles = (ops.sink_attention_tiles([n_new], [L], H, G, D, dev)
                 if dev == "cuda" else None)
        out = ops.attention_sink_paged(
            qd, kc, vc, i32([order[:19]], dev), i32([L], dev), i32([0, n_new], dev),
            i32([0] * n_new, dev), 1.0, sink=True, inv_freq_v=None,
            max_q_len=n_new, positions=torch.arange(L - n_new, L, device=dev),
            tiles=tiles)
        got = out[-1].float().cpu()
        # e^36 against 300 keys near e^0 and the sink's e^0
        assert torch.allclose(got, Vv[far, 0].expand(H, D).to(dtype).float(),
                              atol=3e-2 if dtype == torch.bfloat16 else 1e-4), (n_new, far)


@pytest.mark.parametrize("dev,dtype", DEVICES)
@pytest.mark.parametrize("D", [16, 64])
def test_sink_takes_its_share(dev, dtype, D):
    """All scores 0: n keys and the sink share the weight, so the output is
    sum(v) / (n + 1), not the mean; very negative scores give 0."""
    L, G, H, bs = 37, 1, 1, 16
    Vv = torch.randn(L, G, D)
    kc, vc = paged_cache(torch.zeros(L, G, D), Vv, bs, [2, 0, 1], 3, dtype, dev)
    q = torch.zeros(1, H, D, dtype=dtype, device=dev)
    args = (kc, vc, i32([[2, 0, 1]], dev), i32([L], dev), i32([0, 1], dev), i32([0], dev))
    tiles = ops.sink_attention_tiles([1], [L], H, G, D, dev) if dev == "cuda" else None
    kw = dict(inv_freq_v=None, max_q_len=1, positions=torch.tensor([L - 1], device=dev),
              tiles=tiles)
    out = ops.attention_sink_paged(q, *args, 1.0, sink=True, **kw)
    want = Vv[:, 0].to(dtype).float().sum(0) / (L + 1)
    tol = 2e-2 if dtype == torch.bfloat16 else 1e-5
    assert torch.allclose(out[0, 0].float().cpu(), want, atol=tol)
    out = ops.attention_sink_paged(q, *args, 1.0, sink=False, **kw)
    assert torch.allclose(out[0, 0].float().cpu(), want * (L + 1) / L, atol=tol)
    kc2, _ = paged_cache(torch.full((L, G, D), -4.0), Vv, bs, [2, 0, 1], 3, dtype, dev)
    q1 = torch.ones(1, H, D, dtype=dtype, device=dev)
    out = ops.attention_sink_paged(q1, kc2, *args[1:], 1.0, sink=True, **kw)
    assert out.float().abs().max() < 1e-6 * math.exp(30)  # e^(-4D) << 1
    assert out.float().abs().max() < 1e-3


@pytest.mark.parametrize("dev,dtype", DEVICES)
def test_rotated_values_come_back_in_the_query_frame(dev, dtype):
    """One key at position j holds value v turned by j; a query at position i
    that sees only it (strongly) must return v turned by j - i."""
    D, bs = 8, 16
    inv = torch.tensor([1.0, 0.5, 0.1, 0.01])
    j, i = 5, 21
    v = torch.randn(D)
    k = torch.zeros(i + 1, 1, D)
    k[j, 0, 0] = 8.0
    vals = torch.zeros(i + 1, 1, D)
    kc, vc = paged_cache(k, vals, bs, [1, 0], 2, dtype, dev)
    # store v through the op that fills the cache (rotation by the position)
    qkv_q = torch.zeros(1, 1, D, dtype=dtype, device=dev)
    ops.qk_norm_rope_cache(
        qkv_q, k[j:j + 1].to(dtype).to(dev), v.view(1, 1, D).to(dtype).to(dev), None, None,
        1e-5, torch.tensor([j], device=dev), torch.zeros(0, device=dev),
        inv.to(dev), kc, vc, torch.tensor([1 * bs + j], device=dev))
    q = torch.zeros(1, 1, D, dtype=dtype, device=dev)
    q[0, 0, 0] = 8.0
    out = ops.attention_sink_paged(
        q, kc, vc, i32([[1, 0]], dev), i32([i + 1], dev), i32([0, 1], dev), i32([0], dev),
        1.0, sink=True, inv_freq_v=inv.to(dev), max_q_len=1,
        positions=torch.tensor([i], device=dev))
    ang = (j - i) * inv
    want = torch.empty(D)
    want[0::2] = v[0::2] * torch.cos(ang) - v[1::2] * torch.sin(ang)
    want[1::2] = v[1::2] * torch.cos(ang) + v[0::2] * torch.sin(ang)
    assert torch.allclose(out[0, 0].float().cpu(), want,
                          atol=5e-2 if dtype == torch.bfloat16 else 1e-4)


@pytest.mark.parametrize("dev,dtype", DEVICES)
def test_lightning_keeps_a_far_token_with_decay_one_and_forgets_with_small(dev, dtype):
    H, D, V, T = 2, 8, 8, 200
    q = torch.zeros(T, H, D)
    k = torch.zeros(T, H, D)
    v = torch.zeros(T, H, V)
    k[0, :, 1] = 5.0   # silu(5) ~ 4.97
    v[0, :, 2] = 5.0
    q[T - 1, :, 1] = 5.0
    decay = torch.tensor([1.0, 0.5])
    state = torch.zeros(3, H, D, V, device=dev)
    s5 = 5.0 / (1 + math.exp(-5.0))
    # whole, and cut in portions through a reused slot holding garbage
    for cuts in ([T], [1, 2, 64, 33, 100]):
        state.fill_(7.0)
        at, o_last = 0, None
        for n in cuts:
            o = ops.lightning_scan(
                q[at:at + n].to(dtype).to(dev), k[at:at + n].to(dtype).to(dev),
                v[at:at + n].to(dtype).to(dev), decay.to(dev), state,
                i32([0, n], dev), i32([at + n], dev), i32([1], dev), max_q_len=n)
            at += n
            o_last = o[-1].cpu()
        assert abs(float(o_last[0, 2]) - s5 ** 3) < 0.05 * s5 ** 3
        assert abs(float(o_last[1, 2])) < 1e-20
        assert float(state[0].min()) == 7.0 and float(state[2].min()) == 7.0


@pytest.mark.parametrize("dev,dtype", DEVICES)
@pytest.mark.parametrize("taps", [1, 2, 4])
def test_conv_history_across_portions_of_one_and_two(dev, dtype, taps):
    C, T = 5, 9
    x = torch.randn(T, C)
    w = torch.randn(C, taps)
    b = torch.randn(C)
    xd = x.to(dtype).float()
    want = torch.zeros(T, C)
    for t in range(T):
        acc = b.clone()
        for j in range(taps):
            s = t - (taps - 1 - j)
            if s >= 0:
                acc += w[:, j] * xd[s]
        want[t] = acc * torch.sigmoid(acc)
    state = (torch.full((2, taps - 1, C), 9.0, device=dev) if taps > 1 else None)
    outs, at = [], 0
    for n in (1, 1, 2, 1, 4):
        outs.append(ops.causal_conv_silu(
            x[at:at + n].to(dtype).to(dev), w.to(dev), b.to(dev), state,
            i32([0, n], dev), i32([at + n], dev), i32([1], dev), i32([0] * n, dev)))
        at += n
    got = torch.cat(outs).float().cpu()
    assert torch.allclose(got, want, atol=5e-2 if dtype == torch.bfloat16 else 1e-5)


@pytest.mark.parametrize("dev,dtype", DEVICES)
def test_token_shift_first_row_and_padding_rows(dev, dtype):
    W = 6
    x = torch.randn(5, W, device=dev)
    w = torch.rand(W, device=dev)
    state = torch.full((2, W), 3.0, device=dev)
    # seq 0: 3 rows starting at position 0 (slot 1); seq 1: one row at
    # position 4 (slot 0, reads the stored row); seq 2: padding row
    xs, xa = ops.token_shift(x, w, state, i32([0, 3, 4, 5], dev), i32([3, 5, 1], dev),
                             i32([1, 0, -1], dev), i32([0, 0, 0, 1, 2], dev), dtype)
    xc = x.cpu()
    wc = w.cpu()
    want = torch.stack([
        xc[0] * (1 - wc), xc[1] + (xc[0] - xc[1]) * wc, xc[2] + (xc[1] - xc[2]) * wc,
        xc[3] + (3.0 - xc[3]) * wc, xc[4] * (1 - wc)])
    tol = 3e-2 if dtype == torch.bfloat16 else 1e-6
    assert torch.allclose(xs.float().cpu(), want, atol=tol)
    assert torch.allclose(xa.float().cpu(), xc, atol=tol)
    assert torch.equal(state[1].cpu(), xc[2]) and torch.equal(state[0].cpu(), xc[3])


@pytest.mark.parametrize("dev,dtype", DEVICES)
def test_selective_scan_remembers_through_a_slow_channel(dev, dtype):
    """Channel 0 decays slowly (A ~ 0), channel 1 fast: an input at the first
    token is still read out 150 tokens later on channel 0 only."""
    C, N, R, T = 2, 4, 1, 151
    u = torch.zeros(T, C)
    u[0] = 2.0
    dbc = torch.zeros(T, R + 2 * N)
    dbc[:, R:R + N] = 1.0       # B
    dbc[:, R + N:] = 1.0        # C
    z = torch.full((T, C), 20.0)  # silu(20) ~ 20
    dt_w = torch.zeros(C, R)
    dt_b = torch.zeros(C)       # dt = softplus(0) = ln 2
    A = torch.tensor([[-1e-4] * N, [-3.0] * N])
    Dp = torch.zeros(C)
    ln2 = math.log(2.0)
    want0 = N * ln2 * 2.0 * math.exp(-1e-4 * ln2 * (T - 1)) * 20.0
    state = torch.full((2, C, N), 5.0, device=dev)
    for cuts in ([T], [2, 1, 100, 48]):
        at = 0
        for n in cuts:
            y = ops.selective_scan(
                u[at:at + n].to(dtype).to(dev), dbc[at:at + n].to(dtype).to(dev),
                z[at:at + n].to(dtype).to(dev), dt_w.to(dev), dt_b.to(dev), A.to(dev),
                Dp.to(dev), state, i32([0, n], dev), i32([at + n], dev), i32([0], dev),
                max_q_len=n)
            at += n
        last = y[-1].float().cpu()
        assert abs(float(last[0]) - want0) < 0.02 * want0
        assert abs(float(last[1])) < 1e-6
        assert float(state[1].min()) == 5.0


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lens", [[65], [64, 1, 200], [129, 128, 63]])
def test_chunk_parallel_scans_equal_row_by_row(dtype, lens):
    """The chunk-parallel prefill of both recurrent mixers against the same
    kernels walking every row in order, with old state in the slots."""
    dev = "cuda"
    torch.manual_seed(sum(lens))
    T, S = sum(lens), len(lens)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    starts = [0, 7, 300][:S]
    seq_lens = [s + n for s, n in zip(starts, lens)]
    slots = [2, 0, 3][:S]
    meta = (i32(cu, dev), i32(seq_lens, dev), i32(slots, dev))
    chunks = ops.scan_chunks(lens, torch.device(dev))
    # lightning
    H, D, V = 3, 16, 24
    q, k, v = (torch.randn(T, H, n, device=dev).to(dtype) for n in (D, D, V))
    decay = torch.tensor([1.0, 0.97, 0.6], device=dev)
    st0 = torch.randn(4, H, D, V, device=dev)
    sa, sb = st0.clone(), st0.clone()
    a = ops.lightning_scan(q, k, v, decay, sa, *meta, max_q_len=max(lens))
    b = ops.lightning_scan(q, k, v, decay, sb, *meta, max_q_len=max(lens), chunks=chunks)
    assert torch.allclose(a, b, rtol=1e-4, atol=1e-4)
    assert torch.allclose(sa, sb, rtol=1e-4, atol=1e-4)
    # selective scan, with dt from a GEMM and projected in the kernel
    C, N, R = 40, 12, 5
    u = torch.randn(T, C, device=dev).to(dtype)
    dbc = torch.randn(T, R + 2 * N, device=dev).to(dtype)
    z = torch.randn(T, C, device=dev).to(dtype)
    dt_w = torch.randn(C, R, device=dev) * 0.3
    dt_b = torch.randn(C, device=dev) - 1.0
    A = -torch.rand(C, N, device=dev) * 2
    Dp = torch.randn(C, device=dev)
    st0 = torch.randn(4, C, N, device=dev)
    dt_pre = dbc[:, :R].float() @ dt_w.t()
    outs = []
    for kw in ({}, {"chunks": chunks}, {"dt_pre": dt_pre, "chunks": chunks}):
        st = st0.clone()
        y = ops.selective_scan(u, dbc, z, dt_w, dt_b, A, Dp, st, *meta,
                               max_q_len=max(lens), **kw)
        outs.append((y.float(), st))
    tol = 2e-2 if dtype == torch.bfloat16 else 2e-4
    for y, st in outs[1:]:
        assert torch.allclose(y, outs[0][0], rtol=tol, atol=tol)
        assert torch.allclose(st, outs[0][1], rtol=1e-4, atol=1e-4)


@pytest.mark.gpu
@pytest.mark.parametrize("D,V", [(32, 32), (64, 64), (64, 128), (128, 64), (128, 128)])
def test_lightning_matrix_core_prefill_equals_general_kernel(D, V):
    """bf16 rows, head sizes the matrix-core kernels are built for: chunk
    ends of 1, 63, 64 and 65 rows, decays 1, 0 and in between, old state."""
    dev = "cuda"
    torch.manual_seed(D + V)
    lens = [65, 129, 200, 64]
    T, H = sum(lens), 4
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    starts = [0, 9, 500, 0]
    meta = (i32(cu, dev), i32([s + n for s, n in zip(starts, lens)], dev),
            i32([1, 3, 0, 2], dev))
    chunks = ops.scan_chunks(lens, torch.device(dev))
    q, k, v = (torch.randn(T, H, n, device=dev).to(torch.bfloat16) for n in (D, D, V))
    decay = torch.tensor([1.0, 0.0, 0.9, 0.999], device=dev)
    st0 = torch.randn(4, H, D, V, device=dev)
    res = {}
    for flag in (False, True):
        ops.use_lightning_mfma = flag
        try:
            st = st0.clone()
            o = ops.lightning_scan(q, k, v, decay, st, *meta, max_q_len=max(lens),
                                   chunks=chunks)
        finally:
            ops.use_lightning_mfma = True
        res[flag] = (o, st)
    scale = res[False][0].abs().max()
    assert (res[True][0] - res[False][0]).abs().max() < 1e-2 * scale
    sscale = res[False][1].abs().max()
    assert (res[True][1] - res[False][1]).abs().max() < 1e-2 * sscale


def _scan64(u, dbc, z, dt_w, dt_b, A, Dp, st, R):
    """One sequence, row by row in float64; (y, state, bound of |y|)."""
    u, dbc, z, dt_w, dt_b, A, Dp, st = (
        t.double().cpu() for t in (u, dbc, z, dt_w, dt_b, A, Dp, st))
    N = A.shape[1]
    dt = torch.nn.functional.softplus(dbc[:, :R] @ dt_w.t() + dt_b, threshold=1e9)
    ys, mag, sm = [], [], st.abs()
    for t in range(len(u)):
        e = torch.exp(dt[t][:, None] * A)
        dx = (dt[t] * u[t])[:, None] * dbc[t, R:R + N]
        st, sm = e * st + dx, e * sm + dx.abs()
        c = dbc[t, R + N:]
        g = z[t] * torch.sigmoid(z[t])
        ys.append(((st * c).sum(1) + Dp * u[t]) * g)
        mag.append(((sm * c.abs()).sum(1) + (Dp * u[t]).abs()) * g.abs())
    return torch.stack(ys), st, torch.stack(mag), sm


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("C,N,lens", [
    (8, 16, [1]),               # whole states, one row
    (257, 16, [1, 64, 3]),      # a second workgroup with one channel
    (300, 8, [65, 129]),        # chunks with a last row of one
    (256, 32, [70]), (40, 64, [66]),
    (129, 12, [1, 67]),         # fewer states than lanes hold
    (33, 5, [64, 2])])
def test_selective_scan_lanes_against_64_bits(C, N, lens, dtype):
    """dt from a product, old states, and dt arguments from far below zero to
    far above. A row's decay and step have a relative error of some 2^-23
    (|argument of exp| < 88 at most counts, times 2^-24), and the rows add
    theirs up; bf16 outputs are rounded once more."""
    dev = "cuda"
    torch.manual_seed(C + N)
    T, S, R = sum(lens), len(lens), 4
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    meta = (i32(cu, dev), i32([n + 5 for n in lens], dev),
            i32(list(range(S))[::-1], dev))
    u = torch.randn(T, C, device=dev).to(dtype)
    dbc = torch.randn(T, R + 2 * N, device=dev).to(dtype)
    z = (torch.randn(T, C, device=dev) * 4).to(dtype)
    z[0, :4] = torch.tensor([-200.0, 200.0, -90.0, 0.0], device=dev).to(dtype)
    dt_w = torch.randn(C, R, device=dev) * 0.3
    dt_b = torch.linspace(-120.0, 6.0, C, device=dev)
    dt_b[1::2] = torch.linspace(-3.0, 3.0, C, device=dev)[1::2]
    A = -torch.rand(C, N, device=dev) * 2
    Dp = torch.randn(C, device=dev)
    st0 = torch.randn(S + 1, C, N, device=dev)
    dt_pre = (dbc[:, :R].double() @ dt_w.double().t()).float()
    st = st0.clone()
    y = ops.selective_scan(u, dbc, z, dt_w, dt_b, A, Dp, st, *meta,
                           max_q_len=max(lens), dt_pre=dt_pre,
                           chunks=ops.scan_chunks(lens, torch.device(dev)))
    assert torch.equal(st[S], st0[S])
    for i, n in enumerate(lens):
        a, b, slot = cu[i], cu[i + 1], S - 1 - i
        want, wst, mag, sm = _scan64(u[a:b], dbc[a:b], z[a:b], dt_w, dt_b, A, Dp,
                                     st0[slot], R)
        # a step's argument carries dt_pre + dt_b's rounding: up to 2^-24 * 120
        rel = 2.0 ** -24 * (160 + 16 * n)
        assert bool(((st[slot].double().cpu() - wst).abs() <= rel * sm + 1e-30).all())
        tol = (rel + (2.0 ** -8 if dtype == torch.bfloat16 else 0.0)) * mag + 1e-30
        assert bool(((y[a:b].double().cpu() - want).abs() <= tol).all())


@pytest.mark.gpu
@pytest.mark.parametrize("C,N", [(4096, 16), (4097, 5)])
def test_selective_scan_gate_of_bf16_rows(C, N):
    """The gate of bf16 rows is fp32 work, seen in how often its rounding to bf16
    is another one than that of the fp64 value. With C = 0 the output is D u
    silu(z): exp to 1 ulp, a sum, a quotient and two products, at most 3 * 2^-23
    of it in all, fall on the other side of a rounding border (2^-8 apart, or
    more) for at most 2 * 3 * 2^-23 / 2^-8 of the values. An argument of exp2
    that is rounded, at 64 and more by 2^-18, would do so for three times that."""
    dev = "cuda"
    torch.manual_seed(N)
    T, R = 128, 4
    z = -torch.linspace(45.0, 87.0, T, device=dev)[:, None].expand(T, C).bfloat16()
    u = torch.ones(T, C, device=dev).bfloat16()
    dbc = torch.zeros(T, R + 2 * N, device=dev).bfloat16()
    Dp = torch.rand(C, device=dev) + 1
    y = ops.selective_scan(
        u, dbc, z.contiguous(), torch.zeros(C, R, device=dev), torch.zeros(C, device=dev),
        -torch.rand(C, N, device=dev), Dp, torch.zeros(1, C, N, device=dev),
        i32([0, T], dev), i32([T], dev), i32([0], dev), max_q_len=T,
        dt_pre=torch.zeros(T, C, device=dev))
    want = (Dp.double() * torch.nn.functional.silu(z.double())).bfloat16()
    share = (y != want).double().mean().item()
    assert share <= 2 * 3 * 2.0 ** -23 / 2.0 ** -8, share


@pytest.mark.gpu
@pytest.mark.parametrize("D,V", [(16, 64), (128, 128), (256, 64),  # whole
                                 (128, 72), (100, 64), (17, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_lightning_rows_against_64_bits(D, V, dtype):
    """Rows walked one by one: states whole in a wave's registers and not, an
    old state, a fresh one and a padding row. A state value takes two
    operations a row and a sum of D terms: 2^-23 of the terms' size each."""
    dev = "cuda"
    torch.manual_seed(D + V)
    H, lens = 3, [1, 5, 1]
    T = sum(lens)
    q, k, v = (torch.randn(T, H, n, device=dev).to(dtype) for n in (D, D, V))
    decay = torch.tensor([1.0, 0.9, 0.0], device=dev)
    st0 = torch.randn(4, H, D, V, device=dev)
    st = st0.clone()
    o = ops.lightning_scan(q, k, v, decay, st, i32([0, 1, 6, 7], dev),
                           i32([9, 5, 4], dev), i32([2, 0, -1], dev), max_q_len=5)
    silu = lambda t: torch.nn.functional.silu(t.double())
    a, b, c, lam = silu(q), silu(k), silu(v), decay.double()[:, None, None]
    at = 0
    for n, slot, old in zip(lens, (2, 0, -1), (True, False, False)):
        S = st0[slot].double() if old else torch.zeros_like(st0[0]).double()
        M = S.abs()
        for t in range(at, at + n):
            kv = b[t][:, :, None] * c[t][:, None, :]
            S, M = lam * S + kv, lam * M + kv.abs()
            want = (S * a[t][:, :, None]).sum(1)
            tol = (M * a[t].abs()[:, :, None]).sum(1) * 2.0 ** -23 * (D + 16)
            assert bool(((o[t].double() - want).abs() <= tol + 1e-12).all())
        if slot >= 0:
            assert bool(((st[slot].double() - S).abs()
                         <= 2.0 ** -23 * 16 * M + 1e-12).all())
        at += n
    assert torch.equal(st[1], st0[1]) and torch.equal(st[3], st0[3])


@pytest.mark.gpu
@pytest.mark.parametrize("W", [4, 1024, 1028, 2052, 4096, 8192, 8196, 1030])
@pytest.mark.parametrize("gated", [False, True])
def test_rms_norm_of_float_rows_against_64_bits(W, gated):
    """Rows of every width class to bf16, plain and times a gate's sigmoid from
    strided rows, on 8 bytes and off them: one rounding (2^-9 either way) of a
    value with a relative error of some 2^-22."""
    dev, T = "cuda", 3
    torch.manual_seed(W)
    x = torch.randn(T, W, device=dev) * 5
    w = torch.randn(W, device=dev)
    want = x.double() * torch.rsqrt(x.double().pow(2).mean(1, keepdim=True) + 1e-5)
    want = want * w.double()
    if not gated:
        got = [ops.rms_norm_f32(x, w, 1e-5, torch.bfloat16)]
    else:
        buf = torch.randn(T, 2 * W + 9, device=dev).bfloat16()
        got, wants = [], []
        for gate in (buf[:, :W], buf[:, 1:W + 1], buf[:, :W].contiguous()):
            out = torch.empty(T, W, device=dev, dtype=torch.bfloat16)
            ops._native_seq().gated_rmsnorm(out, x, w, gate, 1e-5)
            got.append(out)
            wants.append(want * torch.sigmoid(gate.double()))
    for i, g in enumerate(got):
        ref = wants[i] if gated else want
        assert bool(((g.double() - ref).abs() <= (2.0 ** -8) * ref.abs() + 1e-30).all())


@pytest.mark.gpu
@pytest.mark.parametrize("D,V", [(64, 64), (128, 128)])
@pytest.mark.parametrize("n", [33, 65, 200, 700, 1100])
def test_masked_rows_merge_their_key_splits(D, V, n):
    """A row behind contexts that are cut in 1 to 16 runs, a full one among
    sequences of other lengths. The weights are rounded to bf16 (2^-9 of
    each term) and the result once more."""
    dev, G, H = "cuda", 2, 8
    torch.manual_seed(n)
    lens = [n, 1, n // 2 + 1]
    pages = -(-n // 16)
    kc = torch.randn(3 * pages, G, 16, D, device=dev).bfloat16()
    vc = torch.randn(3 * pages, G, 16, V, device=dev).bfloat16()
    table = torch.randperm(3 * pages).view(3, pages)
    q = torch.randn(3, H, D, device=dev).bfloat16()
    out = torch.empty(3, H, V, dtype=torch.bfloat16, device=dev)
    assert ops._native_seq().attention_masked_mfma(
        out, q, kc, vc, table.int().to(dev), i32(lens, dev), i32([0, 1, 2, 3], dev),
        i32([0, 1, 2], dev), D ** -0.5, None, 0.0, 0, 0, 1.0, False, 1)
    for i, L in enumerate(lens):
        k, v = (c[table[i].to(dev)].transpose(1, 2).reshape(-1, G, c.shape[3])[:L]
                .double().repeat_interleave(H // G, 1) for c in (kc, vc))
        p = torch.softmax((k * q[i].double()).sum(2) * D ** -0.5, 0)
        want = (p[:, :, None] * v).sum(0)
        tol = 2.0 ** -7 * (p[:, :, None] * v.abs()).sum(0)
        assert bool(((out[i].double() - want).abs() <= tol).all())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_head_norm_rotation_of_few_and_many_rows(dtype):
    """The same bits whether a row's heads are shared by several workgroups (up
    to 256 rows) or walked by one; turned values, a row without a page."""
    dev, T, H, G, D, V = "cuda", 300, 5, 3, 24, 40
    torch.manual_seed(1)
    q, k, v = (torch.randn(T, h, d, device=dev).to(dtype)
               for h, d in ((H, D), (G, D), (G, V)))
    qw, kw = torch.randn(2, D, device=dev)
    f, fv = torch.rand(10, device=dev), torch.rand(V // 2, device=dev)
    pos = torch.randint(0, 5000, (T,), device=dev)
    slots = torch.randperm(320, device=dev)[:T]
    slots[5] = -1
    res = []
    for cut in (T, 37):
        kc = torch.zeros(20, G, 16, D, device=dev, dtype=dtype)
        vc = torch.zeros(20, G, 16, V, device=dev, dtype=dtype)
        qo = torch.cat([ops.qk_norm_rope_cache(
            *(t[a:a + cut] for t in (q, k, v)), qw, kw.contiguous(), 1e-5,
            pos[a:a + cut], f, fv, kc, vc, slots[a:a + cut])
            for a in range(0, T, cut)])
        res.append((qo, kc, vc))
    for a, b in zip(*res):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("D,V", [(32, 32), (64, 64), (64, 128), (128, 64),
                                 (128, 128), (64, 32), (128, 32)])
def test_lightning_chunks_off_16_bytes(D, V):
    """Rows on 16 bytes are staged by wide loads, others one value at a time:
    the same bits. Chunk ends of one to 64 rows, odd ones among them."""
    dev, H, lens = "cuda", 3, [1, 64, 130, 35, 99]
    torch.manual_seed(D + V)
    T, cu = sum(lens), [0]
    for n in lens:
        cu.append(cu[-1] + n)
    meta = (i32(cu, dev), i32([n + 3 for n in lens], dev), i32([4, 1, 0, 2, 3], dev))
    chunks = ops.scan_chunks(lens, torch.device(dev))
    data = [torch.randn(T, H * n, device=dev).bfloat16() * 4 for n in (D, D, V)]
    decay = torch.tensor([1.0, 0.0, 0.98], device=dev)
    st0 = torch.randn(5, H, D, V, device=dev)
    res = []
    for pads in ((0, 0, 0), (8, 8, 8), (2, 0, 0), (0, 4, 0), (0, 0, 1)):
        rows = []
        for t, n, pad in zip(data, (D, D, V), pads):
            buf = torch.empty(T, H * n + pad, device=dev, dtype=torch.bfloat16)
            buf[:, :H * n] = t
            rows.append(buf[:, :H * n].view(T, H, n) if not pad
                        else buf.as_strided((T, H, n), (H * n + pad, n, 1)))
        st = st0.clone()
        o = ops.lightning_scan(*rows, decay, st, *meta, max_q_len=max(lens),
                               chunks=chunks)
        res.append((o, st))
    for o, st in res[1:]:
        assert torch.equal(o, res[0][0]) and torch.equal(st, res[0][1])


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 2, 8, 9, 16])
@pytest.mark.parametrize("E,top,ff,W", [(16, 4, 256, 512), (4, 1, 512, 1024),
                                        (64, 2, 256, 1536), (12, 12, 1024, 512)])
@pytest.mark.parametrize("act", ["product", "input", "clamped"])
def test_routed_experts_read_the_chosen_alone(rows, E, top, ff, W, act):
    """The chosen experts' weighted sum against float64, strided rows; the
    weights of experts that nobody chose are NaN, and no weight at all gives
    zeros. Projections, activation and result are each rounded to bf16, the
    activation turning 2^-8 of the gate into up to 4 of its own."""
    torch.manual_seed(rows + E)
    dev = "cuda"
    h = torch.randn(rows, 2 * W, device=dev).bfloat16()[:, :W]
    w_gu = (torch.randn(2 * E * ff, W, device=dev) * W ** -0.5).bfloat16()
    w_down = (torch.randn(W, E * ff, device=dev) * ff ** -0.5).bfloat16()
    scale = torch.zeros(rows, E, device=dev)
    ids = torch.randn(rows, E, device=dev).topk(top).indices
    scale.scatter_(1, ids, torch.rand(rows, top, device=dev) + 0.1)
    unused = (scale == 0).all(0)
    w_gu.view(E, 2 * ff, W)[unused] = math.nan
    w_down.view(W, E, ff)[:, unused] = math.nan
    assert ops.routed_takes(h, w_gu, w_down, E, ff)
    limit, alpha = 1.5, 1.7
    out = ops.routed_experts(
        h, w_gu, w_down, scale, act == "input",
        "clamped" if act == "clamped" else "swiglu", limit, alpha).double()
    expect = torch.zeros(rows, W, dtype=torch.float64, device=dev)
    slack = torch.zeros_like(expect)
    for e in range(E):
        if unused[e]:
            continue
        t = (scale[:, e] != 0).nonzero()[:, 0]
        s = scale[t, e].double()[:, None]
        g, u = (h[t].double() @ w_gu.view(E, 2, ff, W)[e].double().flatten(0, 1).t()
                ).split(ff, 1)
        if act == "clamped":
            g, u = g.clamp(max=limit), u.clamp(-limit, limit) + 1
            a = s * g * torch.sigmoid(alpha * g) * u
        elif act == "input":
            a = torch.nn.functional.silu(s * g) * s * u
        else:
            a = torch.nn.functional.silu(g) * s * u
        d = w_down.view(W, E, ff)[:, e].double()
        expect[t] += a @ d.t()
        near = a.abs() + s * (g.abs() + 1) * 2 ** -8  # where a factor is near 0
        slack[t] += 6 * 2 ** -8 * near @ d.abs().t()
    assert bool(((out - expect).abs() <= slack + 2 ** -8 * expect.abs()).all())
    scale.zero_()
    w_gu.nan_to_num_(0.5), w_down.nan_to_num_(0.5)
    assert not ops.routed_experts(h, w_gu, w_down, scale).any()


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,top,W,gate", [
    (1, 16, 4, 4096, False), (64, 64, 8, 2048, False), (5, 63, 32, 4104, True),
    (3, 1, 1, 8, False), (7, 5, 2, 520, True)])
@pytest.mark.parametrize("score", ["softmax", "sigmoid"])
def test_route_rows(T, E, top, W, gate, score):
    """Router product and routing against moe_route_grouped of logits in float64:
    ends of a row's pieces, every lane an expert, ties, a correction that decides;
    a row's choice does not turn with the rows beside it."""
    torch.manual_seed(E + W)
    dev = "cuda"
    h = torch.randn(T, 2 * W, device=dev).bfloat16()[:, :W]
    router = (torch.randn(E + gate, W, device=dev) * W ** -0.5).bfloat16()
    if E > 2:
        router[1] = router[0]  # equal scores: the lower index first
    bias = torch.randn(E, device=dev) * 0.1
    bias[:2] = 0.2
    corr = torch.randn(E, device=dev) * 0.05
    corr[:2] = 0.1
    assert ops.route_rows_takes(h, router) and not ops.route_rows_takes(h, router, 2)
    assert not ops.route_rows_takes(h.float(), router.float())
    z = (h.double() @ router.double().t()).float()
    for kw in ({}, dict(bias=bias), dict(bias=bias, correction=corr)):
        kw.update(score=score, shared_gate=gate)
        out = ops.moe_route_rows(h, router, top, matrix=True, **kw)
        want = ops.moe_route_grouped(z, top, matrix=True, **kw)
        # a logit is chains of 8 products, of a lane's W / 512 such and of 6 steps over
        # the lanes; the weights move by up to twice that much (renormed ones are
        # quotients), and by a dozen roundings of their own
        adds = 8 + -(-W // 512) + 6 + 1
        slack = 2 * adds * 2 ** -24 * (h.double().abs() @ router.double().abs().t()).max().item()
        for a, b in ((out[0], want[0]), (out[2], want[2])):
            assert (a - b).abs().max().item() <= slack + 1e-6
        assert torch.equal(out[1], want[1])
        for n in {1, T // 2} - {0}:
            for a, b in zip(ops.moe_route_rows(h[:n], router, top, matrix=True, **kw), out):
                assert torch.equal(a, b[:n])
    # rows that hold no numbers stay in bounds
    h = h.clone()
    h[0, 0] = float("nan")
    ids = ops.moe_route_rows(h, router, top)[1]
    assert ids.min() >= 0 and ids.max() < E + gate
    assert all(len(set(r)) == top for r in ids.tolist())


@pytest.mark.gpu
def test_route_rows_steps_aside(monkeypatch):
    """Rows under a transform, with gradients or tangents, or without the kernels, are
    left to the products that follow them."""
    h = torch.randn(3, 5, 256, device="cuda").bfloat16()
    router = torch.randn(16, 256, device="cuda").bfloat16()
    takes = []
    torch.vmap(lambda x: (takes.append(ops.route_rows_takes(x, router)), x)[1])(h)
    torch.vmap(lambda r: (takes.append(ops.route_rows_takes(h[0], r)), r)[1])(
        router.expand(3, -1, -1))
    takes.append(ops.route_rows_takes(h[0], router.clone().requires_grad_()))
    with torch.autograd.forward_ad.dual_level():
        takes.append(ops.route_rows_takes(h[0], router))
    assert takes == [False] * 4 and ops.route_rows_takes(h[0], router)
    monkeypatch.setattr(ops, "seq_native_available", lambda: False)
    assert not ops.route_rows_takes(h[0], router)


@pytest.mark.gpu
@pytest.mark.parametrize("E,top,ff,W,most", [
    (4, 2, 512, 1024, 48),     # weights of linear_fixed
    # larger: routed_experts up to 16 rows, linear_fixed's cut from 17 on
    (16, 4, 1024, 2560, 32)])
def test_routed_layer_order_of_sums(E, top, ff, W, most, monkeypatch):
    """A row's experts add up to the same bits whatever rows share its step; large
    weights have one order up to 16 rows and another from 17 on."""
    from arks_amd.models.feedforward import RoutedMoE

    torch.manual_seed(E)
    m = RoutedMoE(W, E, ff, top, torch.bfloat16, weigh="output").to("cuda")
    for p in m.parameters():
        torch.nn.init.normal_(p, std=p.shape[-1] ** -0.5)
    ops.fix_sums(m.parameters())
    h = torch.randn(most, W, device="cuda").bfloat16()
    scale = torch.zeros(most, E, device="cuda")
    scale.scatter_(1, torch.randn(most, E, device="cuda").topk(top).indices,
                   torch.rand(most, top, device="cuda") + 0.1)
    monkeypatch.setattr(ops, "moe_route_rows", lambda h, *a, **k: (
        None, None, scale[:h.shape[0]]))
    routed = ops.routed_experts
    took = []
    monkeypatch.setattr(ops, "routed_experts", lambda h, *a: (
        took.append(h.shape[0]), routed(h, *a))[1])
    with torch.no_grad():
        whole = m(h)
        few = m(h[:16])
        for T in (1, 2, 7, 8, 9, 15, 16, 17, 31, 33):
            if T <= most:
                want = few if E == 16 and T <= 16 else whole
                assert torch.equal(m(h[:T]), want[:T]), T
        assert E == 16 or torch.equal(few, whole[:16])
    err = (few.double() - whole[:16].double()).norm() / few.double().norm()
    assert err <= 2 ** -8  # a rounding of the activation and of the result apart
    assert took == ([] if E == 4 else [16, 1, 2, 7, 8, 9, 15, 16])


@pytest.mark.gpu
@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("T,E,top,W,ff,extra", [
    (1, 3, 1, 64, 64, 0), (300, 16, 4, 128, 192, 0), (257, 3, 2, 192, 64, 64),
    (700, 5, 1, 320, 576, 128), (33, 64, 16, 64, 320, 0), (2100, 9, 4, 64, 128, 8)])
def test_moe_wide_rows(T, E, top, W, ff, extra, scaled):
    """Experts in whole tiles against float64: strided rows, weights that hold
    more behind them, experts with 0, 1, 255, 256 and 257 rows, ends of the
    tiles. Projections, activation and result are each rounded to bf16."""
    torch.manual_seed(T)
    dev = "cuda"
    h = torch.randn(T, 2 * W, device=dev).bfloat16()[:, :W]
    w_gu = (torch.randn(2 * E * ff + 2 * extra, W, device=dev) * W ** -0.5).bfloat16()
    w_down = (torch.randn(W, E * ff + extra, device=dev) * ff ** -0.5).bfloat16()
    ids = torch.rand(T, E, device=dev).topk(top).indices.int()
    if E == 9:  # every row takes expert 8; the first choices are as below
        near = torch.repeat_interleave(
            torch.arange(4, device=dev), torch.tensor([1, 255, 256, 257], device=dev))
        ids[:] = torch.tensor([4, 5, 6, 8], device=dev)
        ids[:near.numel(), 0] = near.int()
    weights = torch.rand(T, top, device=dev) + 0.1
    assert ops.moe_wide_takes(h, w_gu, w_down, E, ff, top)
    y, place = ops.moe_wide_rows(h, w_gu, w_down, weights, ids, E, ff, scaled)
    assert sorted(place.flatten().tolist()) == list(range(T * top))
    for e in range(E):
        t, j = (ids == e).nonzero(as_tuple=True)
        s = weights[t, j].double()[:, None] if scaled else 1.0
        g, u = (h[t].double() @ w_gu[2 * e * ff:2 * (e + 1) * ff].double().t()
                ).split(ff, 1)
        a = torch.nn.functional.silu(s * g) * s * u
        d = w_down[:, e * ff:(e + 1) * ff].double()
        # a gate's or up's rounding (2^-9 of it; silu's slope is at most 1.1)
        # and the activation's own
        near = 2 ** -9 * ((1.1 * s * g.abs() + a.abs() / (s * u).abs().clamp(1e-9))
                          * (s * u).abs() + a.abs()) + 1e-6
        err = (y[place[t, j].long()].double() - a @ d.t()).abs()
        assert bool((err <= near @ d.abs().t() + 2 ** -8 * (a @ d.t()).abs() + 1e-6).all())


@pytest.mark.gpu
def test_moe_wide_rows_order_of_sums():
    """A pair's row has the same bits whatever rows share the prompt, in tiles of
    128 pairs and of 256."""
    torch.manual_seed(2)
    E, top, W, ff = 5, 2, 1024, 576
    h = torch.randn(2000, W, device="cuda").bfloat16()
    w_gu = (torch.randn(2 * E * ff, W, device="cuda") * W ** -0.5).bfloat16()
    w_down = (torch.randn(W, E * ff, device="cuda") * ff ** -0.5).bfloat16()
    ids = torch.rand(2000, E, device="cuda").topk(top).indices.int()
    weights = torch.rand(2000, top, device="cuda")
    rows = {}
    for T in (60, 257, 700, 2000):  # 24, 103, 280 and 800 pairs an expert
        y, place = ops.moe_wide_rows(h[:T], w_gu, w_down, weights[:T], ids[:T], E, ff)
        rows[T] = y[place[:60].long()]
        assert torch.equal(rows[T], rows[60]), T


@pytest.mark.gpu
def test_moe_wide_rows_are_the_layers():
    """A layer's prompt rows through the tiles and through one product per
    expert: the same sums up to their order."""
    from arks_amd.models.feedforward import RoutedMoE

    torch.manual_seed(1)
    for weigh, shared in (("input", 0), ("output", 0), ("output", 64)):
        m = RoutedMoE(256, 8, 192, 2, torch.bfloat16, shared_ff=shared,
                      weigh=weigh).to("cuda")
        for p in m.parameters():
            torch.nn.init.normal_(p, std=256 ** -0.5)
        h = torch.randn(400, 256, device="cuda").bfloat16()
        with torch.no_grad():
            assert ops.moe_wide_takes(h, m.w_gu, m.w_down, m.E, m.ff, m.top)
            out, takes = m(h).double(), ops.moe_wide_takes
            ops.moe_wide_takes = lambda *a: False
            try:
                other = m(h).double()
            finally:
                ops.moe_wide_takes = takes
        assert (out - other).norm() <= 2 ** -8 * other.norm()
