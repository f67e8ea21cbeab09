"""Products over several activation rows (gemm.hip, gemm_bf3.hip) against float64 products
of the dequantized weights, at the edges of their tiles: 16 / 32 / 64-row
tiles and one row past each, K of one block up to steps and windows with
remainders, column counts off the tile, unaligned rows, rows of very
different magnitudes, and rows that hold inf or NaN."""
import ctypes as C
import importlib

import numpy as np
import pytest

from _util import assert_close, dev, empty, host, ok, rng, stream

pytestmark = pytest.mark.gpu


def weights(orc, qt, r, n):
    if qt == 6:
        w = (r.standard_normal(n) * 0.02).astype(np.float32)
        return w, w.astype(np.float64)
    if qt == 10:
        w = importlib.import_module("rina_amd.synth").random_q2k(int(r.integers(1 << 30)), n)
    else:
        w = orc.pack(qt, (r.standard_normal(n) * 0.02).astype(np.float32))
    return w, orc.dequant(qt, w, n).astype(np.float64)


def product(rina, w, qt, x, N, K, epi=0, w2=None, y0=None, off=0):
    """x [M, K] through rina_hip_linear_fused; off: floats the rows start past a 16-byte boundary."""
    M = x.shape[0]
    buf = np.zeros(M * K + 4, np.float32)
    buf[off:off + M * K] = x.reshape(-1)
    y = dev(y0) if y0 is not None else empty(M * N)
    seg = rina.LinearSeg(dev(w).data_ptr(), dev(w2).data_ptr() if w2 is not None else None, y.data_ptr(), N)
    ok(rina.load_hip().rina_hip_linear_fused(C.byref(seg), 1, qt, dev(buf).data_ptr() + 4 * off, M, K, epi, 0, None, 0.0,
                                             stream()), "product")
    return host(y).reshape(M, N)


@pytest.mark.parametrize("qt", [5, 7, 10, 6])
@pytest.mark.parametrize("M,N,K", [(2, 16, 32), (15, 33, 96), (16, 40, 128), (17, 100, 160), (31, 17, 512), (32, 130, 544),
                                   (33, 64, 1024), (64, 65, 640), (65, 31, 2080), (80, 300, 256), (200, 96, 1408),
                                   (15, 200, 320), (16, 200, 320), (97, 130, 512), (97, 130, 544), (129, 8000, 640),
                                   (120, 8000, 640), (130, 1100, 8192)])
def test_rows_product_edges(rina, orc, qt, M, N, K):
    """Every row tile and its successor, K of 1 .. 65 blocks (whole and partial
    128-value steps, Q2_K rows that start inside pages), odd column counts; for
    Q4 weights both sides of the lines between one launch and two (16 rows, K
    512, outputs against K squared) and between 32- and 64-row tiles."""
    r = rng(M * 3 + N + K + qt)
    w, W = weights(orc, qt, r, N * K)
    x = r.standard_normal((M, K)).astype(np.float32)
    got = product(rina, w, qt, x, N, K)
    # largest fp32 sum here: 2080 terms, error below 2080 * 2^-24 of the sum of magnitudes
    assert_close(got, x.astype(np.float64) @ W.reshape(N, K).T, what="rows q%d %s" % (qt, (M, N, K)))


@pytest.mark.parametrize("qt", [5, 7, 10])
@pytest.mark.parametrize("M,off", [(5, 1), (40, 2), (70, 3)])
def test_rows_product_unaligned_and_epilogues(rina, orc, qt, M, off):
    """Rows at 4-byte alignment; residual add and SiLU * up on the same rows."""
    r = rng(M + off + qt)
    N, K = 72, 416
    w, W = weights(orc, qt, r, N * K)
    w2, W2 = weights(orc, qt, r, N * K)
    x = r.standard_normal((M, K)).astype(np.float32)
    y0 = r.standard_normal((M, N)).astype(np.float32)
    g, u = (x.astype(np.float64) @ m.reshape(N, K).T for m in (W, W2))
    assert_close(product(rina, w, qt, x, N, K, epi=1, y0=y0, off=off), y0 + g, what="add")
    assert_close(product(rina, w, qt, x, N, K, epi=2, w2=w2, off=off), g / (1 + np.exp(-g)) * u, what="swiglu")


@pytest.mark.parametrize("qt", [5, 7, 10])
@pytest.mark.parametrize("K", [512, 640])
def test_rows_product_magnitudes(rina, orc, qt, K):
    """Every row is held to its own scale: rows of 1e-30 .. 1e30 (one of
    zeros), and rows whose values span 2^40: the sums of exact products stay
    within 1e-6 of sum |w x| (chains of at most 20 blocks of 32)."""
    r = rng(qt)
    M, N = 24, 48
    w, W = weights(orc, qt, r, N * K)
    x = r.standard_normal((M, K))
    x[:12] *= (10.0 ** np.linspace(-30, 30, 12))[:, None]
    x[12] = 0.0
    x[13:] *= 2.0 ** r.integers(-40, 1, (M - 13, K))
    x = x.astype(np.float32)
    got = product(rina, w, qt, x, N, K).astype(np.float64)
    W = W.reshape(N, K)
    ref, scale = x.astype(np.float64) @ W.T, np.abs(x.astype(np.float64)) @ np.abs(W.T)
    assert np.all(got[12] == 0)
    assert np.all(np.abs(got - ref) <= 1e-6 * scale + 1e-45)


@pytest.mark.parametrize("qt", [5, 7, 10])
@pytest.mark.parametrize("M,K", [(5, 480), (24, 480), (24, 672), (70, 672)])
def test_rows_product_outlier_facing_zero_weights(rina, orc, qt, M, K):
    """A value 2^12 .. 2^60 times the others whose weights are zero adds
    nothing: the product of the others is as close as without it.  fp32 sums in
    chains of at most 21 blocks of 32: below 1e-6 of sum |w x|."""
    r = rng(qt + M)
    N, at = 48, 37
    w, _ = weights(orc, qt, r, N * K)
    if qt == 10:                             # scale and minimum of the group of 16 that holds it
        g = (np.arange(N) * K + at) // 16
        w = w.reshape(-1, 84).copy()
        w[g // 16, g % 16] = 0
        w = w.reshape(-1)
    else:
        wf = (r.standard_normal((N, K)) * 0.02).astype(np.float32)
        wf[:, at] = 0
        w = orc.pack(qt, wf.reshape(-1))
    W = orc.dequant(qt, w, N * K).astype(np.float64).reshape(N, K)
    assert not W[:, at].any()
    x = r.standard_normal((M, K)).astype(np.float32)
    x[:, at] = (2.0 ** np.linspace(12, 60, M)).astype(np.float32)
    got = product(rina, w, qt, x, N, K).astype(np.float64)
    x[:, at] = 0
    ref, scale = x.astype(np.float64) @ W.T, np.abs(x.astype(np.float64)) @ np.abs(W.T)
    assert np.all(np.abs(got - ref) <= 1e-6 * scale)


@pytest.mark.parametrize("qt", [5, 7, 10])
@pytest.mark.parametrize("M,K", [(20, 256), (20, 416), (70, 256), (70, 416), (20, 640), (70, 672), (300, 640)])
def test_rows_product_nonfinite(rina, orc, qt, M, K):
    """inf and NaN stay in their rows, and rows that hold them give what the
    fp32 products give: an infinity of the weight's sign, NaN where the weight
    is zero, the row holds NaN or infinities of both signs meet."""
    r = rng(qt + 50)
    N = 100
    w, W = weights(orc, qt, r, N * K)
    x = r.standard_normal((M, K)).astype(np.float32)
    x[3, 77], x[7, 5], x[18, 200], x[11, 64], x[11, 65] = np.inf, np.nan, -np.inf, np.inf, -np.inf
    got = product(rina, w, qt, x, N, K)
    W = W.reshape(N, K)
    with np.errstate(invalid="ignore"):
        ref = np.stack([(W * xr).sum(1) for xr in x.astype(np.float64)])
    bad = [3, 7, 11, 18]
    fine = [m for m in range(M) if m not in bad]
    assert_close(got[fine], ref[fine], what="finite rows")
    assert not np.isfinite(ref[bad]).any()
    assert np.array_equal(got[bad], ref[bad].astype(np.float32), equal_nan=True)


@pytest.mark.parametrize("qt", [10])
@pytest.mark.parametrize("M,epi", [(12, 1), (40, 1), (12, 2), (40, 2)])
def test_rows_product_nonfinite_epilogues(rina, orc, qt, M, epi):
    """The same through the residual add (the infinity stays) and SiLU * up."""
    r = rng(qt + M + epi)
    N, K = 40, 288
    w, W = weights(orc, qt, r, N * K)
    w2, W2 = weights(orc, qt, r, N * K)
    x = r.standard_normal((M, K)).astype(np.float32)
    x[4, 99] = np.inf
    y0 = r.standard_normal((M, N)).astype(np.float32)
    got = product(rina, w, qt, x, N, K, epi=epi, w2=w2 if epi == 2 else None, y0=y0 if epi == 1 else None)
    with np.errstate(invalid="ignore", over="ignore"):
        g, u = ((m.reshape(N, K)[None] * x.astype(np.float64)[:, None]).sum(2) for m in (W, W2))
        ref = y0 + g if epi == 1 else g / (1 + np.exp(-g)) * u
    fine = np.arange(M) != 4
    assert_close(got[fine], ref[fine], what="finite rows")
    assert np.array_equal(got[4], ref[4].astype(np.float32), equal_nan=True)


def test_rows_product_under_capture(rina, orc):
    """A first product captured into a graph (its scratch is allocated during
    the capture), replayed with larger eager products on the capture stream
    between (they overwrite and grow the stream's scratch), equals the eager
    result."""
    import torch
    r = rng(9)
    M, N, K = 300, 96, 3200
    w, W = weights(orc, 7, r, N * K)
    x = r.standard_normal((M, K)).astype(np.float32)
    hip, wd, xd, y = rina.load_hip(), dev(w), dev(x), empty(M * N)
    seg = rina.LinearSeg(wd.data_ptr(), None, y.data_ptr(), N)
    big, yb = dev(r.standard_normal((4 * M, K)).astype(np.float32)), empty(4 * M * N)
    segb = rina.LinearSeg(wd.data_ptr(), None, yb.data_ptr(), N)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        ok(hip.rina_hip_linear_fused(C.byref(seg), 1, 7, xd.data_ptr(), M, K, 0, 0, None, 0.0, s.cuda_stream), "captured")
    ref = x.astype(np.float64) @ W.reshape(N, K).T
    for k in range(4):
        y.zero_()
        ok(hip.rina_hip_linear_fused(C.byref(segb), 1, 7, big.data_ptr(), (k + 1) * M, K, 0, 0, None, 0.0, s.cuda_stream), "eager")
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert_close(host(y).reshape(M, N), ref, what="replay %d" % k)


@pytest.mark.parametrize("qt", [7, 10])
def test_graphs_of_one_capture_stream_replayed_on_two(rina, orc, qt):
    """Two graphs captured on one stream and replayed on two others, beside
    eager products on the capture stream: every product has its own rows (the
    same bits as alone)."""
    import torch
    hip, M, N, K = rina.load_hip(), 40, 64, 2048
    w, _ = weights(orc, qt, rng(qt), N * K)
    wd = dev(w)
    xs = [dev(rng(s).standard_normal((M, K)).astype(np.float32)) for s in range(3)]
    alone = [empty(M * N) for _ in xs]
    n = 60
    ys = [[empty(M * N) for _ in range(n)] for _ in xs]

    def call(i, y, st):
        seg = rina.LinearSeg(wd.data_ptr(), None, y.data_ptr(), N)
        ok(hip.rina_hip_linear_fused(C.byref(seg), 1, qt, xs[i].data_ptr(), M, K, 0, 0, None, 0.0, st.cuda_stream), "product")

    cap, s1, s2 = (torch.cuda.Stream() for _ in range(3))
    torch.cuda.synchronize()
    for i in range(3):
        call(i, alone[i], cap)
    torch.cuda.synchronize()
    graphs = [torch.cuda.CUDAGraph() for _ in range(2)]
    for i, g in enumerate(graphs):
        with torch.cuda.graph(g, stream=cap):
            for y in ys[i]:
                call(i, y, cap)
    for k in range(5):
        for i in (0, 1):
            for y in ys[i]:
                y.zero_()
        torch.cuda.synchronize()
        for g, s in zip(graphs, (s1, s2)):
            with torch.cuda.stream(s):
                g.replay()
        for y in ys[2]:
            call(2, y, cap)
        torch.cuda.synchronize()
        for i in range(3):
            assert all(torch.equal(y, alone[i]) for y in ys[i]), "replay %d, rows %d" % (k, i)


def test_scratch_of_graphs_goes_back(rina, orc):
    """Graphs captured and destroyed one after the other: what their captures
    allocated (the split rows of 1024 x 8192: 48 MB and more) goes back."""
    import gc

    import torch
    hip, M, N, K = rina.load_hip(), 1024, 32, 8192
    w, _ = weights(orc, 7, rng(3), N * K)
    wd, xd, y = dev(w), dev(rng(4).standard_normal((M, K)).astype(np.float32)), empty(M * N)
    seg = rina.LinearSeg(wd.data_ptr(), None, y.data_ptr(), N)
    s = torch.cuda.Stream()

    def call():
        ok(hip.rina_hip_linear_fused(C.byref(seg), 1, 7, xd.data_ptr(), M, K, 0, 0, None, 0.0, s.cuda_stream), "product")

    call()
    torch.cuda.synchronize()
    want = y.clone()
    low = []
    for k in range(24):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            call()
        y.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        del g
        gc.collect()
        call()
        torch.cuda.synchronize()
        low.append(torch.cuda.mem_get_info()[0])
    assert low[-1] > low[3] - 5 * M * K * 4     # far less than the 20 buffers of the captures between


def test_scratch_of_ended_threads(rina, orc):
    """Threads on their own default streams (hipStreamPerThread), one after the
    other without a synchronization between: a new thread's split rows are
    never written over those of one that ended, and what ended threads held
    (48 MB and more each) goes back."""
    import threading

    import torch
    hip, M, N, K, per_thread = rina.load_hip(), 1024, 32, 8192, 2
    w, _ = weights(orc, 7, rng(5), N * K)
    wd = dev(w)
    xs = [dev(rng(s).standard_normal((M, K)).astype(np.float32)) for s in range(2)]
    n = 24
    ys = [empty(M * N) for _ in range(n)]
    rcs = []
    low = []

    def call(k):
        seg = rina.LinearSeg(wd.data_ptr(), None, ys[k].data_ptr(), N)
        rcs.append(hip.rina_hip_linear_fused(C.byref(seg), 1, 7, xs[k % 2].data_ptr(), M, K, 0, 0, None, 0.0, per_thread))

    torch.cuda.synchronize()
    for k in range(n):
        t = threading.Thread(target=call, args=(k,))
        t.start()
        t.join()
        low.append(torch.cuda.mem_get_info()[0])
    torch.cuda.synchronize()
    assert rcs == [0] * n
    for k in range(2, n):
        assert torch.equal(ys[k], ys[k % 2])
    assert not torch.equal(ys[0], ys[1])
    assert low[-1] > low[3] - 5 * M * K * 4


@pytest.mark.parametrize("qt", [7, 10, 6])
@pytest.mark.parametrize("T,E,k,d,F,S", [(150, 4, 2, 256, 96, 128), (61, 8, 3, 128, 160, 0), (5, 16, 4, 256, 64, 64)])
def test_moe_rows_groups(rina, orc, qt, T, E, k, d, F, S):
    """The MoE block over rows grouped by expert against float64: groups of
    more than one 64-row tile, of 16-row tiles, an expert no row selects (its
    router row loses everywhere), no shared experts; a row of NaN selects
    nothing and leaves the other rows alone."""
    hip = rina.load_hip()
    r = rng(T + E + d + qt)
    ex = {n: [weights(orc, qt, r, F * d) for _ in range(E)] for n in ("g", "u", "dn")}
    packed = {n: np.concatenate([w for w, _ in ex[n]]) for n in ex}
    sh = [weights(orc, qt, r, S * d) for _ in range(3)] if S else [(None, None)] * 3
    wr = (r.standard_normal((E, d)) * 0.2).astype(np.float32)
    ln2 = r.uniform(0.8, 1.2, d).astype(np.float32)
    h0 = (r.standard_normal((T, d)) * 2).astype(np.float32)
    h0[:, 0] = 40.0                          # a common component that expert E - 1's router row opposes
    wr[E - 1, 0] = -20.0
    bad = T // 2
    h0[bad, 3] = np.nan
    hd = dev(h0)
    keep = [dev(x) for x in (ln2, wr, packed["g"], packed["u"], packed["dn"])]
    shd = [dev(w) if S else None for w, _ in sh]
    ptr = [x.data_ptr() if x is not None else None for x in shd]
    sb = packed["g"].nbytes // E
    wb = hip.rina_hip_moe_rows_workspace(T, d, E, k, F, S)
    ws = empty(wb // 4 + 4)
    ok(hip.rina_hip_moe_rows(hd.data_ptr(), T, keep[0].data_ptr(), np.float32(1e-5), keep[1].data_ptr(), 6, *ptr, S, qt,
                             keep[2].data_ptr(), keep[3].data_ptr(), keep[4].data_ptr(), qt, sb, packed["dn"].nbytes // E,
                             E, k, d, F, ws.data_ptr(), wb, stream()), "moe rows")
    got = host(hd).reshape(T, d)

    def silu(v):
        return v / (1 + np.exp(-v))

    h = h0.astype(np.float64)
    seen = 0
    for t in range(T):
        if t == bad:
            continue
        a = h[t] / np.sqrt((h[t] ** 2).mean() + 1e-5) * ln2
        lg = wr.astype(np.float64) @ a
        p = np.exp(lg - lg.max())
        p /= p.sum()
        order = np.argsort(-p, kind="stable")
        assert E - 1 not in order[:k]
        if p[order[k - 1]] - p[order[k]] < 1e-5:
            continue                         # a tie the fp32 router may break the other way
        ref = h[t].copy()
        if S:
            G, U, D = (W for _, W in sh)
            ref += D.reshape(d, S) @ (silu(G.reshape(S, d) @ a) * (U.reshape(S, d) @ a))
        for e in order[:k]:
            g, u = (ex[n][e][1].reshape(F, d) @ a for n in ("g", "u"))
            ref += p[e] * (ex["dn"][e][1].reshape(d, F) @ (silu(g) * u))
        assert_close(got[t], ref, what="row %d" % t)
        seen += 1
    assert seen >= T * 3 // 4


@pytest.mark.parametrize("qt,M", [(7, 16), (10, 40)])
def test_rows_product_two_threads_one_stream(rina, orc, qt, M):
    """Two host threads on one stream, each with rows of its own: the split
    rows of one call are never another's (the products repeat bit for bit)."""
    import threading

    import torch

    hip, N, K, st = rina.load_hip(), 64, 256, stream()
    w, _ = weights(orc, qt, rng(qt), N * K)
    wd = dev(w)
    xs = [dev(rng(s).standard_normal((M, K)).astype(np.float32)) for s in (1, 2)]
    ys = [[empty(M * N) for _ in range(300)] for _ in xs]
    rcs = [[], []]

    def calls(i, n0, n1):
        for y in ys[i][n0:n1]:
            seg = rina.LinearSeg(wd.data_ptr(), None, y.data_ptr(), N)
            rcs[i].append(hip.rina_hip_linear_fused(C.byref(seg), 1, qt, xs[i].data_ptr(), M, K, 0, 0, None, 0.0, st))

    for i in (0, 1):
        calls(i, 0, 1)                      # alone: the expected products
    ts = [threading.Thread(target=calls, args=(i, 1, 300)) for i in (0, 1)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    torch.cuda.synchronize()
    for i in (0, 1):
        assert rcs[i] == [0] * 300
        assert all(torch.equal(y, ys[i][0]) for y in ys[i])
    assert not torch.equal(ys[0][0], ys[1][0])


@pytest.mark.parametrize("qt", [7, 10, 6])
@pytest.mark.parametrize("M,K,pro", [(2, 2176, 1), (20, 4160, 2), (33, 8320, 1), (3, 12416, 1), (18, 12416, 2), (40, 256, 1)])
def test_rows_product_norm_prologue(rina, orc, qt, M, K, pro):
    """RMSNorm / LayerNorm fused into the split of rows of every register
    count, and of rows longer than the registers hold (past 12288)."""
    r = rng(M + K + qt)
    N = 40
    w, W = weights(orc, qt, r, N * K)
    x = (r.standard_normal((M, K)) + (0.5 if pro == 2 else 0.0)).astype(np.float32)
    nw = r.uniform(0.8, 1.2, K).astype(np.float32)
    y = empty(M * N)
    seg = rina.LinearSeg(dev(w).data_ptr(), None, y.data_ptr(), N)
    ok(rina.load_hip().rina_hip_linear_fused(C.byref(seg), 1, qt, dev(x).data_ptr(), M, K, 0, pro, dev(nw).data_ptr(),
                                             np.float32(1e-5), stream()), "product")
    a = x.astype(np.float64)
    if pro == 2:
        a = a - a.mean(1, keepdims=True)
    a = a / np.sqrt((a ** 2).mean(1, keepdims=True) + 1e-5) * nw
    assert_close(host(y).reshape(M, N), a @ W.reshape(N, K).T, what="norm + rows")


@pytest.mark.parametrize("qt", [7, 10])
def test_moe_rows_workspace_or_scratch(rina, orc, qt):
    """A workspace that only holds the one-expert-at-a-time form (T k (2 d + F)
    floats and the head) is taken as before, the grouped rows then in library
    scratch: the same bits as with rina_hip_moe_rows_workspace() bytes, of which
    nothing past the end is written; a little less is refused."""
    hip, T, E, k, d, F = rina.load_hip(), 45, 8, 3, 128, 96
    r = rng(qt)
    w = [dev(weights(orc, qt, r, E * F * d)[0]) for _ in range(3)]
    wr, ln2 = dev((r.standard_normal((E, d)) * 0.3).astype(np.float32)), dev(np.ones(d, np.float32))
    h0 = r.standard_normal((T, d)).astype(np.float32)
    sb = w[0].numel() * w[0].element_size() // E
    up = lambda n: (n + 3) // 4 * 4
    least = 4 * (up(T * d) + up(T * E) + 4 * up(T * k) + 2 * up(T * k * d) + up(T * k * F))
    full = hip.rina_hip_moe_rows_workspace(T, d, E, k, F, 0)
    assert full >= least

    def call(nbytes):
        ws, h = dev(np.full(nbytes + 4096, 0xA5, np.uint8)), dev(h0)
        rc = hip.rina_hip_moe_rows(h.data_ptr(), T, ln2.data_ptr(), np.float32(1e-5), wr.data_ptr(), 6, None, None, None, 0, qt,
                                   w[0].data_ptr(), w[1].data_ptr(), w[2].data_ptr(), qt, sb, sb, E, k, d, F, ws.data_ptr(),
                                   nbytes, stream())
        assert (host(ws)[nbytes:] == 0xA5).all()
        return rc, host(h)

    rc0, a = call(full)
    rc1, b = call(least)
    assert rc0 == rc1 == 0 and np.array_equal(a, b) and not np.array_equal(a.reshape(T, d), h0)
    assert call(least - 4)[0] == -6          # RINA_ERR_WORKSPACE
