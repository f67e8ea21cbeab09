"""Products over several activation rows (gemm.hip) against float64 products
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
                                   (33, 64, 1024), (64, 65, 640), (65, 31, 2080), (80, 300, 256), (200, 96, 1408)])
def test_rows_product_edges(rina, orc, qt, M, N, K):
    """Every row tile and its successor, K of 1 .. 65 blocks (whole and partial
    128-value steps, Q2_K rows that start inside pages), odd column counts."""
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
def test_rows_product_magnitudes(rina, orc, qt):
    """Every row is held to its own scale: rows of 1e-30 .. 1e30 (one of
    zeros), and rows whose values span 2^40.  The f16 split of a row keeps 22
    bits of each value down to 2^-16 of the row's maximum and an absolute
    2^-39 of it below, so the error stays under 1e-5 of sum |w x|."""
    r = rng(qt)
    M, N, K = 24, 48, 512
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
    assert np.all(np.abs(got - ref) <= 1e-5 * scale + 1e-45)


@pytest.mark.parametrize("qt", [5, 7, 10])
def test_rows_product_nonfinite(rina, orc, qt):
    """inf and NaN stay in their rows: Q4 rows give fp32's results (inf where
    the weight is not zero, NaN where it is), Q2_K rows are not finite."""
    r = rng(qt + 50)
    M, N, K = 20, 32, 256
    w, W = weights(orc, qt, r, N * K)
    x = r.standard_normal((M, K)).astype(np.float32)
    x[3, 77], x[7, 5], x[18, 200] = np.inf, np.nan, -np.inf
    got = product(rina, w, qt, x, N, K)
    W = W.reshape(N, K)
    with np.errstate(invalid="ignore"):
        ref = np.stack([(W * xr).sum(1) for xr in x.astype(np.float64)])
    fine = [m for m in range(M) if m not in (3, 7, 18)]
    assert_close(got[fine], ref[fine], what="finite rows")
    assert not np.isfinite(got[[3, 7, 18]]).any()
    if qt != 10:
        assert np.array_equal(np.isnan(got[[3, 18]]), np.isnan(ref[[3, 18]]))
        m = ~np.isnan(ref[[3, 18]])
        assert np.array_equal(got[[3, 18]][m], ref[[3, 18]][m].astype(np.float32))


def test_rows_product_under_capture(rina, orc):
    """A first product captured into a graph (its scratch is allocated during
    the capture), replayed with other work between, equals the eager result."""
    import torch
    r = rng(9)
    M, N, K = 300, 96, 3200
    w, W = weights(orc, 7, r, N * K)
    x = r.standard_normal((M, K)).astype(np.float32)
    hip, wd, xd, y = rina.load_hip(), dev(w), dev(x), empty(M * N)
    seg = rina.LinearSeg(wd.data_ptr(), None, y.data_ptr(), N)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        ok(hip.rina_hip_linear_fused(C.byref(seg), 1, 7, xd.data_ptr(), M, K, 0, 0, None, 0.0, s.cuda_stream), "captured")
    ref = x.astype(np.float64) @ W.reshape(N, K).T
    for k in range(3):
        y.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert_close(host(y).reshape(M, N), ref, what="replay %d" % k)
