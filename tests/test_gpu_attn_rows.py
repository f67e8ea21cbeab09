"""Attention of several query rows (attn_rows.hip) where its tiles end: row
tiles of 16 per wave and 16 / 32 / 64 per workgroup with 1, 2 or 4 query
heads sharing a KV head, key blocks of 64 with the cache / current-row border
inside one, key ranges split over workgroups (few rows over a long cache),
device positions, raw (pre-RoPE) cached keys, RINA-MLA widths off the tile,
values that are not finite in rows a query row does not see."""
import numpy as np
import pytest

from _util import assert_close_elem, dev, empty, host, ok, rng, stream
from test_gpu_jamba import test_dq_prompt_attention_kv_matches_decode_rows as dq_rows_case
from test_gpu_kernels import attention_case

pytestmark = pytest.mark.gpu


# the oracle adds the positions one by one in fp32 and renormalizes at each:
# contexts stay below 700, where its own error is under the tolerance
@pytest.mark.parametrize("mode", [0, 1, 2, 3, 4, 5])
@pytest.mark.parametrize("P,T,H,Hkv", [(1, 2, 32, 8), (63, 17, 8, 8), (64, 16, 8, 4), (65, 33, 6, 2), (600, 3, 4, 1),
                                       (200, 65, 16, 8), (0, 70, 10, 5), (0, 12, 16, 8), (0, 13, 10, 5)])
def test_rows_continue_a_cache(rina, orc, mode, P, T, H, Hkv):
    got, ref = attention_case(rina, orc, mode, P, T, H=H, Hkv=Hkv)
    assert_close_elem(got, ref, what="mode %d P %d T %d H %d/%d" % (mode, P, T, H, Hkv))


@pytest.mark.parametrize("mode,P,T", [(0, 130, 1), (1, 500, 1), (2, 70, 19), (5, 300, 5)])
def test_rows_pre_rope_cache(rina, orc, mode, P, T):
    got, ref = attention_case(rina, orc, mode, P, T, pre_rope=1)
    assert_close_elem(got, ref, what="pre-RoPE mode %d P %d T %d" % (mode, P, T))


@pytest.mark.parametrize("mode,P,T", [(0, 40, 3), (1, 333, 20)])
def test_rows_device_position(rina, orc, mode, P, T):
    got, ref = attention_case(rina, orc, mode, P, T, use_dpos=True)
    assert_close_elem(got, ref, what="device position mode %d P %d T %d" % (mode, P, T))


@pytest.mark.parametrize("T,start,H,Hkv,da,db,mode", [(63, 1, 10, 5, 64, 32, 0), (2, 63, 10, 5, 64, 16, 5), (17, 400, 3, 3, 80, 34, 0), (5, 700, 6, 2, 64, 10, 5),
                                                      (65, 63, 10, 5, 64, 64, 5), (33, 1, 8, 2, 48, 22, 0),
                                                      (2, 254, 10, 5, 64, 32, 5), (2, 255, 10, 5, 64, 32, 0)])
def test_dq_rows_other_widths(rina, T, start, H, Hkv, da, db, mode):
    dq_rows_case(rina, T, start, H, Hkv, da, db, mode)


def earlier_rows(call, T, bad, dim, after=True):
    """call(value): the rows' outputs [T, width] with `value` in dim `dim` of
    row `bad`'s value row.  A row sees the values up to its own position: with
    inf or NaN there, the rows before stay what they are, and the row itself and
    (after: they read the value itself, not a packed record) the rows after it
    are not finite in that dim."""
    want = call(0.5)
    assert np.isfinite(want).all()
    for value in (np.inf, np.nan):
        got = call(value)
        for t in range(bad):
            assert_close_elem(got[t], want[t], what="row %d of %d before a row with %s" % (t, T, value))
        assert not np.isfinite(got[bad:T if after else bad + 1, dim]).any()


@pytest.mark.parametrize("mode", [0, 1, 5])
@pytest.mark.parametrize("P,T,H,Hkv,bad", [(100, 40, 32, 8, 21), (0, 70, 8, 4, 65), (30, 130, 4, 4, 33), (500, 3, 8, 2, 2)])
def test_rows_before_a_non_finite_value(rina, orc, mode, P, T, H, Hkv, bad):
    hip, kvd = rina.load_hip(), Hkv * 64
    r = rng(P + T + mode)
    max_seq = P + T
    q, kcur, vcur = (r.standard_normal((T, w)).astype(np.float32) for w in (H * 64, kvd, kvd))
    kc, vc = (r.standard_normal((max_seq, kvd)).astype(np.float32) for _ in range(2))
    kf, vf = orc.kv_mode_formats(mode) if mode else (None, None)
    ck, cv = (dev(kc), dev(vc)) if mode == 0 else (dev(orc.kv_quantize(kf, kc)), dev(orc.kv_quantize(vf, vc)))
    ws_bytes = hip.rina_hip_gqa_attention_workspace(T, H, 64, max_seq)
    ws, qd, kd = empty(ws_bytes, "uint8"), dev(q), dev(kcur)
    dim = 37

    def call(value):
        v = vcur.copy()
        v[bad, (Hkv - 1) * 64 + dim] = value
        k = kd
        if np.isnan(value):                  # and its key
            kn = kcur.copy()
            kn[bad] = np.nan
            k = dev(kn)
        od = empty(T * H * 64)
        ok(hip.rina_hip_gqa_attention(qd.data_ptr(), k.data_ptr(), dev(v).data_ptr(), ck.data_ptr(), cv.data_ptr(), mode, 0,
                                      None, None, T, H, Hkv, 64, P, None, max_seq, od.data_ptr(), ws.data_ptr(), ws_bytes,
                                      stream()), "attention")
        return host(od).reshape(T, -1)

    earlier_rows(call, T, bad, (H - 1) * 64 + dim)


@pytest.mark.parametrize("mode", [0, 5])
@pytest.mark.parametrize("start,T,bad", [(0, 100, 50), (40, 30, 27), (300, 20, 7)])
def test_dq_rows_before_a_non_finite_value(rina, mode, start, T, bad):
    """RINA-MLA rows (10 / 5 heads, 64 + 32), also where the per-row kernel
    and the tiles meet (64 positions)."""
    hip, H, Hkv, da, db, dv = rina.load_hip(), 10, 5, 64, 32, 64
    r = rng(start + T + mode)
    max_seq = start + T
    qa, qb, ka, kb, v0 = (dev(r.standard_normal((T, w)).astype(np.float32)) for w in (H * da, H * db, Hkv * da, Hkv * db, Hkv * dv))
    before = [dev(r.standard_normal((start + 1, w)).astype(np.float32)) for w in (Hkv * da, Hkv * db, Hkv * dv)]
    sizes = [hip.rina_hip_dq_kv_region_bytes(mode, part, max_seq, Hkv, da, db, dv) for part in range(3)]
    dim = 37

    def rows(c, k1, k2, v, at, n, out):
        ok(hip.rina_hip_dq_prompt_attention_kv(qa.data_ptr(), qb.data_ptr(), k1.data_ptr(), k2.data_ptr(), v.data_ptr(), None,
                                               None, None, None, mode, c[0].data_ptr(), c[1].data_ptr(),
                                               c[2].data_ptr() if sizes[2] else None, H, Hkv, da, db, dv, at, n, max_seq,
                                               out.data_ptr(), stream()), "rows")

    def call(value):
        c = [empty(max(s, 4), "uint8") for s in sizes]
        for at in range(0, start, T):        # the rows before
            n = min(T, start - at)
            k1, k2, v = (dev(host(x)[at:at + n]) for x in before)
            rows(c, k1, k2, v, at, n, empty(n * H * dv))
        v = host(v0).copy()
        v[bad, (Hkv - 1) * dv + dim] = value
        out = empty(T * H * dv)
        rows(c, ka, kb, dev(v), start, T, out)
        return host(out).reshape(T, -1)

    earlier_rows(call, T, bad, (H - 1) * dv + dim, after=mode == 0)


@pytest.mark.parametrize("T,bad", [(40, 17), (300, 200)])
def test_mla_rows_before_a_non_finite_row(rina, orc, T, bad):
    """The latent prompt at the DeepSeek-V2 head shape: a latent row of NaN
    (its keys and values are NaN) and the rows before it."""
    hip, H, nope, rope, vd, dc = rina.load_hip(), 4, 128, 64, 128, 512
    r = rng(T)
    q = dev(r.standard_normal((T, H * (nope + rope))).astype(np.float32))
    kva = r.standard_normal((T, dc + rope)).astype(np.float32)
    w = dev(orc.pack(7, (r.standard_normal(H * (nope + vd) * dc) * 0.05).astype(np.float32)))
    norm, cache = dev(np.ones(dc, np.float32)), empty(T * (dc + rope))
    cd, sd = (dev(f(np.outer(np.arange(T), 0.1 ** np.arange(rope // 2))).astype(np.float32)) for f in (np.cos, np.sin))
    wsb = hip.rina_hip_mla_prompt_workspace(T, H, nope, rope, vd, dc)
    ws = empty(wsb, "uint8")

    def call(value):
        x = kva.copy()
        x[bad, 3] = value
        out = empty(T * H * vd)
        ok(hip.rina_hip_mla_prompt_attention(q.data_ptr(), dev(x).data_ptr(), norm.data_ptr(), np.float32(1e-5), cd.data_ptr(),
                                             sd.data_ptr(), w.data_ptr(), 7, cache.data_ptr(), H, nope, rope, vd, dc, T, T,
                                             out.data_ptr(), ws.data_ptr(), wsb, stream()), "latent prompt")
        return host(out).reshape(T, -1)

    earlier_rows(call, T, bad, 5)


@pytest.mark.parametrize("mode,P,T,H,Hkv", [(0, 0, 70, 8, 4), (0, 33, 20, 8, 2), (1, 0, 70, 32, 8), (1, 80, 5, 4, 4)])
@pytest.mark.parametrize("off", [1, 2, 3])
def test_rows_at_4_byte_alignment(rina, orc, mode, P, T, H, Hkv, off):
    """Query, key, value and output rows (and an fp32 cache) that start `off`
    floats past a 16-byte boundary: the same bits as aligned ones."""
    hip, kvd, max_seq = rina.load_hip(), Hkv * 64, P + T
    r = rng(P + T + mode)
    rows = [r.standard_normal(n * w).astype(np.float32) for n, w in ((T, H * 64), (T, kvd), (T, kvd))]
    kv = [r.standard_normal((max_seq, kvd)).astype(np.float32) for _ in range(2)]
    if mode:
        cache = [dev(orc.kv_quantize(f, x)) for f, x in zip(orc.kv_mode_formats(mode), kv)]

    def at(x, o):
        return dev(np.concatenate([np.zeros(o, np.float32), x.reshape(-1)])).data_ptr() + 4 * o

    def call(o):
        q, k, v = (at(x, o) for x in rows)
        ck, cv = (c.data_ptr() for c in cache) if mode else (at(x, o) for x in kv)
        out = empty(o + T * H * 64)
        ok(hip.rina_hip_gqa_attention(q, k, v, ck, cv, mode, 0, None, None, T, H, Hkv, 64, P, None, max_seq,
                                      out.data_ptr() + 4 * o, None, 0, stream()), "attention")
        return host(out)[o:]

    assert np.array_equal(call(off), call(0))
