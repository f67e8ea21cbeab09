"""Attention of several query rows (attn_rows.hip) where its tiles end: row
tiles of 16 per wave and 16 / 32 / 64 per workgroup with 1, 2 or 4 query
heads sharing a KV head, key blocks of 64 with the cache / current-row border
inside one, key ranges split over workgroups (few rows over a long cache),
device positions, raw (pre-RoPE) cached keys, RINA-MLA widths off the tile."""
import pytest

from _util import assert_close_elem
from test_gpu_jamba import test_dq_prompt_attention_kv_matches_decode_rows as dq_rows_case
from test_gpu_kernels import attention_case

pytestmark = pytest.mark.gpu


# the oracle adds the positions one by one in fp32 and renormalizes at each:
# contexts stay below 700, where its own error is under the tolerance
@pytest.mark.parametrize("mode", [0, 1, 2, 3, 4, 5])
@pytest.mark.parametrize("P,T,H,Hkv", [(1, 2, 32, 8), (63, 17, 8, 8), (64, 16, 8, 4), (65, 33, 6, 2), (600, 3, 4, 1),
                                       (200, 65, 16, 8), (0, 70, 10, 5)])
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
                                                      (65, 63, 10, 5, 64, 64, 5), (33, 1, 8, 2, 48, 22, 0)])
def test_dq_rows_other_widths(rina, T, start, H, Hkv, da, db, mode):
    dq_rows_case(rina, T, start, H, Hkv, da, db, mode)
