"""Dense units of split decode launches around the 64 rows up to which each wave
finds them by itself: 1, 63, 64 and 65 rows of 1 to 700 tokens, rows of an
invalid slot among them (left unwritten), against the fp32 oracle. The search
moves no arithmetic: the decode tolerances hold as they are."""
import numpy as np
import pytest

from tests.kvcase import REL_DECODE, assert_attention_close
from tests.test_gpu_paged_attention import TOL, case, oracle_out, run_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("rows,pps", [(1, 3), (63, 5), (64, 1), (64, 44), (65, 5)])
def test_units_around_one_wave(dev, fp8, rows, pps):
    rng = np.random.default_rng(rows + pps)
    lens = [1, 700] + [int(x) for x in rng.integers(1, 701, 63)] if rows > 1 else [700]
    lens = lens[:rows]
    _, lay, kp, vp, ks, vs, q, slots, pos = case(rows + fp8, lens, 8, 4, 128, 16, fp8, dev)
    bad = [2, rows - 1] if rows > 2 else []
    sl = slots.copy()
    sl[bad] = 1 << 20
    splits = (max(lens) + 16 * pps - 1) // (16 * pps)
    got = run_gpu(lay, 8, q, sl, pos, lay.block_tables, kp, vp, ks, vs, splits=max(splits, 2),
                  pages_per_split=pps)
    assert np.all(got[bad] == 7.0)
    keep = [i for i in range(rows) if i not in bad]
    want = oracle_out(lay, 8, q[keep], slots[keep], pos[keep], lay.block_tables, kp, vp, ks, vs)
    assert_attention_close(got[keep], want, TOL[fp8], REL_DECODE, "test_gpu_decode_wave_units 1")
