"""Two-part tiles (the prefill launchers' implicit tiles): one head per wave, the
even and the odd 32-token chunks of a tile on two waves, joined in LDS. Each
heads-per-workgroup variant (2, 4, 6, 8), around the range that stays one part
(256 tokens), with ragged last tiles and pages that 16-token halves straddle,
against the fp32 oracle. Joining adds three fp32 roundings (2^-24 each) to
values whose bound is set by the 11 and 16 mantissa bits of P: the tiles'
tolerances hold unchanged."""
import pytest

from tests.kvcase import REL_TILE, assert_attention_close
from tests.test_gpu_paged_attention import TOL, oracle_out
from tests.test_gpu_psq import REL as PSQ_REL
from tests.test_gpu_psq import TOL as PSQ_TOL
from tests.test_gpu_psq import oracle_attn, prefill_rows_case, run_attn
from tests.test_gpu_tiles import run_tile, tile_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv", ["bf16", "fp8", "psq4", "psq8"])
@pytest.mark.parametrize("qh,kvh,D,page,prefix,rows", [
    (24, 4, 256, 16, 239, 17),    # 256 tokens: one part; 2 heads a workgroup
    (24, 4, 256, 16, 240, 17),    # 257 tokens: the last tile has two parts
    (24, 4, 256, 16, 300, 200),   # 2 heads (PSQ 4, the last workgroup 2 of them)
    (24, 4, 256, 24, 700, 500),   # 4 heads, straddling pages
    (20, 4, 256, 16, 90, 520),    # 5 heads on 6
    (16, 2, 128, 16, 40, 1040),   # 8 heads
    (4, 4, 128, 16, 280, 33),     # 1 head, few rows: one part
    (4, 4, 128, 16, 280, 300),    # 1 head on 2
    (32, 4, 256, 16, 300, 100),   # 8 heads at 256: workgroups of 2 or 4
])
def test_two_part_tiles(dev, kv, qh, kvh, D, page, prefix, rows):
    seed = qh + D + rows
    if kv.startswith("psq"):
        fmt = int(kv[3])
        lay, pools, slots, pos, q = prefill_rows_case(dev, fmt, qh, kvh, D, page, prefix, rows, seed=seed)
        want = oracle_attn(lay, fmt, qh, q, slots, pos, lay.block_tables, pools)
        got = run_attn(dev, lay, fmt, qh, q, slots, pos, lay.block_tables, pools, kind="prefill")
        assert_attention_close(got, want, PSQ_TOL, PSQ_REL, "test_gpu_tile_parts 1")
        return
    fp8 = kv == "fp8"
    lay, kp, vp, ks, vs, q, slots, pos = tile_case(seed, prefix, rows, qh, kvh, D, fp8, dev, P_=page)
    want = oracle_out(lay, qh, q, slots, pos, lay.block_tables, kp, vp, ks, vs)
    got = run_tile(lay, qh, q, slots, pos, kp, vp, ks, vs)
    assert_attention_close(got, want, TOL[fp8], REL_TILE[fp8], "test_gpu_tile_parts 2")
