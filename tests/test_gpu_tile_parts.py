"""Two-part tiles: one head per wave, the even and the odd 32-token chunks of a
tile on two waves, joined in LDS. The prefill launchers' implicit tiles in each
heads-per-workgroup variant (2, 4, 6, 8), around the range that stays one part
(256 tokens), with ragged last tiles and pages that 16-token halves straddle;
split tiles and verify blocks of 5-6 heads at every head_dim that has two parts;
and invalid pages in an even or an odd chunk. All against the fp32 oracle.
Joining adds three fp32 roundings (2^-24 each) to values whose bound is set by
the 11 and 16 mantissa bits of P: the tiles' tolerances hold unchanged."""
import ctypes as C

import numpy as np
import pytest
import torch

import phaseshift_amd as P
from phaseshift_amd import ops, state
from tests.kvcase import INVALID, REL_TILE, assert_attention_close, bf16_normal, paged_layout, to_dev
from tests.test_gpu_paged_attention import TOL, make_pools, oracle_out
from tests.test_gpu_psq import REL as PSQ_REL
from tests.test_gpu_psq import TOL as PSQ_TOL
from tests.test_gpu_psq import dev_pools, geom_of, oracle_attn, prefill_rows_case, run_attn
from tests.test_gpu_tiles import run_tile, tile_case

pytestmark = pytest.mark.gpu

KV = {"bf16": P.KV_BF16, "fp8": P.KV_FP8, "psq4": P.KV_PSQ4, "psq8": P.KV_PSQ8}
ALL = ("bf16", "fp8", "psq4", "psq8")


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


# Split tiles that run in two parts (tests/test_tile_parts.py holds the rule to
# it): formats, q heads, kv heads, head_dim, page, contexts of the 16-row blocks,
# splits, pages per split.
SPLIT_CASES = [
    (ALL, 24, 4, 256, 16, [2000, 1200], 4, 33),    # 528 tokens a split, a one-part last split
    (ALL, 24, 4, 256, 16, [2000, 1200], 2, 64),
    (ALL, 20, 4, 256, 16, [2000, 700], 4, 33),     # 5 heads: the sixth wave pair is empty
    (ALL, 24, 4, 256, 24, [2000, 1400], 3, 29),    # 16-token halves straddle pages
    (ALL, 24, 4, 128, 16, [2000, 1300], 3, 48),
    (ALL, 10, 2, 128, 16, [1500, 1300], 2, 48),
    (("bf16", "fp8"), 24, 4, 64, 16, [2000, 1300], 3, 48),
    (("bf16",), 24, 4, 32, 16, [2000, 1300], 3, 48),
    (ALL, 24, 4, 256, 16, [1300] * 17, 64, 40),    # 17 tiles x 64 splits: past the dense units, the plain grid
]


def blocks_case(dev, kv, qh, kvh, D, page, lens, seed):
    """16-row blocks, block i the last 16 tokens of sequence i (context lens[i])."""
    rng = np.random.default_rng(seed)
    lay = paged_layout(rng, lens, page, kvh, D, spare_pages=2)
    pools = dev_pools(lay, int(kv[3]), dev, seed=seed) if kv.startswith("psq") else make_pools(lay, kv == "fp8", seed, dev)
    slots = np.repeat(np.arange(len(lens), dtype=np.uint32), 16)
    pos = np.concatenate([np.arange(n - 16, n, dtype=np.uint32) for n in lens])
    return lay, pools, slots, pos, bf16_normal(rng, (len(slots), qh * D))


def oracle_blocks(lay, kv, qh, q, slots, pos, bt, pools):
    if kv.startswith("psq"):
        return oracle_attn(lay, int(kv[3]), qh, q, slots, pos, bt, pools)
    return oracle_out(lay, qh, q, slots, pos, bt, *pools)


def close_kv(got, want, kv, what):
    if kv.startswith("psq"):
        assert_attention_close(got, want, PSQ_TOL, PSQ_REL, what)
    else:
        assert_attention_close(got, want, TOL[kv == "fp8"], REL_TILE[kv == "fp8"], what)


def run_blocks(dev, lay, kv, qh, q, slots, pos, bt, pools, splits, pps):
    """psk_attention_paged_tile_split and its combine over implicit tiles."""
    out = torch.full((q.shape[0], qh * lay.head_dim), 7.0, dtype=torch.float32, device=dev)
    part = torch.empty(ops.split_partials_bytes(q.shape[0], qh, lay.kv_heads, splits) // 4, device=dev)
    dq, ds, dp, dbt = to_dev(q), to_dev(slots), to_dev(pos), to_dev(bt)
    a = ops.attention_args(geom_of(lay), 0, dq, out, ds, dp, dbt, qh)
    L = P.lib()
    P.check("tile_split", L.psk_attention_paged_tile_split(
        C.byref(a), KV[kv], *(None if t is None else t.data_ptr() for t in pools), part.data_ptr(), splits, pps, None))
    P.check("reduce", L.psk_attention_paged_split_reduce_ex(C.byref(a), part.data_ptr(), splits, pps, None))
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("kv,case", [(kv, c[1:]) for c in SPLIT_CASES for kv in c[0]])
def test_two_part_split_tiles(dev, kv, case):
    qh, kvh, D, page, lens, splits, pps = case
    lay, pools, slots, pos, q = blocks_case(dev, kv, qh, kvh, D, page, lens, qh + D + pps)
    want = oracle_blocks(lay, kv, qh, q, slots, pos, lay.block_tables, pools)
    got = run_blocks(dev, lay, kv, qh, q, slots, pos, lay.block_tables, pools, splits, pps)
    close_kv(got, want, kv, f"test_gpu_tile_parts 3 {kv} {case}")


@pytest.mark.parametrize("kv,qh,D", [(kv, qh, D) for qh, D in ((24, 256), (20, 256), (24, 128), (24, 64))
                                     for kv in ("bf16", "fp8")] + [("bf16", 24, 32)])
def test_two_part_verify_blocks(dev, kv, qh, D):
    """Unsplit verify blocks past 320 tokens through the step planner."""
    lens = [700, 330, 1500]
    lay, pools, slots, pos, q = blocks_case(dev, kv, qh, 4, D, 16, lens, qh + D)
    out = torch.full((48, qh * D), 7.0, dtype=torch.float32, device=dev)
    dq, ds, dp, dbt = to_dev(q), to_dev(slots), to_dev(pos), to_dev(lay.block_tables)
    a = ops.attention_args(geom_of(lay), 0, dq, out, ds, dp, dbt, qh)
    reqs = [(16 * i, 16, 1, n) for i, n in enumerate(lens)]
    plan = state.plan_step(a, KV[kv], reqs, max(lens), 0, None, *pools, launch=True)
    torch.cuda.synchronize()
    assert [k.kind for k in plan.kernels[:plan.count]] == [1] and plan.kernels[0].splits == 1
    want = oracle_blocks(lay, kv, qh, q, slots, pos, lay.block_tables, pools)
    close_kv(out.cpu().numpy(), want, kv, f"test_gpu_tile_parts 4 {kv} {qh} {D}")


@pytest.mark.parametrize("kv", ALL)
@pytest.mark.parametrize("page", [26, 28, 29])   # in chunk 13 (odd); in chunk 14, first and second half
def test_invalid_page_of_either_part(dev, kv, page):
    """Rows whose tile meets an invalid page stay unwritten, whichever part
    would read it; the tiles and blocks that do not meet it are exact."""
    qh, D = 24, 256
    rng = np.random.default_rng(page)
    # implicit tiles at 304, 320, ...: the page begins one
    lay = paged_layout(rng, [304 + 200], 16, 4, D, spare_pages=2)
    pools = dev_pools(lay, int(kv[3]), dev, seed=page) if kv.startswith("psq") else make_pools(lay, kv == "fp8", page, dev)
    bt = lay.block_tables.copy()
    bt[0, page] = INVALID
    slots, pos = np.zeros(200, np.uint32), np.arange(304, 504, dtype=np.uint32)
    q = bf16_normal(rng, (200, qh * D))
    if kv.startswith("psq"):
        got = run_attn(dev, lay, int(kv[3]), qh, q, slots, pos, bt, pools, kind="prefill")
    else:
        lay.block_tables = bt
        got = run_tile(lay, qh, q, slots, pos, *pools)
    n = 16 * page - 304
    assert np.all(got[n:] == 7.0)
    want = oracle_blocks(lay, kv, qh, q[:n], slots[:n], pos[:n], bt, pools)
    close_kv(got[:n], want, kv, f"test_gpu_tile_parts 5 {kv} {page}")

    # split blocks: the first one's first split meets it
    lay, pools, slots, pos, q = blocks_case(dev, kv, qh, 4, D, 16, [2000, 1200], page)
    bt = lay.block_tables.copy()
    bt[0, page] = INVALID
    got = run_blocks(dev, lay, kv, qh, q, slots, pos, bt, pools, 2, 64)
    assert np.all(got[:16] == 7.0)
    want = oracle_blocks(lay, kv, qh, q[16:], slots[16:], pos[16:], bt, pools)
    close_kv(got[16:], want, kv, f"test_gpu_tile_parts 6 {kv} {page}")
