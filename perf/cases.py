"""What a serving engine asks of this library, as cases that can be timed.

The engine (a paged-KV continuous-batching server for qwen35-style GQA models)
appends each step's new K/V rows to its pages and then attends: one-token
decode rows, speculative-verify blocks, prompt chunks, or all of them in one
step. KV is held as BF16, FP8 E4M3 (one f32 scale per token and head), PSQ8 or
PSQ4 (one bf16 scale per 32 values). Head geometry: 24 query / 4 KV heads of
256 with pages of 16 tokens, and the other GQA groups and head sizes that the
tests use.

A case is a dict of plain values; its context lengths follow from `lens_seed`,
its contents (K, V, Q, page order) from the seed given to `prepare`.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from phaseshift_amd import KV_BF16, KV_FP8, KV_PSQ4, KV_PSQ8, ops, state

KV = {"bf16": KV_BF16, "fp8": KV_FP8, "psq4": KV_PSQ4, "psq8": KV_PSQ8}
DECODE, VERIFY, PREFILL = 0, 1, 2
QWEN = {"q_heads": 24, "kv_heads": 4, "head_dim": 256, "page": 16}
WORKSPACE_BYTES = 256 << 20   # split-K workspace the engine keeps
DRAW_MAX_BYTES = 4.0e9
DRAW_MAX_FLOPS = 0.9e12


def listed():
    return [
        # one user's chat, a token at a time: latency and launches
        {"name": "decode_fp8_b1", "op": "decode", "kv": "fp8", **QWEN, "rows": 1, "ctx_lo": 4099, "ctx_hi": 4099,
         "lens_seed": 1, "out": "bf16"},
        # an ordinary decode batch, ragged contexts
        {"name": "decode_fp8_b16", "op": "decode", "kv": "fp8", **QWEN, "rows": 16, "ctx_lo": 500, "ctx_hi": 8000,
         "lens_seed": 2, "out": "bf16"},
        # a full decode batch of long contexts: the largest call
        {"name": "decode_fp8_b64_32k", "op": "decode", "kv": "fp8", **QWEN, "rows": 64, "ctx_lo": 32768,
         "ctx_hi": 32768, "lens_seed": 3, "out": "bf16"},
        # decode over unquantized KV, contexts 1k to 32k
        {"name": "decode_bf16_b32", "op": "decode", "kv": "bf16", **QWEN, "rows": 32, "ctx_lo": 1024, "ctx_hi": 32768,
         "lens_seed": 4, "out": "f32"},
        # decode over 4-bit KV
        {"name": "decode_psq4_b24", "op": "decode", "kv": "psq4", **QWEN, "rows": 24, "ctx_lo": 2048, "ctx_hi": 16384,
         "lens_seed": 5, "out": "f32"},
        # chunked prefill: 512-token chunks of eight prompts in one planned step
        {"name": "prefill_fp8_chunks", "op": "prefill", "api": "step", "kv": "fp8", **QWEN, "requests": 8,
         "chunk": 512, "ctx_lo": 2048, "ctx_hi": 16384, "lens_seed": 6, "out": "bf16"},
        # one fresh prompt of an odd length, one launch
        {"name": "prefill_bf16_prompt", "op": "prefill", "api": "launcher", "kv": "bf16", **QWEN, "requests": 1,
         "chunk": 2039, "ctx_lo": 0, "ctx_hi": 0, "lens_seed": 7, "out": "f32"},
        # prompts that continue cached prefixes, 8-bit block-scaled KV, a launch each
        {"name": "prefill_psq8_suffix", "op": "prefill", "api": "launcher", "kv": "psq8", **QWEN, "requests": 2,
         "chunk": 1000, "ctx_lo": 2048, "ctx_hi": 6144, "lens_seed": 8, "out": "bf16"},
        # speculative verification of 16-token drafts
        {"name": "verify_fp8_8x16", "op": "verify", "kv": "fp8", **QWEN, "blocks": 8, "draft": 16, "ctx_lo": 2048,
         "ctx_hi": 16384, "lens_seed": 9, "out": "bf16"},
        # one new token for each of 128 sequences
        {"name": "append_fp8_128", "op": "append", "kv": "fp8", **QWEN, "seqs": 128, "count": 1, "pos_lo": 0,
         "pos_hi": 32767, "lens_seed": 10, "estimator": 0},
        # a prefill step's rows into 4-bit pages, least-squares scales
        {"name": "append_psq4_16k", "op": "append", "kv": "psq4", **QWEN, "seqs": 16, "count": 1024, "pos_lo": 0,
         "pos_hi": 15000, "lens_seed": 11, "estimator": 1},
        # continuous batching: append, attention of every class, copy of shared prefix pages
        {"name": "step_fp8_mixed", "op": "step", "kv": "fp8", **QWEN, "requests": 8, "chunk": 512, "rows": 48,
         "blocks": 8, "draft": 16, "ctx_lo": 2048, "ctx_hi": 16384, "lens_seed": 12, "copies": 32, "out": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    """One more case of the ranges the listed ones stand for."""
    while True:
        geo = dict(rng.choice([QWEN, QWEN, QWEN,
                               {"q_heads": 16, "kv_heads": 4, "head_dim": 256, "page": 16},
                               {"q_heads": 16, "kv_heads": 2, "head_dim": 128, "page": 16},
                               {"q_heads": 24, "kv_heads": 4, "head_dim": 256, "page": 32}]))
        case = {"op": rng.choice(["decode", "decode", "decode", "prefill", "prefill", "verify", "append", "append",
                                  "step"]),
                "kv": rng.choice(["fp8", "fp8", "bf16", "psq4", "psq8"]), **geo,
                "lens_seed": rng.randrange(1, 1 << 30)}
        op = case["op"]
        if op != "append":
            case["out"] = rng.choice(["bf16", "f32"])
            case["ctx_lo"] = _log_int(rng, 256, 16384)
            case["ctx_hi"] = min(32768, int(case["ctx_lo"] * rng.uniform(1.0, 6.0)))
        if op == "decode":
            case["rows"] = _log_int(rng, 1, 64)
        elif op == "prefill":
            case["api"] = rng.choice(["step", "launcher"])
            case["requests"] = rng.randint(1, 8)
            case["chunk"] = _log_int(rng, 48, 2048)
            if rng.random() < 0.3:
                case["ctx_lo"] = case["ctx_hi"] = 0
        elif op == "verify":
            case["blocks"] = _log_int(rng, 1, 32)
            case["draft"] = rng.randint(4, 16)
        elif op == "append":
            case["estimator"] = rng.randint(0, 1) if case["kv"] in ("psq4", "psq8") else 0
            case["pos_lo"] = 0
            case["pos_hi"] = _log_int(rng, 1024, 32768)
            if rng.random() < 0.5:
                case["seqs"], case["count"] = _log_int(rng, 1, 256), 1
            else:
                case["seqs"], case["count"] = rng.randint(1, 16), _log_int(rng, 64, 4096)
        else:
            case["kv"] = rng.choice(["fp8", "bf16"])   # the one-launch metadata + append
            case["requests"] = rng.randint(1, 6)
            case["chunk"] = _log_int(rng, 128, 512)
            case["rows"] = _log_int(rng, 4, 48)
            case["blocks"] = rng.randint(0, 8)
            case["draft"] = rng.randint(8, 16)
            case["copies"] = rng.randint(1, 32)
        w = work(case)
        if w["bytes"] <= DRAW_MAX_BYTES and w["flops"] <= DRAW_MAX_FLOPS:
            return case


# ------------------------------------------------------------------ geometry
def _requests(case):
    """[(class, tokens before the rows, rows)] of an attention case, in row order."""
    rng = random.Random(case["lens_seed"])
    lo, hi = case["ctx_lo"], case["ctx_hi"]

    def ctx():
        if hi > 4 * lo and lo > 0:   # a wide range: spread over its logarithm
            return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        return rng.randint(lo, hi)

    out = []
    if case["op"] in ("decode", "step"):
        out += [(DECODE, max(0, ctx() - 1), 1) for _ in range(case["rows"])]
    if case["op"] in ("verify", "step"):
        out += [(VERIFY, ctx(), case["draft"]) for _ in range(case["blocks"])]
    if case["op"] in ("prefill", "step"):
        out += [(PREFILL, ctx(), case["chunk"]) for _ in range(case["requests"])]
    return out


def _append_spans(case):
    """[(first position, rows)] of an append case, one per sequence."""
    rng = random.Random(case["lens_seed"])
    return [(rng.randint(case["pos_lo"], case["pos_hi"]), case["count"]) for _ in range(case["seqs"])]


def _token_bytes(case):
    """K and V bytes of one token in the pool, scales included."""
    d, h = case["head_dim"], case["kv_heads"]
    per_head = {"bf16": 2 * d, "fp8": d + 4, "psq8": d + d // 16, "psq4": d // 2 + d // 16}[case["kv"]]
    return 2 * h * per_head


def work(case):
    """Each K/V token a sequence's rows see read once, each new row read and
    written once; a multiply-add is two operations."""
    tok, in_tok = _token_bytes(case), 4 * case["kv_heads"] * case["head_dim"]
    if case["op"] == "append":
        rows = case["seqs"] * case["count"]
        return {"bytes": rows * (in_tok + tok + 12), "flops": 0}
    qd = case["q_heads"] * case["head_dim"]
    nbytes = flops = 0
    for _, before, n in _requests(case):
        nbytes += (before + n) * tok + n * qd * (2 + (4 if case["out"] == "f32" else 2))
        flops += 4 * qd * (n * before + n * (n + 1) // 2)
        if case["op"] == "step":
            nbytes += n * (in_tok + tok)
    if case["op"] == "step":
        nbytes += 2 * case["copies"] * case["page"] * tok
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------------------ contents
E4M3_MAX = 448.0
PSQ4_EDGES = [0.5, 1.5, 2.5, 3.5, 5.0, 7.0, 9.0]
PSQ4_VALUES = [0.0, 1.0, 2.0, 3.0, 4.0, 6.0, 8.0, 10.0]


def _e4m3(x):
    return x.clamp(-E4M3_MAX, E4M3_MAX).to(torch.float8_e4m3fn).view(torch.uint8)


def _quantize(x, kv):
    """(codes, scales) of K or V rows x [n, head_dim] float32 as the pools hold them."""
    if kv == "bf16":
        return x.to(torch.bfloat16).view(torch.int16), None
    if kv == "fp8":
        amax = x.abs().amax(-1)
        scale = torch.where(amax == 0, torch.ones_like(amax), amax / torch.full_like(amax, E4M3_MAX))
        return _e4m3(x / scale[:, None]), scale
    b = x.view(-1, 32)
    top = b.abs().amax(-1)
    scale = (top * (np.float32(0.1).item() if kv == "psq4" else np.float32(1.0 / 448.0).item())).to(torch.bfloat16)
    inv = torch.where(scale > 0, 1.0 / scale.float(), torch.zeros_like(top))[:, None]
    if kv == "psq8":
        codes = _e4m3(b * inv)
    else:
        edges = torch.tensor(PSQ4_EDGES, device=x.device)
        c = torch.bucketize((b * inv).abs(), edges, out_int32=True).to(torch.uint8) + (b < 0).to(torch.uint8) * 8
        codes = c[:, :16] | (c[:, 16:] << 4)
    return codes.reshape(-1), scale.view(torch.int16)


def _dequantize(codes, scales, case):
    """float64 values [n, head_dim] of n (token, head) slices."""
    kv, d = case["kv"], case["head_dim"]
    if kv == "bf16":
        return codes.view(torch.bfloat16).view(-1, d).double()
    if kv == "fp8":
        return codes.view(torch.float8_e4m3fn).float().view(-1, d).double() * scales.double()[:, None]
    s = scales.view(torch.bfloat16).double()[:, None]
    if kv == "psq8":
        v = codes.view(torch.float8_e4m3fn).float().view(-1, 32).double()
    else:
        c = codes.view(-1, 16)
        c = torch.cat([c & 15, c >> 4], 1).long()
        v = torch.tensor(PSQ4_VALUES, dtype=torch.float64, device=codes.device)[c & 7] * (1.0 - 2.0 * (c >> 3).double())
    return (v * s).view(-1, d)


def _pool_sizes(case):
    """(code values, scale values) of one (token, head) slice."""
    d = case["head_dim"]
    return {"bf16": (d, 0), "fp8": (d, 1), "psq8": (d, d // 32), "psq4": (d // 2, d // 32)}[case["kv"]]


def _empty_pool(case, pages):
    codes, scales = _pool_sizes(case)
    n = pages * case["page"] * case["kv_heads"]
    dt = torch.int16 if case["kv"] == "bf16" else torch.uint8
    st = torch.float32 if case["kv"] == "fp8" else torch.int16
    pool = {"k": torch.zeros(n * codes, dtype=dt, device="cuda"), "v": torch.zeros(n * codes, dtype=dt, device="cuda")}
    if scales:
        pool["k_scale"] = torch.zeros(n * scales, dtype=st, device="cuda")
        pool["v_scale"] = torch.zeros(n * scales, dtype=st, device="cuda")
    return pool


def _filled_pool(case, pages, gen):
    """A pool whose every slot holds the codes of N(0, 1) values."""
    pool = _empty_pool(case, pages)
    codes, scales = _pool_sizes(case)
    n, step = pages * case["page"] * case["kv_heads"], (1 << 26) // case["head_dim"]
    for t in ("k", "v"):
        for at in range(0, n, step):
            m = min(step, n - at)
            c, s = _quantize(torch.randn((m, case["head_dim"]), generator=gen, device="cuda"), case["kv"])
            pool[t][at * codes:(at + m) * codes] = c.view(-1)
            if scales:
                pool[t + "_scale"][at * scales:(at + m) * scales] = s.view(-1)
    return pool


def _new_rows(case, rows, gen):
    """bf16 K or V rows: N(0, 1) with 1 % outliers x 20."""
    x = torch.randn((rows, case["kv_heads"] * case["head_dim"]), generator=gen, device="cuda")
    x = torch.where(torch.rand(x.shape, generator=gen, device="cuda") < 0.01, x * 20.0, x)
    return x.to(torch.bfloat16)


def _device_i32(values):
    return torch.from_numpy(np.ascontiguousarray(values, dtype=np.int32)).cuda()


def _attention_state(case, seed):
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    page, reqs = case["page"], _requests(case)
    need = [-(-(before + n) // page) for _, before, n in reqs]
    spare = case.get("copies", 0)
    pages = sum(need) + spare
    order = rng.permutation(pages).astype(np.int32)
    table = np.full((len(reqs), max(need)), -1, np.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = order[at:at + n]
        at += n
    rows = sum(n for _, _, n in reqs)
    s = {"case": case, "requests": reqs, "table": table, "block_tables": _device_i32(table)}
    s["geom"] = ops.PoolGeometry(1, pages, page, case["kv_heads"], case["head_dim"])
    s["pool"] = _filled_pool(case, pages, gen)
    q = torch.randn((rows, case["q_heads"] * case["head_dim"]), generator=gen, device="cuda") * 2.0
    s["q"] = q.to(torch.bfloat16).view(torch.int16)
    s["out"] = torch.zeros(q.shape, dtype=torch.float32 if case["out"] == "f32" else torch.bfloat16, device="cuda")
    s["slots"] = _device_i32(np.concatenate([np.full(n, i) for i, (_, _, n) in enumerate(reqs)]))
    s["positions"] = _device_i32(np.concatenate([np.arange(b, b + n) for _, b, n in reqs]))
    if case["op"] == "step":
        s["k_in"], s["v_in"] = _new_rows(case, rows, gen), _new_rows(case, rows, gen)
        s["cache"] = _filled_pool(case, 64, gen)
        src = rng.permutation(64)[:spare]
        s["pairs"] = _device_i32(np.stack([order[at:at + spare], src], 1))
    return s


def prepare(case, seed):
    if case["op"] == "append":
        return _append_state(case, seed)
    s = _attention_state(case, seed)
    row, reqs, descs = 0, [], []
    for i, (cls, before, n) in enumerate(s["requests"]):
        reqs.append((row, n, cls, before + n))
        descs.append(dict(slot=i, row_begin=row, row_count=n, prefix_length=before, sequence_length=before + n,
                          execution_class=cls))
        row += n
    s["plan_requests"] = reqs
    s["max_visible"] = max(r[3] for r in reqs)
    s["partials"] = torch.empty(WORKSPACE_BYTES // 4, dtype=torch.float32, device="cuda")
    if case["op"] == "step":
        s["descriptors"] = torch.from_numpy(np.frombuffer(ops.pack_requests(descs), np.uint8).copy()).cuda()
        s["num_descriptors"] = len(descs)
    return s


def _append_state(case, seed):
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    page, spans = case["page"], _append_spans(case)
    held = [(p // page, (p + n - 1) // page + 1) for p, n in spans]   # pages that take new rows
    pages = sum(b - a for a, b in held)
    order = rng.permutation(pages).astype(np.int32)
    table = np.full((len(spans), max(b for _, b in held)), -1, np.int32)
    at = 0
    for i, (a, b) in enumerate(held):
        table[i, a:b] = order[at:at + b - a]
        at += b - a
    rows = sum(n for _, n in spans)
    return {"case": case, "geom": ops.PoolGeometry(1, pages, page, case["kv_heads"], case["head_dim"]),
            "block_tables": _device_i32(table), "pool": _empty_pool(case, pages),
            "k_in": _new_rows(case, rows, gen), "v_in": _new_rows(case, rows, gen),
            "slots": _device_i32(np.concatenate([np.full(n, i) for i, (_, n) in enumerate(spans)])),
            "positions": _device_i32(np.concatenate([np.arange(p, p + n) for p, n in spans]))}


# ---------------------------------------------------------------------- run
def run(s):
    case, g, pool = s["case"], s["geom"], s["pool"]
    op, kv = case["op"], case["kv"]
    if op == "append":
        rows = (g, 0, s["k_in"], s["v_in"], s["slots"], s["positions"], s["block_tables"], pool["k"], pool["v"])
        if kv in ("psq4", "psq8"):
            ops.kv_append_psq(*rows, pool["k_scale"], pool["v_scale"], 4 if kv == "psq4" else 8, case["estimator"])
        else:
            ops.kv_append(*rows, pool.get("k_scale"), pool.get("v_scale"))
        return pool
    if op == "prefill" and case["api"] == "launcher":
        for begin, n, _, _ in s["plan_requests"]:
            rows = slice(begin, begin + n)
            a = (g, 0, s["q"][rows], s["out"][rows], s["slots"][rows], s["positions"][rows], s["block_tables"],
                 pool["k"], pool["v"])
            if kv in ("psq4", "psq8"):
                ops.paged_attention_psq(*a, pool["k_scale"], pool["v_scale"], case["q_heads"],
                                        4 if kv == "psq4" else 8, kind="prefill")
            else:
                ops.paged_attention(*a, case["q_heads"], pool.get("k_scale"), pool.get("v_scale"), kind="prefill")
        return s["out"]
    if op == "step":
        ops.kv_append_from_requests(g, 0, s["k_in"], s["v_in"], s["descriptors"], s["num_descriptors"], s["slots"],
                                    s["positions"], s["block_tables"], pool["k"], pool["v"], pool.get("k_scale"),
                                    pool.get("v_scale"))
    args = ops.attention_args(g, 0, s["q"], s["out"], s["slots"], s["positions"], s["block_tables"], case["q_heads"])
    state.plan_step(args, KV[kv], s["plan_requests"], s["max_visible"], WORKSPACE_BYTES, s["partials"], pool["k"],
                    pool["v"], pool.get("k_scale"), pool.get("v_scale"), launch=True)
    if op != "step":
        return s["out"]
    ops.copy_pages(g, pool, s["cache"], s["pairs"], src_num_pages=64)
    return {"out": s["out"], **pool}


# ------------------------------------------------------------ what is right
# About four times the largest distance from the 64-bit result seen over the
# listed cases and 80 drawn ones: BF16 KV and FP8 decode carry the weights P in
# 16 bits of mantissa (2.7e-6 / 4.2e-5), FP8 tiles P in f16 and Q in E4M3 parts
# (2.6e-4 / 8.0e-3), PSQ decode P x V scale in bf16 (8.0e-4 / 8.0e-3); a bf16
# output adds its own rounding (1.7e-3 / 3.9e-3). Appended bytes are exact.
def tolerance(case):
    if case["op"] == "append":
        return "exact"
    fine = case["kv"] == "bf16" or (case["kv"] == "fp8" and case["op"] == "decode")
    if case["out"] == "bf16":
        return {"rel": 7e-3, "max": 1.6e-2 if fine else 3.5e-2}
    if fine:
        return {"rel": 1.7e-5, "max": 1.7e-4}
    return {"rel": 1.1e-3 if case["kv"] == "fp8" else 3.2e-3, "max": 3.2e-2}


def exact(case, seed):
    if case["op"] == "append":
        return None   # whole codes, and scales that follow from them
    s = _attention_state(case, seed)
    pool, page, h, d = s["pool"], case["page"], case["kv_heads"], case["head_dim"]
    codes, scales = _pool_sizes(case)
    group = case["q_heads"] // h
    q = s["q"].view(torch.bfloat16).double().view(-1, h, group, d)
    out = torch.empty((q.shape[0], h, group, d), dtype=torch.float64, device="cuda")
    row = 0
    for i, (_, before, n) in enumerate(s["requests"]):
        total = before + n
        held = torch.from_numpy(s["table"][i, :-(-total // page)].astype(np.int64)).cuda()
        kv64 = {}
        for t in ("k", "v"):
            c = pool[t].view(-1, page * h * codes)[held].reshape(-1)
            sc = pool[t + "_scale"].view(-1, page * h * scales)[held].reshape(-1) if scales else None
            x = _dequantize(c, sc, case).view(-1, h, d)[:total]
            if case["op"] == "step":   # the rows appended in this step
                new, ns = _quantize(s[t + "_in"][row:row + n].float().view(-1, d), case["kv"])
                x = torch.cat([x[:before], _dequantize(new, ns, case).view(n, h, d)])
            kv64[t] = x
        hidden = torch.arange(total, device="cuda")[None, :] > torch.arange(before, total, device="cuda")[:, None]
        for j in range(h):
            scores = q[row:row + n, j].reshape(n * group, d) @ kv64["k"][:, j].contiguous().T / math.sqrt(d)
            scores = scores.view(n, group, total).masked_fill_(hidden[:, None, :], -math.inf)
            p = torch.softmax(scores, -1).view(n * group, total)
            out[row:row + n, j] = (p @ kv64["v"][:, j].contiguous()).view(n, group, d)
        row += n
    out = out.view(-1, case["q_heads"] * d)
    if case["op"] != "step":
        return out
    return {"out": out, **{k: None for k in pool}}
