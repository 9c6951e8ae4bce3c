"""Performance cases of the paged-KV path.

Each case is one call (or one layer's append and decode) as a serving program
makes it on tensors it already holds: KV caches filled by earlier steps, block
or slot tables, context lengths, queries.  Kinds:

  decode   block-table decode attention, paged 5-D caches (paged_attention_v1,
           or paged_attention_v2 when the case names a partition size)
  rows     decode straight from token-major pool rows (block size 1)
  cascade  decode of a batch with radix-shared prefixes and its plan
  append   slot-mapped KV append, paged 5-D or token-major
  step     one layer's decode step: append of one token per sequence, then
           decode over the updated cache

Contexts (and prompt lengths) of a batch are spread evenly over [lo, hi] and
dealt in an order that the seed draws, so every seed has the same work.
"""

import math
import os
import sys

import numpy as np
import torch

# The package sits one level below the repository's root.
sys.path.insert(0, os.path.abspath("sglang-mlx_amd"))

from sglang_mlx_amd import kernels  # noqa: E402
from sglang_mlx_amd.srt.mem_cache import build_cascade_plan  # noqa: E402

DEV = "cuda:0"
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "fp8": torch.uint8}
BYTES = {"f32": 4, "f16": 2, "bf16": 2, "fp8": 1}
# Scales of FP8 caches: codes hold K / k_scale and V / v_scale.
K_SCALE, V_SCALE = 0.05, 0.02
# Queries are this much wider than unit normal, so that a softmax row has the
# peaks that attention over a real context has.
Q_GAIN = 2.0

# Bytes that a drawn decode case may read (the largest listed one reads 605 MB),
# and tokens that a drawn append may write: prompts of a chunked prefill, or
# single tokens at scattered slots.
DRAW_BYTES = 5.0e8
DRAW_TOKENS = {"prompts": 16384, "scatter": 4096}


def listed():
    return [
        # One user, a short context: the reference's own decode benchmark
        # (batch 1, fp16); launch and latency bound.
        dict(name="decode_b1_1k", kind="decode", q="f16", cache="f16", batch=1, heads=32, kv_heads=8, head_size=128,
             block_size=16, lo=1024, hi=1024, partition=0, alibi=False),
        # A lightly loaded server's layer: 16 sequences append their new token
        # and decode.
        dict(name="step_b16", kind="step", q="bf16", cache="bf16", batch=16, heads=32, kv_heads=8, head_size=128,
             block_size=16, lo=256, hi=4096, partition=0, alibi=False),
        # A loaded server's layer (the repository's headline workload).
        dict(name="decode_b64", kind="decode", q="bf16", cache="bf16", batch=64, heads=32, kv_heads=8, head_size=128,
             block_size=16, lo=512, hi=4096, partition=0, alibi=False),
        # The same layer over FP8 caches.
        dict(name="decode_fp8_b64", kind="decode", q="bf16", cache="fp8", batch=64, heads=32, kv_heads=8,
             head_size=128, block_size=16, lo=512, hi=4096, partition=0, alibi=False),
        # A small model (head size 64) serving many short ragged chats.
        dict(name="decode_d64_b96", kind="decode", q="f16", cache="f16", batch=96, heads=32, kv_heads=8, head_size=64,
             block_size=32, lo=33, hi=2011, partition=0, alibi=False),
        # Multi-head attention with ALiBi, 8-token blocks, float32 activations
        # over a half-precision cache.
        dict(name="decode_mha_alibi", kind="decode", q="f32", cache="f16", batch=13, heads=32, kv_heads=32,
             head_size=96, block_size=8, lo=90, hi=3000, partition=0, alibi=True),
        # One long context, split-K (28 query heads over 4 KV heads).
        dict(name="split_b1_32k", kind="decode", q="bf16", cache="bf16", batch=1, heads=28, kv_heads=4, head_size=128,
             block_size=16, lo=32768, hi=32768, partition=512, alibi=False),
        # Decode from the token pool's rows, contexts up to 8K tokens.
        dict(name="rows_b24_8k", kind="rows", q="f16", cache="f16", batch=24, heads=32, kv_heads=8, head_size=128,
             lo=500, hi=8000, alibi=False),
        # 256 requests on one 2048-token system prompt, private tails.
        dict(name="cascade_b256", kind="cascade", q="bf16", cache="bf16", batch=256, heads=32, kv_heads=8,
             head_size=128, block_size=16, prefix=2048, groups=1, lo=64, hi=512),
        # Prefill of a batch of ragged prompts, 16K tokens in all.
        dict(name="append_prefill", kind="append", layout="paged", kv="bf16", cache="bf16", tokens=16384, kv_heads=8,
             head_size=128, block_size=16, lo=97, hi=927, pattern="prompts"),
        # The token pool's append: rows at slots that the free list hands out.
        dict(name="append_pool", kind="append", layout="token", kv="bf16", cache="bf16", tokens=4096, kv_heads=8,
             head_size=128, block_size=1, lo=1, hi=1, pattern="scatter"),
        # Prefill into FP8 caches, 8K tokens.
        dict(name="append_fp8_prefill", kind="append", layout="paged", kv="bf16", cache="fp8", tokens=8192,
             kv_heads=8, head_size=128, block_size=16, lo=97, hi=927, pattern="prompts"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _spread(rng, mean):
    """Shortest and longest context of a batch whose mean is `mean`."""
    lo = max(1, int(mean * rng.uniform(0.05, 1.0)))
    return lo, max(lo, 2 * mean - lo)


def draw(rng):
    kind = rng.choice(["decode"] * 6 + ["rows"] * 2 + ["cascade"] * 2 + ["append"] * 4 + ["step"] * 2)
    if kind == "append":
        layout = rng.choice(["paged", "paged", "token"])
        kv, cache = rng.choice([("bf16", "bf16"), ("f16", "f16"), ("f32", "f16"), ("f32", "bf16"), ("bf16", "fp8"),
                                ("f16", "fp8")])
        kv_heads, head_size = rng.choice([(8, 128), (8, 64), (4, 128), (2, 64), (32, 96), (16, 80), (8, 256)])
        pattern = rng.choice(["prompts", "scatter"]) if layout == "paged" else "scatter"
        # Rows of the listed appends are 1024 elements: no drawn case moves more.
        most = DRAW_TOKENS[pattern]
        tokens = min(_log_int(rng, 1, most), most * 1024 // (kv_heads * head_size))
        lo = _log_int(rng, 1, min(tokens, 2048))
        return dict(kind=kind, layout=layout, kv=kv, cache=cache, tokens=tokens, kv_heads=kv_heads,
                    head_size=head_size, block_size=rng.choice([8, 16, 16, 32]) if layout == "paged" else 1,
                    lo=lo, hi=min(4 * lo, 8192), pattern=pattern)
    if kind == "cascade":
        q, cache = rng.choice([("bf16", "bf16"), ("f16", "f16"), ("bf16", "fp8")])
        groups = rng.choice([1, 1, 2, 5])
        lo = _log_int(rng, 20, 400)
        return dict(kind=kind, q=q, cache=cache, batch=max(2 * groups, _log_int(rng, 16, 256)), heads=32,
                    kv_heads=rng.choice([8, 8, 4]), head_size=rng.choice([128, 128, 64]),
                    block_size=rng.choice([16, 16, 32]), prefix=32 * _log_int(rng, 8, 128), groups=groups, lo=lo,
                    hi=lo + _log_int(rng, 1, 600))
    pairs = [("bf16", "bf16"), ("bf16", "bf16"), ("f16", "f16"), ("f32", "f16"), ("f32", "bf16")]
    if kind == "decode":
        pairs += [("bf16", "fp8"), ("f16", "fp8"), ("f32", "f32")]
    q, cache = rng.choice(pairs)
    kv_heads, group = rng.choice([(8, 4), (8, 4), (8, 8), (4, 7), (2, 7), (1, 8), (32, 1), (16, 2)])
    head_size = rng.choice([64, 80, 96, 128, 128, 128, 256])
    mean = _log_int(rng, 48, 32768 if kind == "decode" else 8192)
    per_token = 2 * kv_heads * head_size * BYTES[cache]
    mean = min(mean, int(DRAW_BYTES / per_token))
    batch = min(_log_int(rng, 1, 256), max(1, int(DRAW_BYTES / (per_token * mean))))
    lo, hi = _spread(rng, mean)
    case = dict(kind=kind, q=q, cache=cache, batch=batch, heads=kv_heads * group, kv_heads=kv_heads,
                head_size=head_size, lo=lo, hi=hi, alibi=rng.random() < 0.15)
    if kind != "rows":
        case["block_size"] = rng.choice([8, 16, 16, 32])
        case["partition"] = 0 if kind == "step" else rng.choice([0, 0, 512, 1024])
    return case


# ---- inputs ---------------------------------------------------------------------


def _lengths(lo, hi, n):
    """n lengths spread evenly over [lo, hi] (the mean (lo + hi) / 2)."""
    return np.array([lo + int((hi - lo) * (i + 0.5) / n + 0.5) for i in range(n)], dtype=np.int64)


def _prompts(case):
    """Lengths of the prompts that a prefill of case["tokens"] tokens packs."""
    out, left, i = [], case["tokens"], 0
    while left > 0:
        n = min(left, case["lo"] + (case["hi"] - case["lo"]) * (i % 5) // 4)
        out.append(n)
        left -= n
        i += 1
    return out


def _values(shape, dtype, gen):
    """Cache contents: unit normal, as codes of x / scale for FP8 (below
    exponent 15, where the format's finite values end)."""
    if dtype == "fp8":
        x = torch.empty(shape, dtype=torch.float16, device=DEV).normal_(generator=gen)
        return x.mul_(20.0).clamp_(-240.0, 240.0).to(torch.float8_e4m3fn).view(torch.uint8)
    return torch.empty(shape, dtype=TORCH[dtype], device=DEV).normal_(generator=gen)


def _paged_caches(nb, case, gen):
    H, D, bs = case["kv_heads"], case["head_size"], case["block_size"]
    x = 16 // BYTES[case["cache"]]
    return _values((nb, H, D // x, bs, x), case["cache"], gen), _values((nb, H, D, bs), case["cache"], gen)


def _device_ints(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).to(DEV)


def _tables(ctx, bs, rng, shared=None):
    """int32 block table and the pool's block count: blocks in random order
    over a pool a tenth larger (block 0 is never handed out).  shared: leading
    blocks that a sequence's group has in common, (group of each, count)."""
    need = -(-ctx // bs)
    group, lead = shared if shared else (None, 0)
    ngroups = 0 if group is None else int(group.max()) + 1
    used = int(need.sum()) - (len(ctx) - ngroups) * lead
    nb = used + used // 10 + 2
    ids = rng.permutation(nb - 1)[:used] + 1
    heads = ids[:ngroups * lead].reshape(ngroups, lead)
    table = np.full((len(ctx), int(need.max())), -1, dtype=np.int32)
    at = ngroups * lead
    for i, n in enumerate(need):
        own = int(n) - lead
        if lead:
            table[i, :lead] = heads[group[i]]
        table[i, lead:lead + own] = ids[at:at + own]
        at += own
    return table, nb


def _query(case, gen):
    shape = (case["batch"], case["heads"], case["head_size"])
    return (torch.empty(shape, dtype=torch.float32, device=DEV).normal_(generator=gen) * Q_GAIN).to(TORCH[case["q"]])


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    s = {"case": case}
    if case["kind"] == "append":
        return _prepare_append(case, s, rng, gen)
    B, D, kind = case["batch"], case["head_size"], case["kind"]
    ctx = rng.permutation(_lengths(case["lo"], case["hi"], B))
    if kind == "cascade":
        ctx = ctx + case["prefix"]
    s["scale"] = 1.0 / math.sqrt(D)
    s["scales"] = {"k_scale": K_SCALE, "v_scale": V_SCALE} if case["cache"] == "fp8" else {}
    s["query"] = _query(case, gen)
    s["max_seq_len"] = int(ctx.max())
    s["alibi"] = None
    if case.get("alibi"):
        slopes = [2.0 ** (-8.0 * (h + 1) / case["heads"]) for h in range(case["heads"])]
        s["alibi"] = torch.tensor(slopes, dtype=torch.float32, device=DEV)
    s["ctx"] = _device_ints(ctx)
    if kind == "rows":
        used = int(ctx.sum())
        slots = used + used // 10 + 2
        ids = rng.permutation(slots - 1)[:used] + 1
        table = np.full((B, int(ctx.max())), -1, dtype=np.int32)
        at = 0
        for i, n in enumerate(ctx):
            table[i, :n] = ids[at:at + n]
            at += n
        s["table"] = _device_ints(table)
        shape = (slots, case["kv_heads"], D)
        s["k"], s["v"] = _values(shape, case["cache"], gen), _values(shape, case["cache"], gen)
        return s
    bs = case["block_size"]
    shared = None
    if kind == "cascade":
        shared = (np.arange(B) * case["groups"] // B, case["prefix"] // bs)
    table, nb = _tables(ctx, bs, rng, shared)
    s["table"] = _device_ints(table)
    s["k"], s["v"] = _paged_caches(nb, case, gen)
    if kind == "cascade":
        s["plan"] = build_cascade_plan(table, ctx, bs, case["heads"], case["kv_heads"], device=DEV)
    if kind == "step":
        # The step's new token is each sequence's last.
        last = ctx - 1
        s["slots"] = _device_ints(table[np.arange(B), last // bs].astype(np.int64) * bs + last % bs)
        shape = (B, case["kv_heads"], D)
        new = TORCH[case["q"]]
        s["key"] = torch.empty(shape, dtype=new, device=DEV).normal_(generator=gen)
        s["value"] = torch.empty(shape, dtype=new, device=DEV).normal_(generator=gen)
    return s


def _prepare_append(case, s, rng, gen):
    N, H, D, bs = case["tokens"], case["kv_heads"], case["head_size"], case["block_size"]
    shape = (N, H, D)
    s["key"] = torch.empty(shape, dtype=TORCH[case["kv"]], device=DEV).normal_(generator=gen)
    s["value"] = torch.empty(shape, dtype=TORCH[case["kv"]], device=DEV).normal_(generator=gen)
    s["scales"] = {"k_scale": K_SCALE, "v_scale": V_SCALE} if case["cache"] == "fp8" else {}
    if case["pattern"] == "prompts":
        # Each prompt fills fresh blocks from offset 0.
        lens = _prompts(case)
        need = [-(-n // bs) for n in lens]
        nb = 2 * sum(need) + 2
        ids = rng.permutation(nb - 1)[:sum(need)].astype(np.int64) + 1
        slots, at = [], 0
        for n, b in zip(lens, need):
            t = np.arange(n)
            slots.append(ids[at + t // bs] * bs + t % bs)
            at += b
        slots = np.concatenate(slots)
        num_slots = nb * bs
    else:
        # Single tokens anywhere in a pool eight times as large.
        nb = 8 * N // bs + 2
        num_slots = nb * bs
        slots = rng.permutation(num_slots - bs)[:N] + bs
    s["slots"] = _device_ints(slots)
    if case["layout"] == "paged":
        s["k"], s["v"] = _paged_caches(nb, case, gen)
    else:
        shape = (num_slots, H, D)
        s["k"], s["v"] = _values(shape, case["cache"], gen), _values(shape, case["cache"], gen)
    return s


# ---- one pass -------------------------------------------------------------------


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "append":
        return kernels.reshape_and_cache(s["key"], s["value"], s["k"], s["v"], s["slots"], **s["scales"])
    if kind == "cascade":
        return kernels.paged_attention_cascade(s["query"], s["k"], s["v"], s["table"], s["ctx"], case["kv_heads"],
                                               s["scale"], case["block_size"], s["max_seq_len"], s["plan"],
                                               **s["scales"])
    bs = 1 if kind == "rows" else case["block_size"]
    if kind == "step":
        kernels.reshape_and_cache(s["key"], s["value"], s["k"], s["v"], s["slots"])
    more = dict(s["scales"])
    if s["alibi"] is not None:
        more["alibi_slopes"] = s["alibi"]
    if case.get("partition"):
        out = kernels.paged_attention_v2(s["query"], s["k"], s["v"], s["table"], s["ctx"], case["kv_heads"],
                                         s["scale"], bs, s["max_seq_len"], partition_size=case["partition"], **more)
    else:
        out = kernels.paged_attention_v1(s["query"], s["k"], s["v"], s["table"], s["ctx"], case["kv_heads"],
                                         s["scale"], bs, s["max_seq_len"], **more)
    return (out, s["k"], s["v"]) if kind == "step" else out


# ---- what a pass cannot do without ------------------------------------------------


def work(case):
    H, D = case["kv_heads"], case["head_size"]
    if case["kind"] == "append":
        row = case["tokens"] * H * D
        return {"bytes": 2 * row * (BYTES[case["kv"]] + BYTES[case["cache"]]) + 4 * case["tokens"], "flops": 0}
    B = case["batch"]
    own = int(_lengths(case["lo"], case["hi"], B).sum())
    prefix = case.get("prefix", 0)
    tokens = own + case.get("groups", 0) * prefix  # tokens whose K and V are read once
    bs = case.get("block_size", 1)
    nbytes = tokens * H * D * 2 * BYTES[case["cache"]]
    nbytes += 2 * B * case["heads"] * D * BYTES[case["q"]] + 4 * (own + B * prefix) // bs + 4 * B
    if case["kind"] == "step":
        nbytes += 2 * B * H * D * (BYTES[case["q"]] + BYTES[case["cache"]]) + 4 * B
    return {"bytes": nbytes, "flops": 4 * (own + B * prefix) * case["heads"] * D}


def tolerance(case):
    if case["kind"] == "append":
        return "exact"  # copies, conversions by a fixed rule, codes of a fixed encoder
    # The output's rounding and that of the softmax weights, which take the
    # cache's 16-bit type (over FP8 caches the query's, or float16 for a
    # float32 query) and stay float32 over float32 caches.  Measured against
    # 64 bits: bf16 2.2e-3, f16 2.6e-4, float32 out 1.8e-4 with f16 weights
    # and 1.5e-3 with bf16 ones; about four times that is allowed.
    if case["cache"] == "f32":
        return {"rel": 1e-5}
    weights = case["cache"] if case["cache"] != "fp8" else ("bf16" if case["q"] == "bf16" else "f16")
    if case["q"] == "f32":
        return {"rel": 6e-3 if weights == "bf16" else 7e-4}
    return {"rel": 1e-2 if weights == "bf16" else 1.1e-3}


# ---- the same in 64 bits ----------------------------------------------------------


def _decode_codes(codes):
    """E4M3 codes (bias 7) below exponent 15 as float64."""
    c = torch.arange(256, dtype=torch.int64)
    e, m = (c >> 3) & 15, (c & 7).double()
    mag = torch.where(e == 0, m / 8 * 2.0 ** -6, (1 + m / 8) * 2.0 ** (e.double() - 7))
    table = torch.where(c >= 128, -mag, mag).to(codes.device)
    return table[codes.long()]


def exact(case, seed):
    if case["kind"] == "append":
        return None  # bytes, compared whole
    s = prepare(case, seed)
    fp8 = case["cache"] == "fp8"
    B, H, D = case["batch"], case["kv_heads"], case["head_size"]
    group = case["heads"] // H
    bs = case.get("block_size", 1)
    if case["kind"] == "step":
        blk, off = s["slots"].long() // bs, s["slots"].long() % bs
        x = s["k"].shape[4]
        s["k"][blk, :, :, off, :] = s["key"].to(s["k"].dtype).view(B, H, D // x, x)
        s["v"][blk, :, :, off] = s["value"].to(s["v"].dtype)
    out = torch.empty((B, case["heads"], D), dtype=torch.float64, device=DEV)
    for i, n in enumerate(s["ctx"].tolist()):
        ids = s["table"][i, :-(-n // bs)].long()
        k, v = s["k"][ids], s["v"][ids]
        k, v = (_decode_codes(k) * K_SCALE, _decode_codes(v) * V_SCALE) if fp8 else (k.double(), v.double())
        if case["kind"] == "rows":
            k, v = k.permute(1, 2, 0), v.permute(1, 0, 2)  # [H, D, T], [H, T, D]
        else:
            k = k.permute(1, 2, 4, 0, 3).reshape(H, D, -1)[..., :n]
            v = v.permute(1, 0, 3, 2).reshape(H, -1, D)[:, :n]
        qi = s["query"][i].double().view(H, group, D)
        sc = torch.bmm(qi, k.contiguous()) * s["scale"]
        if s["alibi"] is not None:
            pos = torch.arange(n, dtype=torch.float64, device=DEV) - (n - 1)
            sc = sc + s["alibi"].double().view(H, group, 1) * pos
        p = torch.softmax(sc, dim=-1)
        out[i] = torch.bmm(p, v.contiguous()).view(case["heads"], D)
    return (out, None, None) if case["kind"] == "step" else out
