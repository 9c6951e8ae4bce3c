"""GPU parity of the split decode kernel: batches of few, long and uneven
contexts whose items are computed in pieces that workgroups merge.  Contexts
around the tile and pass sizes, empty and over-long contexts between live ones,
16- and 32-bit caches and token rows, blocks outside the cache, a repeated call on the same scratch (arrival counters return to zero),
and the same result from run to run."""

import numpy as np
import pytest
import torch

from oracle import pagedkv_oracle as orc
from pkv_cases import decode_oracle, make_decode_case, tolerance
from pkv_torch import to_f64, to_index, to_torch
from sglang_mlx_amd import kernels

pytestmark = pytest.mark.gpu


def rows_of(case):
    """The case's paged caches as token rows [slots, Hkv, D], slot tables."""
    nb, H, dx, bs, x = case.k_cache.shape
    k = case.k_cache.transpose(0, 3, 1, 2, 4).reshape(nb * bs, H, dx * x)
    v = case.v_cache.transpose(0, 3, 1, 2).reshape(nb * bs, H, dx * x)
    t = np.arange(case.block_tables.shape[1] * bs)
    table = np.where(case.block_tables[:, t // bs] < 0, -1, case.block_tables[:, t // bs] * bs + t % bs)
    return np.ascontiguousarray(k), np.ascontiguousarray(v), table.astype(np.int32)


def run(c, rows):
    if rows:
        k, v, table = rows_of(c)
        bs = 1
    else:
        k, v, table, bs = c.k_cache, c.v_cache, c.block_tables, c.block_size
    args = (to_torch(c.q, c.q_dtype), to_torch(k, c.cache_dtype), to_torch(v, c.cache_dtype), to_index(table),
            to_index(c.context_lens), c.num_kv_heads, c.scale, bs, c.max_seq_len)
    alibi = None if c.alibi is None else torch.from_numpy(c.alibi).cuda()
    outs = [kernels.paged_attention_v1(*args, alibi_slopes=alibi) for _ in range(3)]
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    return to_f64(outs[0])


CONTEXTS = [1, 0, 15, 16, 17, 127, 128, 129, 2047, 2048, 2049, 4095, 4096, 4111, 9000, 16400]


@pytest.mark.parametrize("rows", [False, True])
@pytest.mark.parametrize("q,cache,Hq,Hkv,D,bs", [("bfloat16", "bfloat16", 24, 6, 128, 16),
                                                 ("float16", "float16", 42, 6, 80, 32),
                                                 ("float32", "float16", 6, 6, 96, 8),
                                                 ("bfloat16", "bfloat16", 60, 3, 120, 16),  # group of 20
                                                 ("float32", "float32", 12, 6, 64, 16),
                                                 ("float32", "bfloat16", 6, 6, 256, 32)])
def test_uneven_contexts(rows, q, cache, Hq, Hkv, D, bs):
    # 96 (sequence, unit) items, 384 partition workgroups.
    if rows and cache == "float32":
        pytest.skip("float32 caches are read in the paged layout")
    ctx = CONTEXTS
    # The last context of the list is longer than max_seq_len: a zero row.
    c = make_decode_case(7, B=len(ctx), Hq=Hq, Hkv=Hkv, D=D, block_size=bs, ctx_lo=1, ctx_hi=1, q_dtype=q,
                         cache_dtype=cache, alibi=D == 96, context_lens=ctx)
    c.max_seq_len = 16384
    atol, rtol = tolerance(q, cache)
    got, ref = run(c, rows), decode_oracle(c)
    assert not ref[-1].any() and not ref[1].any()
    np.testing.assert_allclose(got, ref, atol=atol, rtol=rtol)


def test_blocks_outside_the_cache_are_masked():
    c = make_decode_case(3, B=12, Hq=32, Hkv=8, D=128, block_size=16, ctx_lo=1, ctx_hi=1,
                         context_lens=[12000, 1500, 700, 9000, 40, 8000, 12000, 300, 11000, 5000, 12000, 2000])
    atol, rtol = tolerance("bfloat16", "bfloat16")
    rng, nb = np.random.default_rng(5), c.k_cache.shape[0]
    for i, n in enumerate(c.context_lens):
        last = -(-int(n) // 16)
        at = rng.integers(1, last, size=last // 10)
        c.block_tables[i, at] = rng.choice([-1, nb, 1 << 30], size=len(at))
    got = run(c, False)
    # The same attention over the tokens of the blocks inside the cache.
    q = orc.decode(c.q, "bfloat16").astype(np.float64)
    k, v, table = rows_of(c)
    for i, n in enumerate(c.context_lens):
        blk = c.block_tables[i, np.arange(n) // 16].astype(np.int64)
        keep = (blk >= 0) & (blk < nb)
        slots = (blk * 16 + np.arange(n) % 16)[keep]
        kk, vv = (orc.decode(x[slots], "bfloat16").astype(np.float64) for x in (k, v))
        for h in range(8):
            s = q[i, 4 * h:4 * h + 4] @ kk[:, h].T * c.scale
            p = np.exp(s - s.max(axis=1, keepdims=True))
            ref = p @ vv[:, h] / (p.sum(axis=1, keepdims=True) + 1e-6)
            np.testing.assert_allclose(got[i, 4 * h:4 * h + 4], ref, atol=atol, rtol=rtol)


def test_more_items_than_workgroups():
    # 304 items, which the persistent kernel would take whole, a few of them
    # long enough to be split.
    ctx = [10000, 300, 0, 5000] + list(range(1, 290, 8))[:34]
    c = make_decode_case(11, B=38, Hq=32, Hkv=8, D=128, block_size=16, ctx_lo=1, ctx_hi=1, context_lens=ctx)
    atol, rtol = tolerance("bfloat16", "bfloat16")
    np.testing.assert_allclose(run(c, False), decode_oracle(c), atol=atol, rtol=rtol)
