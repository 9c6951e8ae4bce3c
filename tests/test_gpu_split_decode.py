"""GPU parity of the split decode kernel: batches of few, long and uneven
contexts whose items are computed in pieces that workgroups merge.  Contexts
around the tile and pass sizes, pieces longer than a pass, empty and over-long
contexts between live ones, 16- and 32-bit and FP8 caches, token rows of one and
of several tokens a block, explicit partition sizes, blocks outside the cache,
contexts short enough for whole items, a workspace without room for the pieces,
a repeated call on the same scratch (arrival counters return to zero), and the
same result from run to run.  Every case checks that the kernel ran."""

import numpy as np
import pytest
import torch

from oracle import pagedkv_oracle as orc
from pkv_cases import X_OF, decode_oracle, make_decode_case, normal, tolerance
from pkv_kernels import kernels_of
from pkv_torch import to_f64, to_index, to_torch
from sglang_mlx_amd import _ext, _lib, kernels
from sglang_mlx_amd.srt.mem_cache import build_cascade_plan

pytestmark = pytest.mark.gpu
FP8 = "fp8_e4m3"
KS, VS = 0.05, 0.02


def split_grid(call):
    """Workgroups of the split kernel that call() launches, and no other kernel."""
    (name, grid), = kernels_of(call)
    assert "split_kernel" in name, name
    return grid


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
    split_grid(lambda: kernels.paged_attention_v1(*args, alibi_slopes=alibi))
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


def pool_case(q, cache, Hq, Hkv, D, bs, ctx, max_seq_len, flash=False, seed=1, nb=96):
    """Contexts over a small pool whose blocks many tables share: (call arguments,
    reference).  flash: token rows [nb, bs, Hkv, D]."""
    rng = np.random.default_rng(seed)
    x = 16 if cache == FP8 else X_OF[cache]
    shapes = [(nb, bs, Hkv, D)] * 2 if flash else [(nb, Hkv, D // x, bs, x), (nb, Hkv, D, bs)]
    if cache == FP8:
        k, v = (orc.fp8_e4m3_encode(rng.standard_normal(s, dtype=np.float32) * 20) for s in shapes)
        scales = dict(k_scale=KS, v_scale=VS)
    else:
        k, v = (normal(rng, s, cache) for s in shapes)
        scales = {}
    ctx = np.asarray(ctx, dtype=np.int32)
    qs = normal(rng, (len(ctx), Hq, D), q)
    table = rng.integers(0, nb, size=(len(ctx), -(-max_seq_len // bs))).astype(np.int32)
    scale = D ** -0.5
    args = (to_torch(qs, q), to_torch(k, cache), to_torch(v, cache), to_index(table), to_index(ctx), Hkv, scale, bs,
            max_seq_len)
    if flash:  # the reference reads the paged layout
        k = k.reshape(nb, bs, Hkv, D // x, x).transpose(0, 2, 3, 1, 4)
        v = v.transpose(0, 2, 3, 1)
    ref = orc.paged_attention(qs, k, v, table, ctx, Hkv, scale, bs, max_seq_len, None, q, cache, **scales)
    return args, scales, ref


def check(q, cache, Hq, Hkv, D, bs, ctx, max_seq_len, partition=0, **kw):
    args, scales, ref = pool_case(q, cache, Hq, Hkv, D, bs, ctx, max_seq_len, **kw)

    def call():
        if partition:
            return kernels.paged_attention_v2(*args, partition_size=partition, **scales)
        return kernels.paged_attention_v1(*args, **scales)

    out = call()
    assert torch.equal(out, call())
    atol, rtol = tolerance(q, "float16" if cache == FP8 else cache)
    np.testing.assert_allclose(to_f64(out), ref, atol=atol, rtol=rtol)
    return split_grid(call)


@pytest.mark.parametrize("q", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("D,bs", [(128, 8), (128, 32), (256, 8), (256, 16), (192, 32)])
def test_fp8(q, D, bs):
    # Above head size 128 in the partition kernel's place; 128: in the persistent
    # kernel's (the line lies above what the partition kernel takes).
    if D > 128:
        check(q, FP8, 12, 6, D, bs, CONTEXTS, 16384)
    else:
        check(q, FP8, 16, 8, D, bs, [15000, 16, 1, 0, 9000, 4097, 16400] + [33] * 31, 16384)


@pytest.mark.parametrize("q,cache,D", [("float16", "float16", 192), ("float32", "float32", 256),
                                       ("bfloat16", FP8, 256)])
@pytest.mark.parametrize("bs", [8, 16])
def test_partition_sizes(q, cache, D, bs):
    for partition in (512, 4096):
        check(q, cache, 12, 6, D, bs, CONTEXTS, 16384, partition=partition)


@pytest.mark.parametrize("bs", [8, 16, 32])
def test_rows_of_blocks(bs):
    check("float16", "float16", 12, 6, 128, bs, CONTEXTS, 16384, flash=True)


@pytest.mark.parametrize("flash", [False, True])
def test_pieces_of_several_passes(flash):
    # A workgroup holds the block ids of 4096 tokens (row ids of 2048) at a
    # time; here its mean load alone is more.
    ctx = [12288 - 7 * i for i in range(16)] if flash else [16384 - 50 * i for i in range(38)]
    grid = check("bfloat16", "bfloat16", 8, 8, 128, 16, ctx, ctx[0], flash=flash)
    assert sum(-(-n // 16) for n in ctx) * 8 > (2048 if flash else 4096) // 16 * grid


def abi_call(args, out, ws):
    """pkv_paged_attention of a pool_case's float16 arguments in a given workspace."""
    q, k, v, table, ctx, Hkv, scale, bs, max_seq = args
    B, Hq, D = q.shape
    _lib.check(_lib.lib().pkv_paged_attention(
        out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), table.data_ptr(), ctx.data_ptr(), None, B, Hq, Hkv, D,
        bs, table.shape[1], max_seq, k.shape[0], scale, q.stride(0), k.stride(0), k.stride(1), v.stride(0), v.stride(1),
        _lib.PKV_LAYOUT_PAGED5D, 0, ws.data_ptr(), ws.numel(), _lib.PKV_F16, _lib.PKV_F16, 1.0, 1.0,
        torch.cuda.current_stream().cuda_stream))


def test_workspace_without_room_for_pieces():
    args, _, ref = pool_case("float16", "float16", 12, 6, 128, 16, CONTEXTS, 16384)
    sizes = (len(CONTEXTS), 12, 6, 128, 16384, 0)
    least = _lib.lib().pkv_paged_attention_workspace_size(*sizes)
    full = _lib.lib().pkv_paged_attention_full_workspace_size(*sizes)
    assert full > least
    for nbytes, split in ((least, False), (full - 1, False), (full, True)):
        ws = torch.zeros(nbytes, dtype=torch.uint8, device="cuda")
        out = torch.empty_like(args[0])
        abi_call(args, out, ws)
        assert any("split_kernel" in name for name, _ in kernels_of(lambda: abi_call(args, out, ws))) == split
        atol, rtol = tolerance("float16", "float16")
        np.testing.assert_allclose(to_f64(out), ref, atol=atol, rtol=rtol)
        assert not ws[:_lib.PKV_COUNTER_BYTES].any()


@pytest.mark.parametrize("q,cache", [("float16", "float16"), ("float32", "float32"), ("float32", FP8)])
@pytest.mark.parametrize("D", [32, 80, 128, 192, 256])
def test_room_is_asked_for_wherever_the_kernel_runs(q, cache, D):
    # The size's rule covers the launch's: sizes on either side of each line.
    if cache == FP8 and D == 80:
        D = 96
    ran = 0
    for B, Hkv, max_seq, flash in ((1, 8, 4096, False), (8, 1, 16384, True), (9, 8, 2730, True), (16, 6, 16384, False),
                                   (12, 6, 5000, False), (33, 8, 16384, False), (63, 8, 4096, False),
                                   (64, 8, 16384, False), (31, 1, 25000, False), (8, 8, 3072, True), (8, 8, 3056, True)):
        if flash and cache != "float16":
            continue
        (qs, k, v, table, ctx, *_), _, _ = pool_case(q, cache, 2 * Hkv, Hkv, D, 16, [1] * B, max_seq, flash=flash, nb=4)
        i = -2 if flash else 1
        least = _lib.lib().pkv_paged_attention_workspace_size(B, 2 * Hkv, Hkv, D, max_seq, 0)
        full = _lib.lib().pkv_paged_attention_full_workspace_size(B, 2 * Hkv, Hkv, D, max_seq, 0)
        ws = torch.zeros(max(full, 64 << 20), dtype=torch.uint8, device="cuda")
        code = {"float16": _lib.PKV_F16, "float32": _lib.PKV_F32, FP8: _lib.PKV_FP8_E4M3}
        out = torch.empty_like(qs)
        names = kernels_of(lambda: _lib.check(_lib.lib().pkv_paged_attention(
            out.data_ptr(), qs.data_ptr(), k.data_ptr(), v.data_ptr(), table.data_ptr(), ctx.data_ptr(), None, B,
            2 * Hkv, Hkv, D, 16, table.shape[1], max_seq, 4, 0.1, qs.stride(0), k.stride(0), k.stride(i), v.stride(0),
            v.stride(i), _lib.PKV_LAYOUT_TOKEN_MAJOR if flash else _lib.PKV_LAYOUT_PAGED5D, 0, ws.data_ptr(),
            ws.numel(), code[q], code[cache], 1.0, 1.0, torch.cuda.current_stream().cuda_stream)))
        split = any("split_kernel" in n for n, _ in names)
        ran += split
        assert full > least or not split, (B, Hkv, max_seq, flash)
    assert ran or cache == FP8 and D < 128


@pytest.mark.parametrize("longest", [0, 31 * 16 + 1, 32 * 16, 32 * 16 + 1])
def test_short_contexts_in_the_partition_kernel_s_place(longest):
    # Whole items up to 32 tiles, pieces above.
    ctx = [longest, 1, 0, 17, 500, 16385] + [min(longest, 100 * i) for i in range(1, 11)]
    check("float16", "float16", 12, 6, 128, 16, ctx, 16384)
    check("float16", "float16", 12, 6, 128, 16, ctx, 16384, flash=True)


@pytest.mark.parametrize("longest", [64 * 16, 64 * 16 + 1])
def test_short_contexts_in_the_persistent_kernel_s_place(longest):
    # The same up to 64 tiles; 304 items.
    ctx = [longest, 1, 0, 17, 500, 16385] + [5 * i for i in range(32)]
    check("bfloat16", "bfloat16", 32, 8, 128, 16, ctx, 16384)


@pytest.mark.parametrize("longest,whole", [(32 * 16, True), (32 * 16 + 1, False)])
def test_whole_items_leave_no_pieces(longest, whole):
    args, _, ref = pool_case("float16", "float16", 12, 6, 128, 16, [longest] * 16, 16384)
    ws = torch.full((_lib.lib().pkv_paged_attention_full_workspace_size(16, 12, 6, 128, 16384, 0),), 77,
                    dtype=torch.uint8, device="cuda")
    ws[:_lib.PKV_COUNTER_BYTES].zero_()
    out = torch.empty_like(args[0])
    abi_call(args, out, ws)
    atol, rtol = tolerance("float16", "float16")
    np.testing.assert_allclose(to_f64(out), ref, atol=atol, rtol=rtol)
    assert bool((ws[_lib.PKV_COUNTER_BYTES:] == 77).all()) == whole


def test_cascade_in_one_pass_does_not_depend_on_the_scratch():
    # Head size 96 has no cascade kernel: the same bytes whatever scratch
    # earlier calls of the stream left.
    args, _, ref = pool_case("float16", "float16", 12, 6, 96, 16, [2000 - 90 * i for i in range(16)], 16384)
    plan = build_cascade_plan(args[3].cpu().numpy(), args[4].cpu().numpy(), 16, 12, 6, device="cuda")
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        first = kernels.paged_attention_cascade(*args, plan)
        assert _ext._ws_cache[(0, stream.cuda_stream)].numel() < 1 << 20
        _ext._decode_scratch(args[0].device, stream.cuda_stream, 64 << 20)
        again = kernels.paged_attention_cascade(*args, plan)
    stream.synchronize()
    atol, rtol = tolerance("float16", "float16")
    np.testing.assert_allclose(to_f64(first), ref, atol=atol, rtol=rtol)
    assert torch.equal(first, again)
