"""GPU parity of the paged append's window kernel, bit-exact over whole caches:
whole-block runs at every offset of a window, runs broken at their first, a
middle and their last token, the cache's last block, padding and slots past the
cache, head sizes whose run tasks do not fill a workgroup, large calls whose
workgroups take several heads, small ones on either side of the search for runs,
and FP8 codes whose quotients are ties, subnormals, overflows and zeros, or come
from every 16-bit pattern, at scales with and without an exact reciprocal and
beyond the range of the corrected division."""

import numpy as np
import pytest
import torch

from oracle import pagedkv_oracle as orc
from pkv_torch import to_index, to_numpy, to_torch
from sglang_mlx_amd import kernels

pytestmark = pytest.mark.gpu

FP8 = "fp8_e4m3"


def window_slots(bs, nb, seed):
    """Slots of one call: whole blocks separated by 1 .. bs-1 other tokens, so
    that runs start at every offset of a window."""
    rng = np.random.default_rng(seed)
    free = [b for b in rng.permutation(nb - 1).tolist()]
    whole = lambda b: list(range(b * bs, (b + 1) * bs))  # noqa: E731
    out = []
    for lead in range(bs):
        out += whole(free.pop())
        single = free.pop()
        out += [single * bs + t for t in rng.permutation(bs)[:lead].tolist()]  # scattered in one block
    out += whole(nb - 1)  # the cache's last block
    broken = whole(free.pop())
    out += broken[1:]  # starts at offset 1
    hole = whole(free.pop())
    hole[bs // 2] = -1
    out += hole + whole(free.pop())
    late = whole(free.pop())
    late[-1] = nb * bs + 5  # past the cache
    out += late + whole(free.pop())[:-1]  # ends a token short, at the batch's end
    return np.array(out, dtype=np.int32)


def check(bs, H, D, kv_dtype, cache_dtype, seed, scales=(1.0, 1.0), values=None, nb=None, slots=None):
    x = 16 if cache_dtype == FP8 else 8
    if slots is None:
        nb = 3 * bs + 16
        slots = window_slots(bs, nb, seed)
    rng = np.random.default_rng(seed)
    N = len(slots)
    if values is None:
        raw = rng.standard_normal((2, N, H, D), dtype=np.float32)
    else:
        raw = rng.choice(values, size=(2, N, H, D)).astype(np.float32)
    key, value = (raw if kv_dtype == "float32" else orc.to_storage(raw, kv_dtype))
    top, word = (256, np.uint8) if cache_dtype == FP8 else (65536, np.uint16)
    kc0 = rng.integers(0, top, size=(nb, H, D // x, bs, x)).astype(word)
    vc0 = rng.integers(0, top, size=(nb, H, D, bs)).astype(word)
    kc, vc = to_torch(kc0, cache_dtype), to_torch(vc0, cache_dtype)
    kernels.reshape_and_cache(to_torch(key, kv_dtype), to_torch(value, kv_dtype), kc, vc, to_index(slots),
                              k_scale=scales[0], v_scale=scales[1])
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        # (Slots past the cache are skipped, as padding is.)
        rk, rv = orc.reshape_and_cache_paged5d(key, value, kc0, vc0, np.where(slots < nb * bs, slots, -1), kv_dtype,
                                               cache_dtype, *scales)
    np.testing.assert_array_equal(to_numpy(kc), rk)
    np.testing.assert_array_equal(to_numpy(vc), rv)


@pytest.mark.parametrize("bs", [8, 16, 32])
@pytest.mark.parametrize("H,D", [(1, 32), (3, 80), (2, 120), (5, 128), (2, 256)])
@pytest.mark.parametrize("pair", [("bfloat16", "bfloat16"), ("float32", "float16")])
def test_16_bit(bs, H, D, pair):
    check(bs, H, D, *pair, seed=bs + D)


# Quotients times the scale: ties of every exponent, subnormals and their
# half-way points, the edges 2^-9, 2^-6, 240, 248, 256 and 2^14, zeros.
QUOTIENTS = np.array([s * v for s in (1.0, -1.0)
                      for v in ([0.0, 1e-30, 2.0 ** -10, 2.0 ** -9 * 0.999, 240.0, 247.9, 248.0, 255.0, 256.0, 300.0,
                                 16383.0, 16384.0, 1e30, np.inf]
                                + [(1 + m / 16) * 2.0 ** e for m in range(16) for e in range(-11, 8)])])


@pytest.mark.parametrize("bs", [8, 16, 32])
@pytest.mark.parametrize("H,D", [(1, 32), (3, 80), (3, 128)])
@pytest.mark.parametrize("kv_dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("scales", [(0.05, 0.02), (-0.7, 1.0 / 3.0), (0.125, 2.0), (1e-25, 2.0 ** 61)])
def test_fp8(bs, H, D, kv_dtype, scales):
    with np.errstate(over="ignore"):
        values = (QUOTIENTS * np.float32(scales[0])).astype(np.float32)
    check(bs, H, D, kv_dtype, FP8, seed=bs + D, scales=scales, values=values)


@pytest.mark.parametrize("bs", [8, 16, 32])
@pytest.mark.parametrize("H,D", [(1, 128), (3, 80), (2, 256)])
@pytest.mark.parametrize("pair", [("bfloat16", "bfloat16"), ("float32", "float16"), ("bfloat16", FP8)])
def test_fewer_tokens_than_a_block(bs, H, D, pair):
    nb = 9
    rng = np.random.default_rng(bs + D)
    scales = (0.05, 0.02) if pair[1] == FP8 else (1.0, 1.0)
    for n in (1, 2, bs // 2 + 1, bs - 1):
        whole = np.arange(3 * bs, 3 * bs + n)  # a block's first tokens in order
        mixed = rng.permutation(nb * bs)[:n]
        if n > 2:
            mixed[[0, n // 2]] = -1, nb * bs + 1
        for slots in (whole, mixed, np.arange(nb * bs - n, nb * bs)):
            check(bs, H, D, *pair, seed=n, scales=scales, nb=nb, slots=slots.astype(np.int32))


@pytest.mark.parametrize("bs,N,H,D,kv", [
    # Either side of the lines: one by one up to 2^17 (from float32 2^18)
    # elements, half of that above head size 128; then the search for runs.
    (16, 128, 8, 128, "bfloat16"), (16, 129, 8, 128, "bfloat16"), (32, 64, 8, 256, "bfloat16"),
    (32, 32, 8, 256, "bfloat16"), (8, 33, 8, 256, "bfloat16"), (32, 1023, 1, 128, "bfloat16"),
    (16, 256, 8, 128, "float32"), (16, 257, 8, 128, "float32"), (32, 131, 8, 256, "float32")])
def test_small_calls_with_whole_blocks(bs, N, H, D, kv):
    # Prompts that fill whole blocks and end inside one, and a first token at
    # an offset.
    rng = np.random.default_rng(N + bs)
    nb = 2 * (N // bs) + 12
    free = (rng.permutation(nb - 1) + 1).tolist()
    slots = [free.pop() * bs + bs - 1]
    while len(slots) < N:
        n = int(rng.integers(1, 3 * bs))
        at = [free.pop() for _ in range(min(-(-n // bs), len(free)))] if free else []
        slots += [b * bs + t for b in at for t in range(bs)][:n] if at else [-1] * n
    check(bs, H, D, kv, "float16" if kv == "float32" else kv, seed=N, nb=nb, slots=np.array(slots[:N], dtype=np.int32))


def many_windows(bs, N, seed):
    """(slots, blocks) of at least N tokens: window_slots over several parts of one cache."""
    part, out = 3 * bs + 16, []
    while sum(len(x) for x in out) < N:
        s = window_slots(bs, part, seed + len(out))
        out.append(np.where(s >= part * bs, 1 << 30, np.where(s < 0, -1, s + len(out) * part * bs)))
    return np.concatenate(out).astype(np.int32), len(out) * part


@pytest.mark.parametrize("bs", [8, 16, 32])
@pytest.mark.parametrize("H,D", [(7, 64), (3, 32), (5, 80), (2, 128), (9, 16)])
@pytest.mark.parametrize("pair", [("bfloat16", "bfloat16"), ("float32", "float16"), ("bfloat16", FP8)])
def test_large_calls_of_several_heads_a_workgroup(bs, H, D, pair):
    # From 8192 (token, head) pairs on a workgroup takes a window of as many
    # heads as give its threads a run task each; odd numbers of heads leave the
    # last group short.
    slots, nb = many_windows(bs, -(-8192 // H), seed=bs + D)
    assert len(slots) * H >= 8192
    check(bs, H, D, *pair, seed=3, scales=(0.05, 0.02) if pair[1] == FP8 else (1.0, 1.0), nb=nb, slots=slots)


@pytest.mark.parametrize("kv_dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("scale", [1.0, 0.05, 0.02, -0.7, 1.0 / 3.0, 0.125, 2.0, 3e-3, 1e3, 7e-5, 2.0 ** -60, 2.0 ** 60,
                                   1e-25])
def test_fp8_codes_of_every_16_bit_pattern(kv_dtype, scale):
    # 64 tokens x 8 heads x 128: half of the tokens fill blocks, half are scattered.
    rng = np.random.default_rng(4)
    key = np.arange(65536, dtype=np.uint16).reshape(64, 8, 128)
    value = rng.permutation(65536).astype(np.uint16).reshape(64, 8, 128)
    slots = np.concatenate([np.arange(32), 32 + rng.permutation(96)[:32]]).astype(np.int32)
    kc0, vc0 = np.zeros((8, 8, 8, 16, 16), np.uint8), np.zeros((8, 8, 128, 16), np.uint8)
    kc, vc = to_torch(kc0, FP8), to_torch(vc0, FP8)
    kernels.reshape_and_cache(to_torch(key, kv_dtype), to_torch(value, kv_dtype), kc, vc, to_index(slots),
                              k_scale=scale, v_scale=scale)
    with np.errstate(all="ignore"):
        rk, rv = orc.reshape_and_cache_paged5d(key, value, kc0, vc0, slots, kv_dtype, FP8, scale, scale)
    np.testing.assert_array_equal(to_numpy(kc), rk)
    np.testing.assert_array_equal(to_numpy(vc), rv)
