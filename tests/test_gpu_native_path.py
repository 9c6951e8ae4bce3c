"""The native call path (_native.so) against the Python path it stands in for:
plain calls are taken and give the same bytes, every other form is handed back
and gives what the Python path gives, refusals keep their messages, streams,
tensor subclasses and function modes are as before, and other threads run
during a call."""

import sys
import threading

import pytest
import torch
from torch.overrides import TorchFunctionMode

from sglang_mlx_amd import _ext

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def decode_args(q=torch.bfloat16, cache=torch.bfloat16, rows=False, B=3, Hq=8, Hkv=2, D=64, bs=16):
    g = torch.Generator(device=DEV)
    g.manual_seed(5)

    def rand(shape, dt):
        x = torch.randn(shape, generator=g, device=DEV)
        return (x * 20).to(torch.float8_e4m3fn).view(dt) & 0xB7 if dt == torch.uint8 else x.to(dt)  # finite codes

    nb, x = 40, 16 // torch.empty((), dtype=cache).element_size()
    if rows:
        k, v, bs = rand((nb * 16, Hkv, D), cache), rand((nb * 16, Hkv, D), cache), 1
        table = torch.randint(0, nb * 16, (B, 160), generator=g, device=DEV, dtype=torch.int32)
    else:
        k, v = rand((nb, Hkv, D // x, bs, x), cache), rand((nb, Hkv, D, bs), cache)
        table = torch.randint(0, nb, (B, 10), generator=g, device=DEV, dtype=torch.int32)
    lens = torch.tensor([1, 77, 160], dtype=torch.int32, device=DEV)[:B]
    return [rand((B, Hq, D), q), k, v, table, lens, Hkv, 0.125, bs, 160]


def append_args(layout="paged", kv=torch.bfloat16, cache=torch.bfloat16, N=19, H=2, D=64, bs=16):
    g = torch.Generator(device=DEV)
    g.manual_seed(6)
    key, value = (torch.randn((N, H, D), generator=g, device=DEV).to(kv) for _ in range(2))
    x = 16 // torch.empty((), dtype=cache).element_size()
    shapes = [(8, H, D // x, bs, x), (8, H, D, bs)] if layout == "paged" else [(8 * bs, H, D)] * 2
    return [key, value] + [torch.zeros(s, dtype=cache, device=DEV) for s in shapes] + \
        [torch.arange(3, 3 + N, dtype=torch.int32, device=DEV)]


def python_path(monkeypatch, fn, *args, **kw):
    with monkeypatch.context() as m:
        m.setattr(_ext, "_native", None)
        return fn(*args, **kw)


def native_decode(args, alibi=None, partition=0):
    return _ext._native.paged_attention(_ext._ws_cache, *args, alibi, partition, 1.0, 1.0)


@pytest.mark.parametrize("q,cache,rows", [(torch.bfloat16, torch.bfloat16, False), (torch.float16, torch.float16, True),
                                          (torch.float32, torch.float16, False), (torch.float32, torch.float32, False),
                                          (torch.bfloat16, torch.uint8, False)])
def test_decode_is_taken_and_equal(monkeypatch, q, cache, rows):
    args = decode_args(q, cache, rows)
    ref = python_path(monkeypatch, _ext.paged_attention_v1, *args)  # (allocates the scratch too)
    slopes = torch.rand(8, device=DEV)
    refa = python_path(monkeypatch, _ext.paged_attention_v1, *args, alibi_slopes=slopes)
    assert isinstance(native_decode(args), torch.Tensor)
    assert torch.equal(_ext.paged_attention_v1(*args), ref)
    assert torch.equal(_ext.paged_attention_v1(*args, alibi_slopes=slopes), refa)
    assert torch.equal(_ext.paged_attention_v2(*args, partition_size=32),
                       python_path(monkeypatch, _ext.paged_attention_v2, *args, partition_size=32))


def test_other_forms_go_to_the_python_path(monkeypatch):
    args = decode_args()
    ref = _ext.paged_attention_v1(*args)
    wide = torch.zeros((3, 8, 66), dtype=torch.bfloat16, device=DEV)
    wide[..., :64] = args[0]

    class Sub(torch.Tensor):
        pass

    forms = {0: [wide[..., :64], args[0].as_subclass(Sub)], 3: [args[3].long(), args[3].t().contiguous().t()],
             4: [args[4].long()], 5: [torch.tensor(2)], 6: [torch.tensor(0.125)], 8: [True + 159]}
    for i, values in forms.items():
        for v in values:
            other = args[:i] + [v] + args[i + 1:]
            if i != 8:
                assert native_decode(other) is None, i
            assert torch.equal(_ext.paged_attention_v1(*other).as_subclass(torch.Tensor), ref), i
    seen = []

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, a=(), kw=None):
            seen.append(func)
            return func(*a, **(kw or {}))

    with Mode():
        assert torch.equal(_ext.paged_attention_v1(*args), ref)
    assert torch.empty in seen


@pytest.mark.parametrize("change,msg", [(dict(i=5, v=3), "divisible"), (dict(i=7, v=8), "block_size"),
                                        (dict(i=8, v=161), "block table capacity"), (dict(i=8, v=0), "positive")])
def test_refusals_keep_their_messages(change, msg):
    args = decode_args()
    _ext.paged_attention_v1(*args)
    args[change["i"]] = change["v"]
    with pytest.raises(ValueError, match=msg):
        _ext.paged_attention_v1(*args)
    with pytest.raises(RuntimeError, match="GPU-only"):
        _ext.paged_attention_v1(*[a.cpu() if isinstance(a, torch.Tensor) else a for a in decode_args()])


@pytest.mark.parametrize("layout", ["paged", "token"])
@pytest.mark.parametrize("kv,cache", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.float16),
                                      (torch.float16, torch.uint8)])
def test_append_is_taken_and_equal(monkeypatch, layout, kv, cache):
    scales = dict(k_scale=0.05, v_scale=0.5) if cache == torch.uint8 else {}
    a, b = append_args(layout, kv, cache), append_args(layout, kv, cache)
    out = _ext.reshape_and_cache(*a, **scales)
    assert out[0] is a[2] and out[1] is a[3]
    python_path(monkeypatch, _ext.reshape_and_cache, *b, **scales)
    assert torch.equal(a[2], b[2]) and torch.equal(a[3], b[3]) and bool(a[2].any())
    assert _ext._native.reshape_and_cache(*a, 0.05, 0.5) is not None
    # A strided source (rows of a wider buffer), one that needs a copy, int64 slots.
    wide = torch.zeros((19, 2 * 64 + 32), dtype=kv, device=DEV)
    wide[:, :128] = a[0].view(19, 128)
    for key, slots, native in ((wide[:, :128].view(19, 2, 64), a[4], True),
                               (a[0].transpose(0, 1).contiguous().transpose(0, 1), a[4], False),
                               (a[0], a[4].long(), False)):
        c = append_args(layout, kv, cache)
        assert (_ext._native.reshape_and_cache(key, c[1], c[2], c[3], slots, 0.05, 0.5) is not None) == native
        _ext.reshape_and_cache(key, c[1], c[2], c[3], slots, **(scales or {}))
        assert torch.equal(c[2], a[2])


def test_append_refusals_keep_their_messages():
    a = append_args()
    with pytest.raises(ValueError, match="key and value dtypes differ"):
        _ext.reshape_and_cache(a[0], a[1].half(), *a[2:])
    with pytest.raises(ValueError, match="contiguous"):
        _ext.reshape_and_cache(a[0], a[1], a[2], a[3].transpose(2, 3).contiguous().transpose(2, 3), a[4])
    with pytest.raises(RuntimeError, match="GPU-only"):
        _ext.reshape_and_cache(*[t.cpu() for t in a])


def test_side_stream_uses_its_own_scratch():
    args = decode_args()
    ref = _ext.paged_attention_v1(*args)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        outs = [_ext.paged_attention_v1(*args) for _ in range(3)]
    side.synchronize()
    assert all(torch.equal(o, ref) for o in outs)
    assert (0, side.cuda_stream) in _ext._ws_cache


@pytest.mark.parametrize("call", ["decode", "append"])
def test_other_threads_run_during_a_call(call):
    # With this switch interval a thread that waits for the interpreter gets it
    # only where the running thread gives it up by itself.
    args = decode_args() if call == "decode" else append_args()
    if call == "decode":
        _ext.paged_attention_v1(*args)  # (allocates the scratch)
        native, full = _ext._native.paged_attention, (_ext._ws_cache, *args, None, 0, 1.0, 1.0)
    else:
        native, full = _ext._native.reshape_and_cache, (*args, 1.0, 1.0)
    torch.cuda.synchronize()
    ran, go = [], threading.Event()

    def other():
        go.wait()
        ran.append(True)

    t = threading.Thread(target=other)
    t.start()
    interval = sys.getswitchinterval()
    sys.setswitchinterval(1000.0)
    try:
        go.set()
        for calls in range(20000):
            if ran:
                break
            assert native(*full) is not None
    finally:
        sys.setswitchinterval(interval)
    seen = bool(ran)
    t.join()
    assert seen
