"""Decode scratch and HIP graphs: a graph's scratch does not depend on another
graph or an eager call having run, and a graph keeps the scratch it was captured
with.  (Each call here splits its contexts, so it counts arrivals and leaves
partial states in the scratch.)"""

import pytest
import torch

from sglang_mlx_amd import _ext, _lib

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def decode(tokens=2000, B=2, Hq=8, Hkv=2, D=64, bs=16, seed=3):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    nb = 160
    k = torch.randn((nb, Hkv, D // 8, bs, 8), generator=g, device=DEV).half()
    v = torch.randn((nb, Hkv, D, bs), generator=g, device=DEV).half()
    q = torch.randn((B, Hq, D), generator=g, device=DEV).half()
    table = torch.randint(0, nb, (B, -(-tokens // bs)), generator=g, device=DEV, dtype=torch.int32)
    lens = torch.arange(tokens, tokens - B, -1, dtype=torch.int32, device=DEV)
    return lambda: _ext.paged_attention_v1(q, k, v, table, lens, Hkv, 0.125, bs, tokens)


def capture(call, stream):
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = call()
    return graph, out


def test_graphs_captured_on_one_stream_replay_alone():
    calls = [decode(), decode(tokens=1500, seed=4), decode(tokens=2400, B=5, seed=5)]
    refs = [c() for c in calls]
    stream = torch.cuda.Stream()
    graphs = [capture(c, stream) for c in calls]
    # Memory that a capture allocated holds anything until the graph has run.
    key = (0, stream.cuda_stream)
    for t in [_ext._ws_cache.get(key)] + [t for _, t in getattr(_ext, "_ws_captured", {}).values()]:
        if t is not None:
            t.fill_(7)
    torch.cuda.synchronize()
    for i in (2, 1, 0, 2, 1):
        graph, out = graphs[i]
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, refs[i]), i
        assert torch.equal(calls[i](), refs[i])
    # An eager call on the stream the graphs were captured on.
    with torch.cuda.stream(stream):
        out = calls[0]()
    stream.synchronize()
    assert torch.equal(out, refs[0])


def test_a_graph_keeps_its_scratch():
    stream = torch.cuda.Stream()
    call, larger = decode(), decode(tokens=2500, B=64, Hq=64)
    ref = call()
    with torch.cuda.stream(stream):
        call()  # the stream's scratch, which the capture then uses
    stream.synchronize()
    held = _ext._ws_cache[(0, stream.cuda_stream)].numel()
    graph, out = capture(call, stream)
    with torch.cuda.stream(stream):
        larger()
        assert _ext._ws_cache[(0, stream.cuda_stream)].numel() > held
        others = [torch.full((held,), 5, dtype=torch.uint8, device=DEV) for _ in range(8)]
    stream.synchronize()
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
        assert all(bool((t == 5).all()) for t in others)


def test_outgrown_scratch_is_bounded():
    stream = torch.cuda.Stream().cuda_stream
    before = len(_ext._ws_outgrown)
    sizes = [(1 << 17) + 4096 * i for i in range(300)]
    for n in sizes:
        assert _ext._decode_scratch(torch.device(DEV), stream, n).numel() >= n
    outgrown = _ext._ws_outgrown[before:]
    now = _ext._ws_cache[(0, stream)]
    assert sum(t.numel() for t in outgrown) < now.numel() < 2 * sizes[-1]
    assert not now[:_lib.PKV_COUNTER_BYTES].any()
