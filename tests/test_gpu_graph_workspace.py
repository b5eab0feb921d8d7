"""K-split calls of the torch ops under HIP graph capture: their workspace (arrival counters and fp32
partials) belongs to the capture. Whole outputs of replays against the eager result, bit for bit (the
split is deterministic)."""

import pytest
import torch

from gpu_util import lib

pytestmark = pytest.mark.gpu

SMALL, LARGE = (33, 128, 2480), (97, 4160, 3984)  # both split over K; LARGE needs a larger workspace


def _call(cuda, hk, M, N, K, seed=0):
    assert lib().feather_scaled_mm_any_m_workspace_size(M, N, K) > 0
    g = torch.Generator(device=cuda).manual_seed(M + N + K + seed)
    a = torch.randn(M, K, generator=g, device=cuda).half()
    bp = (torch.randn(K // 16, N, 16, generator=g, device=cuda) * 0.1).to(torch.float8_e5m2)
    return lambda: hk.scaled_mm_hip_any_m(a, bp, None, None, torch.float16)


def _dirty_pool(cuda, stream):
    """A graph memory pool whose free memory is not zero, and the graph that filled it."""
    pool, graph = torch.cuda.graph_pool_handle(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, pool=pool, stream=stream):
        junk = torch.full((64 << 20,), 0x5A, dtype=torch.uint8, device=cuda)
        del junk
    graph.replay()
    torch.cuda.synchronize()
    return pool, graph


def _eager(fn):
    y = fn()
    torch.cuda.synchronize()
    return y


def test_graph_does_not_rest_on_another_graphs_replay(cuda, hk):
    """Two graphs captured on one stream, only the second replayed, in a memory pool that a first graph
    has filled with non-zero bytes: the second one's arrival counters are zeroed by its own replay."""
    fn = _call(cuda, hk, *LARGE)
    want = _eager(fn)
    stream, first, second = torch.cuda.Stream(), torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    pool, dirty = _dirty_pool(cuda, stream)
    out = torch.zeros_like(want)
    with torch.cuda.graph(first, pool=pool, stream=stream):
        fn()
    with torch.cuda.graph(second, pool=pool, stream=stream):
        out.copy_(fn())
    for rep in range(3):
        out.zero_()
        second.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), rep
        assert torch.equal(_eager(fn), want), rep


def test_eager_call_after_a_capture_that_was_not_replayed(cuda, hk):
    """An eager call on a stream whose first K-split call was captured and not replayed."""
    fn = _call(cuda, hk, *LARGE)
    want = _eager(fn)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    pool, dirty = _dirty_pool(cuda, stream)
    with torch.cuda.graph(graph, pool=pool, stream=stream):
        fn()
    with torch.cuda.stream(stream):
        y = fn()
    torch.cuda.synchronize()
    assert torch.equal(y, want)


def test_replays_after_the_eager_workspace_has_grown(cuda, hk):
    """A graph captured on a stream with a small eager workspace; an eager call then needs a larger one and
    new tensors take the memory it gave back: replays neither write those nor read them."""
    small, large = _call(cuda, hk, *SMALL), _call(cuda, hk, *LARGE)
    want, want_large = _eager(small), _eager(large)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        small()
    torch.cuda.synchronize()
    out = torch.zeros_like(want)
    with torch.cuda.graph(graph, stream=stream):
        out.copy_(small())
    with torch.cuda.stream(stream):
        assert torch.equal(large(), want_large)
        held = [torch.full((1 << 20,), 0x5A, dtype=torch.uint8, device=cuda) for _ in range(64)]
    torch.cuda.synchronize()
    for rep in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), rep
        assert all(bool((t == 0x5A).all()) for t in held), rep
        with torch.cuda.stream(stream):
            assert torch.equal(large(), want_large)
        torch.cuda.synchronize()


def test_graphs_of_one_stream_replayed_on_two(cuda, hk):
    """Graphs captured on one stream share no workspace: replayed on two streams at once, each gives its result."""
    fns = [_call(cuda, hk, *LARGE), _call(cuda, hk, *LARGE, seed=1)]
    wants = [_eager(f) for f in fns]
    outs = [torch.zeros_like(w) for w in wants]
    stream = torch.cuda.Stream()
    graphs = [torch.cuda.CUDAGraph() for _ in fns]
    for g, f, o in zip(graphs, fns, outs):
        with torch.cuda.graph(g, stream=stream):
            for _ in range(8):
                o.copy_(f())
    streams = [torch.cuda.Stream() for _ in fns]
    for rep in range(3):
        for o in outs:
            o.zero_()
        torch.cuda.synchronize()
        for g, s in zip(graphs, streams):
            with torch.cuda.stream(s):
                g.replay()
        torch.cuda.synchronize()
        for o, w in zip(outs, wants):
            assert torch.equal(o, w), rep
