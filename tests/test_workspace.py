"""Scratch handed to the library's entries: one per thread and stream, bounded
while calls grow, no fill where none is needed, none shared with a captured graph.
The bookkeeping is tested on the CPU; the split decode, which makes two launches
over its scratch, also runs from threads, on streams and in a captured graph."""

from __future__ import annotations

import threading

import pytest

torch = pytest.importorskip("torch")
from autotuner_runtime import hip  # noqa: E402

CPU = torch.device("cpu")


@pytest.fixture
def capturing(monkeypatch):
    """Sets whether the current stream counts as capturing."""
    state = {"on": False}
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state["on"])
    return lambda on: state.update(on=on)


def _in_thread(f):
    out = []
    t = threading.Thread(target=lambda: out.append(f()))
    t.start()
    t.join()
    return out[0]


def test_threads_on_one_stream_own_their_scratch(capturing):
    def take():
        return hip._workspace("sdpa", CPU, 11, 5000)

    mine, other = take(), _in_thread(take)
    assert take() is mine
    assert other is not mine and other.data_ptr() != mine.data_ptr()
    assert hip._workspace("sdpa", CPU, 12, 5000) is not mine


def test_a_growing_call_keeps_one_buffer(capturing):
    """A conversation whose scratch grows a little at a time: a logarithm of
    buffers, the outgrown ones not held."""
    held = len(hip._retired)
    sizes = {hip._workspace("sdpa", CPU, 13, 4096 + 1000 * i).numel() for i in range(1000)}
    assert len(sizes) <= 10
    assert max(sizes) <= 2 * (4096 + 1000 * 999)
    assert len(hip._retired) == held


def test_captured_scratch_is_its_graphs_own(capturing):
    eager = hip._workspace("sdpa", CPU, 14, 5000, 1 << 20)
    capturing(True)
    with hip.graph_workspaces():
        a = hip._workspace("sdpa", CPU, 14, 5000, 1 << 20)
        assert a.numel() == 5000                      # the size asked for
        assert hip._workspace("sdpa", CPU, 14, 4000) is a
        assert hip._workspace("sdpa", CPU, 15, 4000) is not a   # a forked stream
        big = hip._workspace("sdpa", CPU, 14, 9000)
        assert any(t is a for t in hip._retired)      # its address is in earlier nodes
    with hip.graph_workspaces():
        b = hip._workspace("sdpa", CPU, 14, 5000)
    lone = [hip._workspace("sdpa", CPU, 14, 5000) for _ in range(2)]
    assert all(any(t is x for t in hip._retired) for x in lone)
    assert len({t.data_ptr() for t in (eager, a, big, b, *lone)}) == 6


def test_only_tickets_are_zero_filled(capturing, monkeypatch):
    """Under capture a fill is a node of the graph."""
    def refuse(*a, **k):
        raise AssertionError("a fill")

    for on in (False, True):
        capturing(on)
        assert not hip._workspace("gelu_mlp", CPU, 16 + on, 5000, zero=True).any()
        with monkeypatch.context() as m:
            m.setattr(torch, "zeros", refuse)
            for kind in ("sdpa", "qmm"):
                hip._workspace(kind, CPU, 16 + on, 5000)


def _decode_inputs(seed, Lk=3000, Lq=1):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    r = lambda h, n: torch.randn((1, h, n, 128), generator=gen, device="cuda").bfloat16()  # noqa: E731
    return r(32, Lq), r(8, Lk), r(8, Lk)


def _sdpa(t):
    from autotuner_runtime import ops
    return ops.scaled_dot_product_attention(*t, 128 ** -0.5)


@pytest.mark.gpu
def test_split_decode_from_two_threads():
    """Two threads on the default stream, each its own conversation."""
    sets = [_decode_inputs(1), _decode_inputs(2, 5000, 4)]
    want = [_sdpa(t) for t in sets]
    torch.cuda.synchronize()
    bad = []

    def loop(i):
        for _ in range(300):
            if not torch.equal(_sdpa(sets[i]), want[i]):
                bad.append(i)

    threads = [threading.Thread(target=loop, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.gpu
def test_split_decode_on_two_streams():
    sets = [_decode_inputs(3), _decode_inputs(4, 6000)]
    want = [_sdpa(t) for t in sets]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(50):
        for i in range(2):
            with torch.cuda.stream(streams[i]):
                got[i].append(_sdpa(sets[i]))
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(o, want[i]) for o in got[i])


@pytest.mark.gpu
def test_split_decode_in_a_captured_graph():
    """Two calls a graph, replayed with eager calls of the same stream between;
    with and without a scope."""
    import contextlib

    sets = [_decode_inputs(5), _decode_inputs(6, 4100)]
    for scope in (hip.graph_workspaces, contextlib.nullcontext):
        want = [_sdpa(t) for t in sets]
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with scope(), torch.cuda.graph(g):
            out = [_sdpa(t) for t in sets]
        for rep in range(4):
            for t in sets:
                t[0].copy_(torch.roll(t[0], 1, dims=-1))   # other queries each replay
            want = [_sdpa(t) for t in sets]
            for o in out:
                o.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(out, want)), rep
