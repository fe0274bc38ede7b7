"""The cached workspaces of the prefill and its backward: calls of two streams never share one,
calls of two threads on one stream do not enqueue between each other's launches, and a graph
holds memory of its own."""

import math
import threading

import pytest
import torch

from ananta_ocr_amd import ops

DEV = "cuda"


@pytest.fixture
def host(monkeypatch):
    """The cache on host memory, with the stream and capture state the test sets."""
    state = [0, False]
    monkeypatch.setattr(ops, "_device_stream", lambda device: tuple(state))
    ops.release_workspaces()
    yield state
    ops.release_workspaces()


def test_one_buffer_per_stream(host):
    a = ops.cached_workspace("t", 1000, "cpu")
    assert ops.cached_workspace("t", 500, "cpu") is a
    assert ops.cached_workspace("u", 500, "cpu") is not a
    host[0] = 5
    b = ops.cached_workspace("t", 1000, "cpu")
    assert b.data_ptr() != a.data_ptr()
    host[0] = 0
    assert ops.cached_workspace("t", 1000, "cpu") is a


def test_the_cache_is_bounded(host):
    for s in range(20):
        host[0] = s
        for kind in "tu":
            ops.cached_workspace(kind, 1000, "cpu")
    assert len(ops._WORKSPACES) == 2 * ops.WORKSPACE_LIMIT
    assert {k[2] for k in ops._WORKSPACES} == set(range(20 - ops.WORKSPACE_LIMIT, 20))
    ops.release_workspaces("cpu")
    assert not ops._WORKSPACES


def test_a_recorded_call_has_its_own_buffer(host):
    a = ops.cached_workspace("t", 1000, "cpu")
    host[1] = True
    b = ops.cached_workspace("t", 2000, "cpu")
    assert b.numel() == 2000 and list(ops._WORKSPACES.values()) == [a]


def _calls():
    """Two prefills and backwards of different shapes, as functions of nothing."""
    out = []
    for i, (S, bs, lw, K) in enumerate([(6000, 64, 256, 16), (5000, 32, 128, 12)]):
        g = torch.Generator().manual_seed(i)
        q, k, v, do = ((torch.randn(1, 2, S, 128, generator=g) * 0.6).bfloat16().to(DEV)
                       for _ in range(4))
        nblk = (S + bs - 1) // bs
        idx = torch.stack([torch.randperm(nblk, generator=g)[:K] for _ in range(S)])[None]
        r = [idx.to(torch.int32).to(DEV), torch.randn(1, S, K, generator=g).to(DEV),
             torch.ones(1, S, K, dtype=torch.uint8, device=DEV)]
        a = (bs, lw, 1 / math.sqrt(128))

        def both(q=q, k=k, v=v, do=do, r=r, a=a):
            o, lse = ops.attn_prefill(q, k, v, *r, *a, return_lse=True)
            return o, *ops.attn_prefill_backward(q, k, v, o, lse, do, *r, *a)
        out.append(both)
    return out


def _close(got, ref):
    """The output's bits; the gradients to the order of a block's pairs, whose places are
    handed out by atomics (bf16 results of sums in another order)."""
    assert torch.equal(got[0], ref[0])
    for x, y in zip(got[1:], ref[1:]):
        err = (x.double() - y.double()).norm() / y.double().norm()
        assert err <= 1e-3, float(err)


@pytest.mark.gpu
def test_calls_of_two_streams():
    calls = _calls()
    ref = [f() for f in calls]
    streams = [torch.cuda.Stream() for _ in calls]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(4):
        for f, s, o in zip(calls, streams, got):
            with torch.cuda.stream(s):
                o.append(f())
    torch.cuda.synchronize()
    for o, r in zip(got, ref):
        for x in o:
            _close(x, r)


@pytest.mark.gpu
def test_calls_of_two_threads_on_one_stream():
    calls = _calls()
    ref = [f() for f in calls]
    torch.cuda.synchronize()
    got = [[], []]

    def loop(f, o):
        for _ in range(6):
            o.append(f())
    threads = [threading.Thread(target=loop, args=a) for a in zip(calls, got)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for o, r in zip(got, ref):
        assert len(o) == 6
        for x in o:
            _close(x, r)


@pytest.mark.gpu
def test_recorded_call_beside_calls_outside():
    """A prefill recorded into a graph and replayed on one stream while another stream's larger
    calls take, grow and give back the cached buffers."""
    large, small = _calls()
    ref = [small(), large()]
    ops.release_workspaces()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        small()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = small()
    for i in range(4):
        with torch.cuda.stream(side):
            graph.replay()
        got = large()
        torch.cuda.synchronize()
        _close(out, ref[0])
        _close(got, ref[1])
        if i == 1:
            ops.release_workspaces()
