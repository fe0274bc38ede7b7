"""The decode step's cached workspace: its routing words and partials are never shared by
steps of two streams or threads, nor by a graph and the steps outside it."""

import threading

import pytest
import torch

from ananta_ocr_amd import ops

DEV = "cuda"


@pytest.fixture
def host(monkeypatch):
    """The cache on host memory, with the capture state the test sets."""
    state = {"capturing": False}
    monkeypatch.setattr(torch._C, "_cuda_isCurrentStreamCapturing", lambda: state["capturing"],
                        raising=False)
    ops.release_workspaces()
    yield state
    ops.release_workspaces()


def _get(nbytes=10000, stream=0):
    return ops._step_workspace(nbytes, torch.device("cpu"), 4, stream)


def test_one_buffer_per_stream_and_thread(host):
    a = _get()
    assert a.numel() >= 10000 and not a.any()
    assert _get(5000) is a
    b = _get(stream=7)
    other = []
    t = threading.Thread(target=lambda: other.append(_get(stream=7)))
    t.start()
    t.join()
    assert len({x.data_ptr() for x in (a, b, other[0])}) == 3
    assert _get() is a and _get(stream=7) is b
    big = _get(50000)
    assert big.numel() >= 50000 and not big.any() and _get() is big


def test_the_cache_is_bounded_and_given_back(host):
    n = ops.STEP_WORKSPACE_LIMIT
    bufs = [_get(stream=s) for s in range(3 * n)]
    assert len(ops._STEP_WORKSPACES) == n
    assert all(_get(stream=s) is bufs[s] for s in range(2 * n, 3 * n))
    assert _get(stream=0) is not bufs[0]
    assert ops.cached_workspace_bytes() == n * bufs[0].numel()
    ops.release_workspaces("cpu")
    assert not ops._STEP_WORKSPACES and ops.cached_workspace_bytes() == 0


def test_partials_of_one_step_end_below_the_words_of_another(host):
    """A step of few sequences and many heads after one of more sequences: its partials, which
    fill its own size but for its own words, end below the words of any step (256 bytes for
    each of up to 255 sequences, at the buffer's end)."""
    words = 255 * 256
    ops._step_workspace(200000, torch.device("cpu"), 8, 0)
    size = next(iter(ops._STEP_WORKSPACES.values())).numel()
    for nbytes in range(size - 80000, size + 3000, 1000):
        buf = ops._step_workspace(nbytes, torch.device("cpu"), 1, 0)
        assert nbytes - 256 <= buf.numel() // 256 * 256 - words
        buf = ops.decode_step_workspace(2, 300, 128, 64, nbytes // 500, "cpu")
        assert buf.numel() // 256 * 256 - words >= ops._step_workspace_size(
            2, 300, 128, 64, nbytes // 500) - 512


def test_a_recorded_step_has_its_own_buffer(host):
    a = _get()
    host["capturing"] = True
    b = _get(10001)
    assert b.data_ptr() != a.data_ptr() and list(ops._STEP_WORKSPACES.values())[0] is a
    assert b.numel() % 256 == 0 and not b[-4 * 256:].any()
    assert len(ops._STEP_WORKSPACES) == 1


def _steps(n):
    """n sets of inputs of different sizes, each with a function of one step."""
    from ananta_ocr_amd import pipeline
    out = []
    for i in range(n):
        g = torch.Generator().manual_seed(40 + i)
        B, H, S, bs = 3 + i, 4, 1500 + 700 * i, 64
        q, k, v = ((torch.randn(B, H, *m, 128, generator=g)).bfloat16().to(DEV)
                   for m in ((), (S,), (S,)))
        iq, ik = torch.randn(B, 128, generator=g).to(DEV), torch.randn(B, S, 128, generator=g).to(DEV)
        hc = (torch.randn(128, generator=g) * 0.1).to(DEV)
        st = pipeline.init_decode_state(ik, hc, bs, (S + bs - 1) // bs)
        out.append(lambda a=(st, q, k, v, iq, ik, hc, bs, 8, 100.0, 1e-4, 1.0, 8, 8):
                   pipeline.decode_step(*a))
    return out


@pytest.mark.gpu
def test_steps_of_two_streams():
    steps = _steps(2)
    ref = [f() for f in steps]
    streams = [torch.cuda.Stream() for _ in steps]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(20):
        for f, s, o in zip(steps, streams, got):
            with torch.cuda.stream(s):
                o.append(f())
    torch.cuda.synchronize()
    for o, r in zip(got, ref):
        assert all(torch.equal(x, r) for x in o)


@pytest.mark.gpu
def test_steps_of_two_threads_on_one_stream():
    steps = _steps(2)
    ref = [f() for f in steps]
    torch.cuda.synchronize()
    got = [[], []]

    def loop(f, o):
        for _ in range(30):
            o.append(f())
    threads = [threading.Thread(target=loop, args=a) for a in zip(steps, got)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for o, r in zip(got, ref):
        assert len(o) == 30 and all(torch.equal(x, r) for x in o)


@pytest.mark.gpu
def test_recorded_steps_beside_steps_outside():
    """A step recorded without a workspace, replayed on another stream than the one whose
    larger steps make the cached buffer grow."""
    small, large = _steps(2)
    ref = [small(), large()]
    ops.release_workspaces()
    small()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = small()
    side = torch.cuda.Stream()
    for _ in range(5):
        with torch.cuda.stream(side):
            graph.replay()
        got = large()
        torch.cuda.synchronize()
        assert torch.equal(out, ref[0]) and torch.equal(got, ref[1])
