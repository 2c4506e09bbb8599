"""Calls of newton_schulz that overlap: on two streams, as a replay of a caller's
graph beside eager calls, and from several threads on one stream. Each gives the
bits of the same call alone. The shapes take the recorded launches (not the
one-launch form), long enough for the GPU work of two calls to run at once."""

from __future__ import annotations

import threading

import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from himuon_amd.engine import newton_schulz

DEV = "cuda"
SHAPE = (24, 512, 1024)


def _inputs(shape, n, dtype=torch.float32):
    g = torch.Generator().manual_seed(n)
    return [(torch.randn(shape, generator=g) * 1e-3).to(dtype).to(DEV) for _ in range(n)]


@pytest.mark.parametrize("shape", [SHAPE, (1024, 700)])
def test_two_streams_at_once(shape):
    xs = _inputs(shape, 4)
    want = [newton_schulz(x) for x in xs]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for _ in range(3):
        outs = []
        for k, x in enumerate(xs):
            with torch.cuda.stream(streams[k % 2]):
                outs.append(newton_schulz(x))
        torch.cuda.synchronize()
        for o, w in zip(outs, want):
            assert torch.equal(o, w)


def test_a_callers_graph_beside_eager_calls():
    a, b, c = _inputs(SHAPE, 3)
    want = [newton_schulz(x) for x in (a, b, c)]
    static = a.clone()
    graph = torch.cuda.CUDAGraph()
    # (a shape of its own besides, which no call before the capture has prepared)
    small = _inputs((5, 300, 260), 1)[0]
    with torch.cuda.graph(graph):
        out = newton_schulz(static)
        out_small = newton_schulz(small.transpose(1, 2))
    want_small = newton_schulz(small.transpose(1, 2))
    other = torch.cuda.Stream()
    for k in (0, 1, 2, 0):
        static.copy_((a, b, c)[k])
        torch.cuda.synchronize()
        graph.replay()
        with torch.cuda.stream(other):
            beside = newton_schulz((b, c, a)[k])
        torch.cuda.synchronize()
        assert torch.equal(out, want[k]) and torch.equal(beside, want[(k + 1) % 3])
        assert torch.equal(out_small, want_small)


def test_threads_on_one_stream():
    shape = (2, 256, 384)
    xs = _inputs(shape, 4)
    want = [newton_schulz(x) for x in xs]
    bad = []

    def work(x, w):
        for _ in range(40):
            if not torch.equal(newton_schulz(x), w):
                bad.append(1)

    threads = [threading.Thread(target=work, args=p) for p in zip(xs, want)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not bad and not any(t.is_alive() for t in threads)
