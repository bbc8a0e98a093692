"""Siddon forwards and solves of one fan plan with many rays on several streams:
none waits for what is queued on another stream, and all return the bits of
the plain order."""
import time

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _busy(stream):
    """Queues some 0.3 s of one idle wave on the stream."""
    if not hasattr(_busy, "cycles"):
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        torch.cuda._sleep(1000)
        e[0].record()
        torch.cuda._sleep(1_000_000)
        e[1].record()
        torch.cuda.synchronize()
        _busy.cycles = int(1_000_000 * 300 / max(e[0].elapsed_time(e[1]), 1e-3))
    with torch.cuda.stream(stream):
        torch.cuda._sleep(_busy.cycles)


def _waits(call):
    """Whether a call and what it returns waited for a stream that _busy filled."""
    t = time.perf_counter()
    call()
    return time.perf_counter() - t > 0.15


@pytest.fixture
def streams(gpu):
    """Two streams that the device runs side by side (they may share a queue)."""
    x = torch.zeros(64, device=gpu)
    for _ in range(6):
        a, b = torch.cuda.Stream(), torch.cuda.Stream()
        torch.cuda.synchronize()
        _busy(a)
        with torch.cuda.stream(b):
            x.add_(1)
        apart = not _waits(b.synchronize)
        torch.cuda.synchronize()
        if apart:
            return a, b
    pytest.skip("no two streams ran side by side")


def _case(gpu):
    from framelab_amd import geometry as G
    from framelab_amd.projector import Projector
    P = Projector(G.fan_para(600, 260, N=(130, 122), SO=4.0, OD=4.0, Ly=G.full_fan_width()))
    x = torch.from_numpy(np.random.default_rng(1).random(P.vol_shape, dtype=np.float32)).to(gpu)
    y = P.forward(x)
    torch.cuda.synchronize()
    return P, x, y


def test_forward_does_not_wait(gpu, streams):
    P, x, y = _case(gpu)
    a, b = streams
    _busy(a)
    with torch.cuda.stream(a):
        ya = P.forward(x)
    with torch.cuda.stream(b):
        yb = [P.forward(x) for _ in range(3)]
    assert not _waits(b.synchronize)
    torch.cuda.synchronize()
    assert torch.equal(ya, y) and all(torch.equal(v, y) for v in yb)


@pytest.mark.parametrize("graph", [False, True])
def test_solve_does_not_wait(gpu, streams, graph):
    from framelab_amd import solvers
    a, b = streams
    for _ in range(6):   # until the solver's own stream runs beside a
        P, x, y = _case(gpu)
        rhs, u0 = P.adjoint(y), torch.zeros_like(x)
        solve = lambda: solvers.cgls(P, rhs, u0, 0.1, 4, graph=graph)[0]  # noqa: E731  (returns when done)
        want = solve()
        torch.cuda.synchronize()
        _busy(a)
        with torch.cuda.stream(b):
            apart = not _waits(solve)
        torch.cuda.synchronize()
        if apart:
            break
    else:
        pytest.skip("the solver's stream never ran beside another")
    _busy(a)
    with torch.cuda.stream(a):
        ya = P.forward(x)
    with torch.cuda.stream(b):
        assert not _waits(solve)
        u = solve()
    torch.cuda.synchronize()
    assert torch.equal(ya, y) and torch.equal(u, want)
    # forwards after the solve, on its caller's stream and beside it
    with torch.cuda.stream(b):
        u = solve()
        yb = P.forward(x)
    with torch.cuda.stream(a):
        ya = P.forward(x)
    torch.cuda.synchronize()
    assert torch.equal(ya, y) and torch.equal(yb, y) and torch.equal(u, want)


def test_forward_while_another_stream_is_captured(gpu, streams):
    """The check for a busy copy is allowed beside a capture in the strictest mode."""
    P, x, y = _case(gpu)
    a, b = streams
    other = torch.zeros(256, device=gpu)
    ya, yb = torch.empty_like(y), torch.empty_like(y)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream(), capture_error_mode="global"):
        other.add_(1)
        with torch.cuda.stream(a):
            P.forward(x, ya)
        with torch.cuda.stream(b):
            P.forward(x, yb)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(ya, y) and torch.equal(yb, y) and other.eq(1).all()
