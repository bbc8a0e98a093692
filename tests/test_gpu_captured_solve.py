"""A CGLS or split-Bregman solve that the caller captures: the graph may be
replayed beside the plan's other forwards, so it must not use the bricked image
copy they share (plans of 150 000 rays and more); its replays return the eager
solve's bits, also beside eager forwards of the plan on another stream."""
import ctypes as C

import numpy as np
import pytest
import torch

from graph_kernels import captured_kernels

pytestmark = pytest.mark.gpu


def _plan(gpu):
    from framelab_amd import geometry as G
    from framelab_amd.projector import Projector
    P = Projector(G.fan_para(600, 260, N=(66, 62), SO=4.0, OD=4.0, Ly=G.full_fan_width()))
    x = torch.from_numpy(np.random.default_rng(3).standard_normal(P.vol_shape).astype(np.float32)).to(gpu)
    return P, x, P.forward(x)


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _cgls(P, b, u, flags=0):
    from framelab_amd import _lib
    return lambda st: _lib.check(_lib.lib().fl_cgls(P.handle, _ptr(b), _ptr(u), 0.1, 3, 0.0, flags, None, None, st))


def _bregman(P, f, u, flags=0):
    from framelab_amd import _lib
    return lambda st: _lib.check(_lib.lib().fl_split_bregman(P.handle, _lib.FL_FRAME_LINEAR, 1, _ptr(f), _ptr(u), 0.01, 1.0,
                                                             2, 2, 0.0, flags, None, None, st))


@pytest.mark.parametrize("storage", [0, 4, 8])
@pytest.mark.parametrize("solve", [_cgls, _bregman])
def test_foreign_capture_leaves_the_shared_copy_alone(gpu, solve, storage):
    P, x, y = _plan(gpu)
    call = solve(P, P.adjoint(y) if solve is _cgls else y, torch.zeros_like(x), storage)
    call(C.c_void_p(torch.cuda.current_stream().cuda_stream))   # the solver's workspace
    names = captured_kernels(call)
    assert sum("k_fwd_fan" in n for n in names) >= 4
    assert not any("k_to_fan_bricks" in n for n in names)


def test_replays_beside_eager_forwards(gpu):
    P, x, y = _plan(gpu)
    other = torch.flip(x, (0,)).contiguous()
    y_other, b, u = P.forward(other), P.adjoint(y), torch.zeros_like(x)
    call = _cgls(P, b, u)
    call(C.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    want = u.clone()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph):
        call(C.c_void_p(torch.cuda.current_stream().cuda_stream))
    for _ in range(4):
        u.zero_()
        torch.cuda.synchronize()
        graph.replay()
        with torch.cuda.stream(side):
            eager = [P.forward(other) for _ in range(4)]
        torch.cuda.synchronize()
        assert torch.equal(u, want) and all(torch.equal(e, y_other) for e in eager)
