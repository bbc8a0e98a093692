"""The fan forward of plans with many rays, which gathers from a bricked copy of
the image: sides on both sides of a brick and of a power of two, frames and
16-bit storage, bit for bit against the oracle; on two streams at once; and
captured by the caller, where replays and eager forwards may interleave."""
import numpy as np
import pytest
import torch

from helpers import bits_equal, first_mismatch

pytestmark = pytest.mark.gpu

SIZES = [(2, 2), (4, 6), (66, 62), (64, 64), (130, 34), (30, 130)]


def _para(nx, ny, nd=600, nv=250):
    from framelab_amd import geometry as G
    L = (2.0, 2.0 * ny / nx)
    r = 0.5 * float(np.hypot(*L))
    return G.fan_para(nd, nv, N=(nx, ny), L=L, SO=3 * r, OD=3 * r, Ly=G.full_fan_width(3 * r, 6 * r, r))


def _case(gpu, p, seed=0):
    from framelab_amd.projector import Projector
    P = Projector(p)
    X = np.random.default_rng(p.nx + seed).standard_normal(int(np.prod(P.vol_shape))).astype(np.float32)
    return P, X, torch.from_numpy(X).reshape(P.vol_shape).to(gpu)


@pytest.mark.parametrize("size", SIZES + ["frames"])
def test_bit_exact(gpu, oracle, size):
    from framelab_amd import geometry as G
    p = G.with_frames(_para(22, 18), [0] * 100 + [2] * 150) if size == "frames" else _para(*size)
    P, X, x = _case(gpu, p)
    y, yo = P.forward(x).cpu().numpy().ravel(), oracle.siddon_fan_f32(X, p)
    assert bits_equal(y, yo), first_mismatch(y, yo)
    xh = x.to(torch.bfloat16)
    assert torch.equal(P.forward(xh).float(), P.forward(xh.float()).to(torch.bfloat16).float())


def test_streams_and_capture(gpu):
    P, _, x = _case(gpu, _para(130, 122))
    a, b = x, torch.flip(x, (0,)).contiguous()
    ya, yb = P.forward(a), P.forward(b)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    out = []
    for k in range(6):
        with torch.cuda.stream(streams[k % 2]):
            out.append(P.forward(b if k % 2 else a))
    torch.cuda.synchronize()
    assert all(torch.equal(o, yb if k % 2 else ya) for k, o in enumerate(out))
    static = a.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        yg = P.forward(static)
    for k in range(4):
        static.copy_(b if k % 2 else a)
        graph.replay()
        with torch.cuda.stream(streams[0]):   # beside the replay
            eager = P.forward(a if k % 2 else b)
        torch.cuda.synchronize()
        assert torch.equal(yg, yb if k % 2 else ya) and torch.equal(eager, ya if k % 2 else yb)
