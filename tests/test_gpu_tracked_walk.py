"""The forward projectors' tracked walk at the edges of its layouts and tiles:
volume sides on both sides of a brick and of a power of two, thin volumes,
unequal voxel heights, helices, axis-parallel views, panels and view counts
around a wave's patch, several frames.  Bit for bit against the oracle in
FP32; 16-bit storage against FP32 on the same rounded input, in the bound of
one rounding of the result."""
import numpy as np
import pytest
import torch

from helpers import bits_equal, first_mismatch

pytestmark = pytest.mark.gpu

# (nx, ny, nz, cells, rows, views, height ratio, source distance)
CONES = [
    (2, 2, 2, 9, 7, 8, 1.0, 4.0), (4, 4, 4, 16, 16, 8, 1.0, 4.0), (6, 10, 2, 17, 15, 8, 1.0, 4.0),
    (16, 16, 16, 31, 33, 16, 1.0, 1.5), (18, 14, 34, 23, 40, 9, 1.0, 4.0), (66, 30, 4, 40, 9, 8, 0.7, 4.0),
    (8, 62, 20, 33, 20, 8, 1.4, 6.0), (32, 32, 60, 5, 70, 8, 0.5, 2.0),
]
# (nx, ny, cells, views, source distance)
FANS = [(2, 2, 1, 1, 4.0), (4, 6, 9, 8, 4.0), (16, 16, 8, 8, 1.5), (34, 18, 31, 9, 4.0), (18, 62, 33, 16, 4.0),
        (64, 64, 65, 63, 1.45), (130, 66, 200, 7, 4.0)]


def _cone(case, **kw):
    from framelab_amd import geometry as G
    nx, ny, nz, na, nb, nv, h, SO = case
    L = (2.0, 2.0 * ny / nx, 2.0 * nz / nx * h)
    r = 0.5 * float(np.hypot(L[0], L[1]))
    SO = SO * r
    return G.cone_para(na, nb, nv, N=(nx, ny, nz), L=L, SO=SO, OD=SO, Ly=G.full_fan_width(SO, 2 * SO, r),
                       Lz=G.full_cone_height(SO, 2 * SO, r, L[2] / 2), **kw)


def _fan(case, **kw):
    from framelab_amd import geometry as G
    nx, ny, nd, nv, SO = case
    L = (2.0, 2.0 * ny / nx)
    r = 0.5 * float(np.hypot(*L))
    SO = SO * r
    return G.fan_para(nd, nv, N=(nx, ny), L=L, SO=SO, OD=SO, Ly=G.full_fan_width(SO, 2 * SO, r), **kw)


def _check(gpu, p, ref, dtypes=()):
    from framelab_amd.projector import Projector
    P = Projector(p)
    X = np.random.default_rng(p.nx + p.nv).standard_normal(int(np.prod(P.vol_shape))).astype(np.float32)
    Xt = torch.from_numpy(X).reshape(P.vol_shape).to(gpu)
    y = P.forward(Xt).cpu().numpy().ravel()
    yo = ref(X, p)
    assert bits_equal(y, yo), first_mismatch(y, yo)
    for dt in dtypes:
        Xh = Xt.to(dt)
        want, got = P.forward(Xh.float()).to(dt), P.forward(Xh)
        assert got.dtype in (dt, torch.float32)
        assert torch.equal(got.to(dt), want)


@pytest.mark.parametrize("case", CONES)
def test_cone(gpu, oracle, case):
    _check(gpu, _cone(case), oracle.siddon_cone_f32, (torch.bfloat16, torch.float16))


def test_cone_frames_and_helix(gpu, oracle):
    from framelab_amd import geometry as G
    p = G.with_frames(_cone((10, 12, 18, 19, 21, 9, 1.0, 4.0)), [0] * 4 + [2] * 5)
    _check(gpu, p, oracle.siddon_cone_f32)
    h = G.cone_para(21, 18, 0, N=(18, 18, 30), L=(2.0, 2.0, 4.0), kind="helix", zmax=2.0, rps=3.0, vtab=2.0, fps=20.0)
    _check(gpu, h, oracle.siddon_cone_f32)


@pytest.mark.parametrize("case", FANS)
def test_fan(gpu, oracle, case):
    _check(gpu, _fan(case), oracle.siddon_fan_f32, (torch.bfloat16, torch.float16))


def test_fan_batch(gpu, oracle):
    from framelab_amd.batch import ProjectorBatch
    ps = [_fan(c) for c in FANS]
    rng = np.random.default_rng(5)
    X = [rng.standard_normal(p.nx * p.ny * p.nt).astype(np.float32) for p in ps]
    y = ProjectorBatch(ps).forward(torch.from_numpy(np.concatenate(X)).to(gpu)).cpu().numpy()
    yo = np.concatenate([oracle.siddon_fan_f32(x, p) for x, p in zip(X, ps)])
    assert bits_equal(y, yo), first_mismatch(y, yo)
