"""The matched cone adjoint at the edges of its forms: bricks cut by the volume,
footprints of one cell and footprints that overflow the staged tables, panels
that see part of a brick, descending rows, rays parallel to the planes, unequal
voxel heights, helices, frames, and volumes of each launch form.  Its dot test
with the forward (2e-6 of the scale of the terms, the bound of the other dot
tests), and 16-bit storage as one rounding of the FP32 result."""
import dataclasses

import numpy as np
import pytest
import torch

from helpers import dot_gap

pytestmark = pytest.mark.gpu

# (nx, ny, nz, cells, rows, views, height ratio, source distance over the radius)
CASES = [
    (2, 2, 2, 3, 3, 8, 1.0, 4.0), (8, 8, 16, 16, 16, 9, 1.0, 4.0), (10, 6, 18, 16, 40, 8, 1.0, 4.0),
    (16, 16, 32, 17, 19, 3, 1.0, 1.3), (16, 16, 16, 120, 100, 5, 1.0, 4.0), (20, 12, 34, 25, 90, 65, 0.4, 2.0),
    (34, 26, 10, 9, 7, 6, 1.7, 3.0), (24, 24, 24, 49, 65, 4, 1.0, 4.0),
    (96, 90, 66, 120, 90, 5, 1.0, 4.0), (96, 96, 70, 110, 260, 3, 1.0, 4.0), (130, 122, 98, 140, 120, 3, 1.0, 4.0),
    (128, 128, 96, 300, 80, 2, 0.8, 2.5),
]


def _para(case, **kw):
    from framelab_amd import geometry as G
    nx, ny, nz, na, nb, nv, h, SO = case
    L = (2.0, 2.0 * ny / nx, 2.0 * nz / nx * h)
    r = 0.5 * float(np.hypot(L[0], L[1]))
    SO = SO * r + 4.0 / nx
    args = dict(N=(nx, ny, nz), L=L, SO=SO, OD=SO, Ly=G.full_fan_width(SO, 2 * SO, r),
                Lz=G.full_cone_height(SO, 2 * SO, r, L[2] / 2))
    args.update(kw)
    return G.cone_para(na, nb, nv, **args)


def _check(gpu, p, dtype=None):
    from framelab_amd.projector import ADJ_MATCHED, Projector
    P = Projector(p)
    rng = np.random.default_rng(p.nx + p.nv)
    X = torch.from_numpy(rng.random(int(np.prod(P.vol_shape))).astype(np.float32)).reshape(P.vol_shape).to(gpu)
    Y = torch.from_numpy(rng.standard_normal(int(np.prod(P.sino_shape))).astype(np.float32)).reshape(P.sino_shape).to(gpu)
    x = P.adjoint(Y, kind=ADJ_MATCHED)
    assert dot_gap(P.forward(X).cpu().numpy(), Y.cpu().numpy(), X.cpu().numpy(), x.cpu().numpy()) <= 2e-6
    for dt in (torch.bfloat16, torch.float16):
        Yh = Y.to(dt)
        got, want = P.adjoint(Yh, kind=ADJ_MATCHED).double(), P.adjoint(Yh.float(), kind=ADJ_MATCHED).double()
        # one rounding of the scaled sum, of which FP32's is another
        ulp = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
        assert (got - want).abs().le((ulp + 2.0 ** -23) * want.abs() + 2.0 ** -25).all()
    return P, Y, x


@pytest.mark.parametrize("case", CASES)
def test_sizes(gpu, case):
    _check(gpu, _para(case))


@pytest.mark.parametrize("kind", ["narrow", "low", "rows down", "frames", "helix", "none"])
def test_geometries(gpu, kind):
    from framelab_amd import geometry as G
    case = (26, 22, 36, 33, 41, 20, 1.0, 3.0)
    if kind == "narrow":
        p = _para(case, Ly=1.0)
    elif kind == "low":
        p = _para(case, Lz=0.3)
    elif kind == "rows down":
        p = _para(case)
        p = dataclasses.replace(p, z_det=p.z_det[::-1].copy())
    elif kind == "frames":
        p = G.with_frames(_para(case), [0] * 3 + [2] * 17)
    elif kind == "helix":
        p = G.cone_para(25, 18, 0, N=(26, 26, 38), L=(2.0, 2.0, 4.0), kind="helix", zmax=2.0, rps=3.0, vtab=2.0, fps=40.0)
    else:   # no view sees the volume
        p = _para(case)
        p = dataclasses.replace(p, sd_z=np.full_like(p.sd_z, 1000.0))
        P, Y, x = _check(gpu, p)
        assert not x.any()
        return
    _check(gpu, p)


def test_values_stay_with_their_rays(gpu):
    """An infinite sinogram value reaches the voxels of its ray and the
    neighbours its shadow windows hold, and no others."""
    from framelab_amd.projector import ADJ_MATCHED, Projector
    p = _para((24, 24, 24, 30, 30, 4, 1.0, 4.0))
    P = Projector(p)
    Y = torch.zeros(P.sino_shape, device=gpu)
    Y.view(4, 30, 30)[1, 15, 15] = float("inf")
    x = P.adjoint(Y, kind=ADJ_MATCHED)
    bad = ~torch.isfinite(x)
    assert bad.any() and bad.sum() <= 24 * 27


# tables of each launch form; a power of two scales every operation exactly
@pytest.mark.parametrize("case", [CASES[1], CASES[5], CASES[8], CASES[10]])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_large_values(gpu, case, dtype):
    """Values up to 2^123 (1e37): nothing overflows that the sums do not."""
    from framelab_amd.projector import ADJ_MATCHED, Projector
    p = _para(case)
    P = Projector(p)
    Y = torch.from_numpy(np.random.default_rng(5).uniform(-1, 1, P.sino_shape).astype(np.float32)).to(gpu).to(dtype)
    k = 119 if p.nv > 8 else 123   # voxel sums of so many views of up to 2 |y| stay finite
    x = P.adjoint(Y, kind=ADJ_MATCHED, dtype=torch.float32)
    assert torch.equal(P.adjoint(Y * 2.0 ** k, kind=ADJ_MATCHED, dtype=torch.float32), x * 2.0 ** k)


def test_columns_down(gpu):
    p = _para((26, 22, 36, 33, 41, 20, 1.0, 3.0))
    _check(gpu, dataclasses.replace(p, y_det=p.y_det[::-1].copy()))
