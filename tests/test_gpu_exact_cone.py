"""The exact cone adjoint bit for bit against the oracle where its forms and
short cuts part: shadows of two, three and more columns, footprints that
overflow the staged tables, wide cones whose rays cross both z faces of a
voxel, flat voxels, views along the axes and diagonals (rays along voxel edges
and through corners), sources close to the volume, panels in descending order
or that see part of a brick, frames, helices and each launch form."""
import dataclasses

import numpy as np
import pytest
import torch

from helpers import bits_equal, first_mismatch

pytestmark = pytest.mark.gpu

# (nx, ny, nz, cells, rows, views, height ratio, source distance over the radius)
CASES = [
    (2, 2, 2, 3, 3, 8, 1.0, 4.0), (8, 8, 8, 9, 9, 8, 1.0, 4.0), (10, 6, 18, 16, 40, 8, 1.0, 4.0),
    (16, 16, 16, 17, 19, 16, 1.0, 1.3), (16, 16, 48, 33, 64, 8, 1.0, 1.2), (16, 16, 16, 40, 24, 8, 1.0, 4.0),
    (16, 16, 16, 120, 100, 5, 1.0, 4.0), (20, 12, 34, 25, 90, 65, 0.3, 2.0), (34, 26, 10, 9, 7, 8, 1.7, 3.0),
    (24, 24, 24, 49, 65, 16, 1.0, 4.0), (24, 24, 24, 48, 48, 8, 0.1, 3.0), (96, 90, 66, 120, 90, 5, 1.0, 4.0),
    (250, 250, 98, 300, 80, 2, 1.0, 4.0),
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


def _check(gpu, oracle, p):
    from framelab_amd.projector import ADJ_EXACT, Projector
    P = Projector(p)
    Y = np.random.default_rng(p.nx + p.nv).standard_normal(int(np.prod(P.sino_shape))).astype(np.float32)
    x = P.adjoint(torch.from_numpy(Y).reshape(P.sino_shape).to(gpu), kind=ADJ_EXACT).cpu().numpy().ravel()
    xo = oracle.atx_cone_f32(Y, p)
    assert bits_equal(x, xo), first_mismatch(x, xo)


@pytest.mark.parametrize("case", CASES)
def test_sizes(gpu, oracle, case):
    _check(gpu, oracle, _para(case))


@pytest.mark.parametrize("kind", ["narrow", "low", "rows down", "columns down", "shifted", "frames", "helix", "near axes"])
def test_geometries(gpu, oracle, kind):
    from framelab_amd import geometry as G
    case = (26, 22, 36, 33, 41, 16, 1.0, 3.0)
    if kind == "narrow":
        p = _para(case, Ly=1.0)
    elif kind == "low":
        p = _para(case, Lz=0.3)
    elif kind == "rows down":
        p = _para(case)
        p = dataclasses.replace(p, z_det=p.z_det[::-1].copy())
    elif kind == "columns down":
        p = _para(case)
        p = dataclasses.replace(p, y_det=p.y_det[::-1].copy())
    elif kind == "shifted":
        p = _para(case, y_os=0.4)
    elif kind == "frames":
        p = G.with_frames(_para(case), [0] * 3 + [2] * 13)
    elif kind == "helix":
        p = G.cone_para(25, 18, 0, N=(26, 26, 38), L=(2.0, 2.0, 4.0), kind="helix", zmax=2.0, rps=3.0, vtab=2.0, fps=40.0)
    else:   # views a little off the axes and diagonals
        phi = (np.arange(16) // 2 * (np.pi / 4) + np.where(np.arange(16) % 2, 3e-5, -2e-7)).astype(np.float32)
        p = _para(case, sd_phi=phi)
    _check(gpu, oracle, p)


@pytest.mark.parametrize("cells", [(33, 29), (60, 44), (90, 70)])
def test_infinite_values_count_once(gpu, cells):
    """Infinite values far enough apart that a voxel's shadow holds one of them:
    its sum is infinite where that cell's chord is positive, never NaN."""
    from framelab_amd.projector import ADJ_EXACT, Projector
    P = Projector(_para((24, 24, 24, *cells, 3, 1.0, 4.0)))
    for a in range(0, 10, 3):
        ones = torch.zeros(P.sino_shape, device=gpu)
        ones[1, a::10, a::10] = 1.0
        chord = P.adjoint(ones, kind=ADJ_EXACT)
        x = P.adjoint(torch.where(ones > 0, torch.inf, 0.0), kind=ADJ_EXACT)
        assert (chord > 0).any() and torch.isposinf(x[chord > 0]).all()


@pytest.mark.parametrize("case", [(24, 24, 24, 8, 7, 9, 1.0, 4.0), (40, 36, 70, 14, 60, 5, 1.0, 3.0), (34, 30, 20, 22, 5, 8, 0.5, 2.0)])
def test_cells_wider_than_shadows(gpu, oracle, case):
    _check(gpu, oracle, _para(case))


@pytest.mark.parametrize("cells, columns", [((8, 7), 1), ((49, 65), 2)])
def test_columns_by_panel(gpu, cells, columns):
    """Panels of less than a cell a voxel take the form for one column or two."""
    from framelab_amd import _lib
    from framelab_amd.projector import ADJ_EXACT, Projector
    from graph_kernels import captured_kernels
    P = Projector(_para((24, 24, 24, *cells, 3, 1.0, 4.0)))
    y, x = torch.zeros(P.sino_shape, device=gpu), torch.zeros(P.vol_shape, device=gpu)
    names = captured_kernels(lambda st: _lib.check(_lib.lib().fl_adjoint(P.handle, y.data_ptr(), _lib.FL_F32, x.data_ptr(),
                                                                         _lib.FL_F32, ADJ_EXACT, st)))
    assert len(names) == 1 and f"k_adj_cone_zcIffLi2ELi{columns}E" in names[0]
