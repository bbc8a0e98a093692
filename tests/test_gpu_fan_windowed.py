"""The fan adjoints' windowed form at its edges: tiles cut by the image, view
counts around a batch of views and around the 64 views a wave prepares at a
time, every cell count it is built for, panels barely wider than that, and the
plans that must fall back to the general form.  Exact adjoint bit for bit
against the oracle; matched adjoint by its dot test with the forward (2e-6 of
the scale of the terms, the bound of the other dot tests), in single plans and
in a batch."""
import dataclasses

import numpy as np
import pytest
import torch

from helpers import bits_equal, dot_gap, first_mismatch

pytestmark = pytest.mark.gpu

# (nx, ny, bins, views): pitches from one to seven cells per pixel's shadow
CASES = [
    (8, 8, 6, 1), (10, 14, 24, 6), (34, 26, 20, 7), (34, 26, 33, 8), (18, 50, 60, 13), (64, 64, 64, 14),
    (62, 40, 100, 15), (40, 72, 140, 28), (48, 48, 160, 29), (30, 30, 200, 9), (16, 24, 30, 447), (16, 24, 30, 448),
    (16, 24, 44, 455), (24, 16, 70, 900), (56, 56, 57, 33), (130, 122, 251, 10),
]


def _para(case, **kw):
    from framelab_amd import geometry as G
    nx, ny, nd, nv = case
    L = (2.0, 2.0 * ny / nx)
    args = dict(N=(nx, ny), L=L, SO=4.0, OD=4.0, Ly=G.full_fan_width(4.0, 8.0, 0.5 * float(np.hypot(*L))))
    args.update(kw)
    return G.fan_para(nd, nv, **args)


def _check(gpu, oracle, p, matched=True):
    from framelab_amd.projector import ADJ_EXACT, ADJ_MATCHED, Projector
    rng = np.random.default_rng(p.nx + p.nd)
    Y = rng.standard_normal(p.nv * p.nd).astype(np.float32)
    X = rng.random(p.nx * p.ny * p.nt).astype(np.float32)
    P = Projector(p)
    Yt = torch.from_numpy(Y).reshape(P.sino_shape).to(gpu)
    x = P.adjoint(Yt, kind=ADJ_EXACT).cpu().numpy().ravel()
    xo = oracle.atx_fan_f32(Y, p)
    assert bits_equal(x, xo), first_mismatch(x, xo)
    if not matched:
        return None
    y = P.forward(torch.from_numpy(X.reshape(P.vol_shape)).to(gpu)).cpu().numpy().ravel()
    xm = P.adjoint(Yt, kind=ADJ_MATCHED).cpu().numpy().ravel()
    assert dot_gap(y, Y, X, xm) <= 2e-6
    return Yt, x, xm


@pytest.mark.parametrize("case", CASES)
def test_sizes(gpu, oracle, case):
    _check(gpu, oracle, _para(case))


@pytest.mark.parametrize("kw", [dict(SO=1.45), dict(y_os=0.3), dict(y_os=-0.9), dict(Ly=-1.0), dict(Ly=2.0), "angles",
                                "nonuniform angles", "frames"])
def test_geometries(gpu, oracle, kw):
    """Sources close to the image, shifted, short and (exact only) reversed panels, angle
    tables off the detector coordinates, several frames (one without views)."""
    from framelab_amd import geometry as G
    case = (34, 26, 40, 21)
    if kw == "frames":
        p = G.with_frames(_para(case), [0] * 9 + [2] * 12)
    elif isinstance(kw, str):
        p = _para(case)
        a = np.arctan2(p.sin_det, p.cos_det).astype(np.float64)
        a = a + 0.004 if kw == "angles" else a * (1 + 0.05 * a)
        p = dataclasses.replace(p, cos_det=np.cos(a).astype(np.float32), sin_det=np.sin(a).astype(np.float32))
    elif kw.get("Ly") == -1.0:   # columns in descending order
        p = _para(case)
        p = dataclasses.replace(p, y_det=p.y_det[::-1].copy(), cos_det=p.cos_det[::-1].copy(),
                                sin_det=p.sin_det[::-1].copy())
    else:
        p = _para(case, **kw)
    _check(gpu, oracle, p, matched=kw != dict(Ly=-1.0))


def test_batch_mixes_forms(gpu, oracle):
    """A batch of windowed and general problems equals the single plans."""
    from framelab_amd.batch import ProjectorBatch
    from framelab_amd.projector import ADJ_EXACT, ADJ_MATCHED
    paras = [_para(c) for c in CASES[:12]] + [_para((34, 26, 40, 21), SO=1.45), _para((34, 26, 300, 5))]
    ref = [_check(gpu, oracle, p) for p in paras]
    B = ProjectorBatch(paras)
    y = B.pack([r[0] for r in ref], sino=True)
    for kind, k in ((ADJ_EXACT, 1), (ADJ_MATCHED, 2)):
        for got, r in zip(B.unpack(B.adjoint(y, kind=kind).cpu()), ref):
            assert bits_equal(got.numpy().ravel(), r[k])


def _names(call):
    from framelab_amd import _lib
    from graph_kernels import captured_kernels
    return captured_kernels(lambda st: _lib.check(call(_lib.lib(), st)))


# (pixels a side, bins, views, exact windowed, matched windowed)
@pytest.mark.parametrize("n, nd, nv, exact, matched", [(512, 512, 2, False, False), (512, 512, 15, False, True),
                                                       (512, 512, 25, True, True), (512, 1024, 5, False, False),
                                                       (512, 1024, 9, False, True), (512, 1024, 10, True, True),
                                                       (512, 512, 30, False, True), (360, 360, 2, True, True),
                                                       (384, 960, 3, False, False), (384, 960, 5, True, True)])
def test_few_views(gpu, oracle, n, nd, nv, exact, matched):
    """Images whose tiles fill the chip take the general form for few views, alone
    and in a batch (one problem here: the same count of tiles)."""
    from framelab_amd.batch import ProjectorBatch
    from framelab_amd.projector import ADJ_EXACT, ADJ_MATCHED, Projector
    p = _para((n, n, nd, nv))
    P, B = Projector(p), ProjectorBatch([p])
    y = torch.from_numpy(np.random.default_rng(n).standard_normal((nv, nd)).astype(np.float32)).to(gpu)
    x = torch.empty(P.vol_shape, device=gpu)
    for kind, windowed in ((ADJ_EXACT, exact), (ADJ_MATCHED, matched)):
        one = _names(lambda L, st: L.fl_adjoint(P.handle, y.data_ptr(), 0, x.data_ptr(), 0, kind, st))
        many = _names(lambda L, st: L.fl_batch_adjoint(B.handle, y.data_ptr(), x.data_ptr(), kind, st))
        assert ["k_adj_fan_w" in k for k in one] == ["k_badj_w" in k for k in many] == [windowed]
        got = P.adjoint(y, kind=kind)
        assert torch.equal(B.adjoint(y.ravel(), kind=kind), got.ravel())
    want = oracle.atx_fan_f32(y.cpu().numpy().ravel(), p)
    got = P.adjoint(y).cpu().numpy().ravel()
    assert bits_equal(got, want), first_mismatch(got, want)
