"""The Gao fan forward, whose columns are shared by four lanes, bit for bit
against a serial walk in float32: images wider and taller than square, one
column short of and beyond a batch, views along the axes and the diagonals,
cell and view counts around a wave's, frames, and the batched form."""
import numpy as np
import pytest
import torch

from helpers import bits_equal, first_mismatch

pytestmark = pytest.mark.gpu
f32 = np.float32

# (nx, ny, cells, views, source distance)
CASES = [(2, 2, 1, 1, 4.0), (2, 6, 5, 8, 4.0), (14, 16, 9, 8, 4.0), (16, 14, 4, 4, 4.0), (18, 18, 33, 24, 4.0),
         (34, 10, 21, 9, 3.0), (10, 34, 21, 9, 3.0), (62, 66, 40, 16, 1.5), (64, 64, 96, 60, 4.0)]


def _para(case):
    from framelab_amd import geometry as G
    nx, ny, nd, nv, SO = case
    L = (2.0, 2.0 * ny / nx)
    r = 0.5 * float(np.hypot(*L))
    SO = SO * r
    return G.fan_para(nd, nv, N=(nx, ny), L=L, SO=SO, OD=SO, Ly=G.full_fan_width(SO, 2 * SO, r))


def _serial(X, p):
    """The column walk (Ax_fan_mf_cpu_new.cpp:28-119), all rays at once, one
    float32 operation at a time."""
    nx, ny = p.nx, p.ny
    X = X.reshape(-1, ny, nx)
    c, s = np.cos(p.sd_phi.astype(np.float64)).astype(f32)[:, None], np.sin(p.sd_phi.astype(np.float64)).astype(f32)[:, None]
    yd, SO, OD = p.y_det.astype(f32)[None, :], f32(p.SO), f32(p.OD)
    x1, y1 = np.broadcast_to(c * -SO, (p.nv, p.nd)), np.broadcast_to(s * -SO, (p.nv, p.nd))
    x2, y2 = c * OD - s * yd, s * OD + c * yd
    img = X[np.broadcast_to(np.asarray(p.id_X)[:, None] if len(X) > 1 else np.zeros((p.nv, 1), int), (p.nv, p.nd))]
    xm = np.abs(x1 - x2) > np.abs(y1 - y2)
    y = np.zeros((p.nv, p.nd), f32)
    for major in (True, False):
        nu, nw = (nx, ny) if major else (ny, nx)
        u0, v0 = (x1, y1) if major else (y1, x1)
        with np.errstate(all="ignore"):
            k = (y2 - y1) / (x2 - x1) if major else (x2 - x1) / (y2 - y1)
            acc = np.zeros_like(y)
            for i in range(nu):
                u = f32(i - nu // 2)
                a, b = (v0 + k * (u - u0)) + f32(nw // 2), (v0 + k * ((u + f32(1)) - u0)) + f32(nw // 2)
                v1, v2 = np.where(k >= 0, a, b), np.where(k >= 0, b, a)
                c1, c2 = np.floor(v1), np.floor(v2)
                d = v2 - v1
                l = np.sqrt(d * d + f32(1))
                def at(cell):
                    j = np.clip(np.nan_to_num(cell), 0, nw - 1).astype(int)
                    return np.take_along_axis(img[:, :, :, i] if major else img[:, :, i, :], j[..., None], 2)[..., 0]
                one, mid = c1 == c2, (c1 != c2) & (c2 > 0) & (c2 < nw)
                rest = (c1 != c2) & ~mid
                t1, t2 = ((c2 - v1) / d) * l * at(c1), ((v2 - c2) / d) * l * at(c2)
                acc = np.where(one & (c1 >= 0) & (c1 <= nw - 1), acc + l * at(c1), acc)
                acc = np.where((mid & (c1 >= 0)) | (rest & (c2 == ny) & (c1 >= 0) & (c1 < nw)), acc + t1, acc)
                acc = np.where(mid | (rest & (c2 == 0)), acc + t2, acc)
        y = np.where(xm == major, acc, y)
    return (y * f32(p.scale)).ravel()


def _image(p, seed):
    return np.random.default_rng(seed).standard_normal(p.nx * p.ny * p.nt).astype(np.float32)


@pytest.mark.parametrize("case", CASES + ["frames"])
def test_serial_sum(gpu, case):
    from framelab_amd import geometry as G
    from framelab_amd.projector import Projector
    p = G.with_frames(_para((18, 22, 13, 11, 3.0)), [0] * 5 + [2] * 6) if case == "frames" else _para(case)
    P = Projector(p)
    X = _image(p, p.nx + p.nd)
    x = torch.from_numpy(X).reshape(P.vol_shape).to(gpu)
    y, ys = P.forward(x, method="gao").cpu().numpy().ravel(), _serial(X, p)
    assert bits_equal(y, ys), first_mismatch(y, ys)
    xh = x.to(torch.bfloat16)
    assert torch.equal(P.forward(xh, method="gao").float(), P.forward(xh.float(), method="gao").to(torch.bfloat16).float())


def test_batch(gpu):
    from framelab_amd.batch import ProjectorBatch
    ps = [_para(c) for c in CASES]
    X = [_image(p, 3) for p in ps]
    y = ProjectorBatch(ps).forward(torch.from_numpy(np.concatenate(X)).to(gpu), method="gao").cpu().numpy()
    ys = np.concatenate([_serial(x, p) for x, p in zip(X, ps)])
    assert bits_equal(y, ys), first_mismatch(y, ys)
