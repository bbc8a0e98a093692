"""CPU checks, in float32, of two rules the GPU kernels rely on.

Tracked cells: a forward walk may name a segment's cell by the planes passed
instead of the reference's floor of the rounded midpoint wherever the segment
is longer than tau, inside the volume and beyond its exit alike.  Shadow
windows: the few cells the fan adjoints evaluate per pixel and view hold every
cell whose line meets the pixel.  Both are emulated operation by operation, on
geometries with axis-parallel rays, sources close to the volume, unequal voxel
heights, odd panels and sizes around a tile's."""
import math

import numpy as np
import pytest

from framelab_amd import geometry as G

f32 = np.float32


def _tracked_walk(p, iv, ia, ib, batch=5):
    """Walks one ray as the kernel does; asserts on the way.  Returns the
    number of long segments compared."""
    n = [p.nx, p.ny, p.nz]
    c, s = f32(math.cos(float(p.sd_phi[iv]))), f32(math.sin(float(p.sd_phi[iv])))
    yd = p.y_det[ia]
    o = [f32(c * -p.SO), f32(s * -p.SO), p.sd_z[iv]]
    q = [f32(f32(c * p.OD) - f32(s * yd)), f32(f32(s * p.OD) + f32(c * yd)), f32(p.z_det[ib] + p.sd_z[iv])]
    d = [f32(q[k] - o[k]) for k in range(3)]
    sp = [f32(1), f32(1), f32(p.dz)]
    on = [v != 0 for v in d]
    st = [1 if v > 0 else -1 for v in d]
    i0 = [-(n[k] // 2) * st[k] for k in range(3)]

    def alpha(k, j):
        return f32(f32(f32(f32(i0[k] + st[k] * j) * sp[k]) - o[k]) / d[k])

    def cell(m):
        t = []
        for k in range(3):
            x = f32(o[k] + f32(m * d[k]))
            if sp[k] != 1:
                x = f32(x / sp[k])
            t.append(int(math.floor(f32(x + f32(n[k] // 2)))))
        return t

    def inside(t):
        return all(0 <= t[k] < n[k] for k in range(3))

    def far(t):
        return any(on[k] and (t[k] >= n[k] if st[k] > 0 else t[k] < 0) for k in range(3))
    if any(not on[k] and not 0 <= cell(f32(0.5))[k] < n[k] for k in range(3)):
        return 0
    entry = max(alpha(k, 0) for k in range(3) if on[k])
    leave = min(alpha(k, n[k]) for k in range(3) if on[k])
    w = [1.5 * n[k] + 3 if sp[k] == 1 else float(sp[k]) * (2.5 * n[k] + 5) for k in range(3)]
    tau = f32(1.01 * 2.0 ** -23 * (4 * max(float(leave), 0.0) + max(w[k] / abs(float(d[k])) for k in range(3) if on[k])))
    cur = entry
    j = [sum(alpha(k, i) <= cur for i in range(n[k] + 1)) if on[k] else 0 for k in range(3)]
    a = [alpha(k, j[k]) if on[k] and j[k] <= n[k] else f32(np.inf) for k in range(3)]
    track = [(j[k] - 1 if st[k] > 0 else n[k] - j[k]) if on[k] else cell(f32(0.5))[k] for k in range(3)]
    frozen = False
    compared = 0
    for _ in range(4 * sum(n)):
        ends, cells, start = [], [], cur
        for _ in range(batch):
            an = min(a)
            ends.append(an)
            cells.append(list(track))
            assert all(-batch <= track[k] < n[k] + batch for k in range(3))   # guard cells
            for k in range(3):
                if a[k] == an:
                    j[k] += 1
                    a[k] = alpha(k, j[k])
                    track[k] += 0 if frozen else st[k]
            cur = an
        out = cur > leave
        done = out and f32(cur - ends[-2]) > tau
        frozen = frozen or out
        c0 = start
        for e, t in zip(ends, cells):
            rule = cell(f32(f32(c0 + e) * f32(0.5)))
            if f32(e - c0) > tau:
                compared += 1
                assert (t == rule and inside(rule)) if e <= leave else (not inside(rule) and far(rule))
            elif not inside(rule) and far(rule):
                done = True
            c0 = e
        if done:
            return compared
    raise AssertionError("the walk does not end")


@pytest.mark.parametrize("seed", range(8))
def test_tracked_cells_are_the_rules(seed):
    rng = np.random.default_rng(seed)
    N = tuple(2 * int(rng.integers(1, 17)) for _ in range(3))
    L = (2.0, 2.0 * N[1] / N[0], 2.0 * N[2] / N[0] * (1.0 if seed % 2 else float(rng.uniform(0.5, 1.5))))
    r = 0.5 * math.hypot(L[0], L[1])
    SO = r * float(rng.uniform(1.3, 3.0)) + 4.0 / N[0]
    na, nb, nv = int(rng.integers(3, 40)), int(rng.integers(2, 30)), 8   # views at multiples of 45 degrees
    p = G.cone_para(na, nb, nv, N=N, L=L, SO=SO, OD=SO, Ly=G.full_fan_width(SO, 2 * SO, r),
                    Lz=G.full_cone_height(SO, 2 * SO, r, L[2] / 2))
    rays = [(int(rng.integers(nv)), int(rng.integers(na)), int(rng.integers(nb))) for _ in range(60)]
    rays += [(v, na // 2, nb // 2) for v in range(nv)] + [(v, na // 2, b) for v in (0, 2, 3) for b in range(nb)]
    assert sum(_tracked_walk(p, *ray) for ray in rays) > 0


WINDOWS = [(8, 8, 6, 9), (34, 26, 20, 24), (18, 50, 60, 12), (62, 40, 100, 16), (48, 48, 160, 8), (64, 64, 64, 20),
           (130, 122, 251, 6)]


@pytest.mark.parametrize("case", WINDOWS)
def test_fan_windows_hold_every_hit(case):
    """The first cell and the count the windowed adjoints take per pixel (from
    its tile's bounds) against every cell whose line passes the pixel."""
    nx, ny, nd, nv = case
    L = (2.0, 2.0 * ny / nx)
    p = G.fan_para(nd, nv, N=(nx, ny), L=L, SO=4.0, OD=4.0, Ly=G.full_fan_width(4.0, 8.0, 0.5 * math.hypot(*L)))
    SO, SD = float(p.SO), float(p.SO) + float(p.OD)
    pa = (float(p.y_det[-1]) - float(p.y_det[0])) / (nd - 1)
    margin, ex = 0.05, 0.5 * float(np.max(np.abs(p.cos_phi) + np.abs(p.sin_phi)))
    rc = 0.5 * math.hypot(nx - 1, ny - 1)
    dmin = SO - rc - 0.01
    grow, tg = 1 + ex / (dmin - ex), rc / math.sqrt(SO * SO - rc * rc)
    hmax = math.sqrt(0.5 * (1 + tg * tg)) * grow
    S = max(2, int(2 * hmax * SD / dmin / pa + 2 * margin + 1e-3) + 1)
    klo, sdp = -float(p.y_det[0]) / pa - margin, SD / pa
    X, Y = np.meshgrid(np.arange(nx), np.arange(ny))
    xc, yc = X + 0.5 - nx // 2, Y + 0.5 - ny // 2
    xt, yt = X // 8 * 8 + 4 - nx // 2, Y // 8 * 8 + 4 - ny // 2
    e0 = 7 * ex
    tile = int((2 * e0 * (1 + tg + e0 / (dmin - 2 * e0)) + 2 * hmax) * SD / (dmin - 2 * e0) / pa) + 4 + S
    hits = 0
    for v in range(nv):
        c, s = float(p.cos_phi[v]), float(p.sin_phi[v])
        e = 3.5 * (abs(c) + abs(s))
        D, yr = c * xt + s * yt + SO, c * yt - s * xt
        rn, rf, t = 1 / (D - e), 1 / (D + e), yr / D
        h = abs(t * c + s) + abs(c - t * s) + e * (1 + abs(t)) * rn * (abs(c) + abs(s))
        hs = np.minimum(h * 0.5 * grow, hmax)
        n = np.minimum((2 * hs * rn * sdp + 0.101).astype(int) + 1, S)
        edge = yr - e - hs
        a0 = np.clip(np.ceil(edge * np.where(edge > 0, rf, rn) * sdp + klo - 0.01), 0, nd - S)
        lo = np.ceil((c * yc - s * xc - hs) / (c * xc + s * yc + SO) * sdp + klo)
        lo = np.minimum(np.maximum(lo, a0), nd - n)
        assert (lo - a0 + n <= tile).all()
        for a in range(nd):
            sd, cd = float(p.sin_det[a]), float(p.cos_det[a])
            Px, Py = -(sd * c + cd * s), cd * c - sd * s
            hit = np.abs(SO * sd - Px * xc - Py * yc) < (abs(Px) + abs(Py)) / 2
            hits += int(hit.sum())
            assert not (hit & ((a < lo) | (a >= lo + n))).any()
    assert hits > 0
