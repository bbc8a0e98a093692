"""The 3D analysis of four neighbours a thread at its edges (one to few voxels a
side, rows around a workgroup's), the marching 2D synthesis at its edges (images narrower than a tile's halo,
widths and heights around a tile's and a run's, every tile form up to the
gather, dilations larger than the image) and the soft threshold at block
edges, odd band sizes and each storage type."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rel(a, b):
    a, b = np.asarray(a, np.float64).ravel(), np.asarray(b, np.float64).ravel()
    return np.linalg.norm(a - b) / np.linalg.norm(b)


# (nx, ny, frame, levels): one-wave tiles to level 3 (cubic) or 4, then tiles
# of four waves, then the gather
CASES = [(2, 2, "linear", 2), (3, 5, "cubic", 3), (60, 17, "cubic", 1), (61, 16, "cubic", 1), (124, 33, "linear", 2),
         (63, 40, "haar", 4), (50, 70, "cubic", 4), (130, 35, "cubic", 6), (250, 21, "linear", 7), (300, 290, "linear", 2)]


@pytest.mark.parametrize("case", CASES)
def test_synthesis(gpu, oracle, case):
    from framelab_amd.framelets import FrameletSystem
    nx, ny, kind, level = case
    u = np.random.default_rng(nx + ny).standard_normal((ny, nx)).astype(np.float32)
    W = FrameletSystem(2, kind, level)
    c = W.forwardTransform(torch.from_numpy(u).to(gpu)).frameletArray
    # coefficients of no image, so that every band counts
    c = c + torch.from_numpy(np.random.default_rng(1).standard_normal(c.shape).astype(np.float32)).to(gpu)
    _, R = oracle.framelet_filters(kind)
    nf, h = len(R), c.cpu().numpy().astype(np.float64)
    ref = [h[L].reshape(nf, nf, ny, nx).swapaxes(0, 1) for L in range(level)]   # band i + nf*j -> [i, j]
    want = oracle.frarec2d(ref, R)
    assert _rel(W.adjointTransform(c).cpu().numpy(), want) < 2e-6


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 9, 1, 1), (2, 4, 5, 7), (1, 9, 32, 64), (3, 25, 33, 63), (1, 27, 9, 911)])
def test_soft_threshold(gpu, shape, dtype):
    from framelab_amd.framelets import FrameletExpansion, FrameletSystem
    kind = {4: "haar", 9: "linear", 25: "cubic", 27: "linear"}[shape[1]]
    a = torch.randn(shape, generator=torch.Generator().manual_seed(4)).to(gpu).to(dtype)
    want = torch.sign(a.float()) * torch.clamp(a.float().abs() - 0.25, min=0.0)
    want = want.to(dtype)
    want[:, 0] = a[:, 0]
    dim = 3 if shape[1] == 27 else 2
    got = FrameletExpansion(dim, FrameletSystem(dim, kind, shape[0]), a).softThreshold(0.25).frameletArray
    assert torch.equal(got, want)


@pytest.mark.parametrize("kind", ["haar", "linear"])
@pytest.mark.parametrize("shape", [(1, 1, 4), (2, 2, 4), (3, 5, 8), (4, 4, 256), (2, 3, 260), (2, 9, 12), (3, 4, 10)])
def test_analysis3(gpu, oracle, shape, kind):
    from framelab_amd.framelets import FrameletSystem
    u = np.random.default_rng(shape[2]).standard_normal(shape).astype(np.float32)
    W = FrameletSystem(3, kind, 1)
    x = torch.from_numpy(u).to(gpu)
    c = W.forwardTransform(x).frameletArray
    D, _ = oracle.framelet_filters(kind)
    nf = len(D)
    ref = oracle.fradec3d(u.astype(np.float64), D, 1)[0]
    want = np.stack([ref[i, j, k] for k in range(nf) for j in range(nf) for i in range(nf)])
    assert _rel(c[0].cpu().numpy(), want) < 2e-6
    assert torch.equal(W.forwardTransform(x, coef_dtype=torch.bfloat16).frameletArray, c.to(torch.bfloat16))
