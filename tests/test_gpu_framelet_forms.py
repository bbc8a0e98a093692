"""Which form of a framelet transform a size takes, on both sides of each line;
and the 3D analysis of four neighbours a thread returns the bits of the form of
one (which buffers off 16-byte alignment take), in every storage type."""
import ctypes as C

import pytest
import torch

from graph_kernels import captured_kernels, captured_launches

pytestmark = pytest.mark.gpu

F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16


def _analysis(kind, shape, u, c):
    from framelab_amd import _lib
    from framelab_amd.framelets import _DT
    return lambda st: _lib.check(_lib.lib().fl_framelet_forward(3, kind, 1, *reversed(shape), C.c_void_p(u.data_ptr()),
                                                                _DT[u.dtype], C.c_void_p(c.data_ptr()), _DT[c.dtype], st))


@pytest.mark.parametrize("ut, ct", [(F32, F32), (F32, BF16), (F32, F16), (BF16, BF16), (F16, F16)])
@pytest.mark.parametrize("nx, ny, nz, frame", [(196, 75, 74, "haar"), (132, 50, 48, "linear"), (500, 35, 19, "linear")])
def test_forms_agree(gpu, nx, ny, nz, frame, ut, ct):
    from framelab_amd.framelets import FrameletSystem
    S, shape = FrameletSystem(3, frame, 1), (nz, ny, nx)
    off = torch.randn(nx * ny * nz + 1, generator=torch.Generator(gpu).manual_seed(nx), device=gpu).to(ut)[1:]
    u = off.clone()
    c, want = (torch.empty((S.nbands,) + shape, device=gpu, dtype=ct) for _ in range(2))
    assert ["k_fwt3v" in n for n in captured_kernels(_analysis(S.kind, shape, u, c))] == [True]
    assert ["k_fwt3v" in n for n in captured_kernels(_analysis(S.kind, shape, off, want))] == [False]
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    _analysis(S.kind, shape, u, c)(st)
    _analysis(S.kind, shape, off, want)(st)
    assert torch.equal(c, want)


# (nx, ny, nz, frame, coefficient type, four a thread): rows of no whole 64-byte
# lines by size and by a row's share of working lanes, whole lines likewise
ANALYSIS = [
    (68, 48, 48, "linear", F32, True), (68, 47, 48, "linear", F32, False), (64, 96, 96, "linear", F32, False),
    (60, 96, 96, "linear", F32, False), (500, 19, 17, "linear", F32, True), (260, 25, 24, "linear", F32, True),
    (132, 50, 48, "linear", BF16, True), (132, 46, 48, "linear", BF16, False), (196, 75, 73, "haar", BF16, True),
    (196, 74, 75, "haar", F16, True), (260, 75, 73, "haar", BF16, False), (100, 75, 73, "haar", F32, True),
    (102, 75, 73, "haar", F32, False),
    (208, 99, 98, "linear", F32, True), (208, 97, 98, "linear", F32, False), (192, 256, 256, "linear", F32, False),
    (256, 199, 200, "linear", F32, True), (256, 128, 128, "linear", F32, False), (16, 192, 192, "linear", F32, False),
    (256, 60, 59, "haar", F32, True), (256, 59, 59, "haar", BF16, False), (192, 81, 81, "haar", F32, True),
    (192, 80, 81, "linear", BF16, False), (320, 112, 112, "linear", BF16, True), (320, 112, 112, "haar", F32, False),
    (128, 128, 128, "linear", BF16, False),
]


@pytest.mark.parametrize("nx, ny, nz, frame, dtype, wide", ANALYSIS)
def test_analysis_form(gpu, nx, ny, nz, frame, dtype, wide):
    from framelab_amd.framelets import FrameletSystem
    S, shape = FrameletSystem(3, frame, 1), (nz, ny, nx)
    u, c = torch.zeros(shape, device=gpu), torch.empty((S.nbands,) + shape, device=gpu, dtype=dtype)
    names = captured_kernels(_analysis(S.kind, shape, u, c))
    assert len(names) == 1 and ("k_fwt3v" in names[0]) == wide


def _synthesis(kind, shape, c, u):
    from framelab_amd import _lib
    nx, ny, nz = (tuple(reversed(shape)) + (1,))[:3]
    return lambda st: _lib.check(_lib.lib().fl_framelet_adjoint(len(shape), kind, 1, nx, ny, nz, C.c_void_p(c.data_ptr()),
                                                                _lib.FL_F32, C.c_void_p(u.data_ptr()), _lib.FL_F32, None, st))


# runs of slices: no more workgroups of 256-wide tiles than CUs if not by whole runs
@pytest.mark.parametrize("nx, ny, nz, groups", [(256, 96, 96, 144), (256, 64, 64, 256), (768, 64, 48, 144), (64, 64, 64, 256),
                                                (192, 64, 48, 288)])
def test_synthesis_runs(gpu, nx, ny, nz, groups):
    from framelab_amd.framelets import FrameletSystem
    S, shape = FrameletSystem(3, "linear", 1), (nz, ny, nx)
    c, u = torch.zeros((S.nbands,) + shape, device=gpu), torch.empty(shape, device=gpu)
    (name, grid), = captured_launches(_synthesis(S.kind, shape, c, u))
    assert "k_iwt3m" in name and grid == (groups, 1, 1)


@pytest.mark.parametrize("nx, ny, frame, march", [(1300, 999, "haar", False), (1300, 1001, "haar", True), (64, 64, "linear", True),
                                                  (64, 64, "cubic", True), (64, 64, "haar", False)])
def test_synthesis_2d_form(gpu, nx, ny, frame, march):
    from framelab_amd.framelets import FrameletSystem
    S, shape = FrameletSystem(2, frame, 1), (ny, nx)
    c, u = torch.zeros((S.nbands,) + shape, device=gpu), torch.empty(shape, device=gpu)
    assert ["k_iwt2m" in n for n in captured_kernels(_synthesis(S.kind, shape, c, u))] == [march]


@pytest.mark.parametrize("level", [1, 3])
def test_synthesis_2d_march_haar(gpu, level):
    """Haar images of the marching form's sizes, against its inverse property."""
    from framelab_amd.framelets import FrameletSystem
    S = FrameletSystem(2, "haar", level)
    u = torch.rand((1019, 1303), generator=torch.Generator(gpu).manual_seed(2), device=gpu)
    back = S.adjointTransform(S.forwardTransform(u).frameletArray)
    assert float((back - u).norm() / u.norm()) < 2e-6


@pytest.mark.parametrize("level", [1, 2, 3])
@pytest.mark.parametrize("frame", ["haar", "linear", "cubic"])
def test_synthesis_2d_forms_agree(gpu, frame, level):
    """The gather's bits are the march's: an image small enough for one form against
    the same rows in a taller one that takes the other (Haar: 1280 x 1000 twice over;
    the other frames march at both sizes)."""
    from framelab_amd.framelets import FrameletSystem
    S = FrameletSystem(2, frame, level)
    c = torch.randn((level, S.nbands, 1000, 1280), generator=torch.Generator(gpu).manual_seed(level), device=gpu)
    assert torch.equal(S.adjointTransform(torch.cat([c, c], 2)), S.adjointTransform(c).repeat(2, 1))
