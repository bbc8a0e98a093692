"""The 3D analysis of four neighbours a thread returns the bits of the form of one
(which buffers off 16-byte alignment take), in every storage type."""
import ctypes as C

import pytest
import torch

from graph_kernels import captured_kernels

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
