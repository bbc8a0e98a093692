"""The default cone forward on both sides of the limit of the tracked walk's copy
(many thin frames here; large volumes alike): each form bit for bit against
the oracle, in FP32 and from 16-bit volumes."""
import numpy as np
import pytest
import torch

from graph_kernels import captured_kernels
from helpers import bits_equal, first_mismatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("nt, tracked", [(13107, True), (13108, False)])
def test_both_copies(gpu, oracle, nt, tracked, dtype):
    from framelab_amd import _lib, geometry as G
    from framelab_amd.projector import _DT, Projector
    seen = [0, 0, 5000, nt - 1, nt - 1, nt - 1]
    p = G.cone_para(40, 24, 6, N=(34, 34, 2), L=(2.0, 2.0, 0.2), SO=4.0, OD=4.0, Ly=G.full_fan_width(), Lz=0.6)
    P = Projector(G.with_frames(p, seen))
    x = torch.zeros(P.vol_shape, device=gpu, dtype=dtype)
    for f in set(seen):
        x[f] = torch.from_numpy(np.random.default_rng(f).random((2, 34, 34), dtype=np.float32)).to(gpu).to(dtype)
    y = torch.empty(P.sino_shape, device=gpu)
    names = captured_kernels(lambda st: _lib.check(_lib.lib().fl_forward(P.handle, x.data_ptr(), _DT[dtype], y.data_ptr(), 0, st)))
    assert [("k_to_cone_bricks" in n, "k_fwd_cone_tr" in n) for n in names] == [(tracked, False), (False, tracked)]
    if not tracked:
        assert "k_to_bricks" in names[0] and "Li4ELi4ELi4E" in names[0]
    y = P.forward(x, dtype=torch.float32).cpu().numpy()
    # the oracle on the frames that views see
    used = sorted(set(seen))
    small = G.with_frames(p, [used.index(f) for f in seen])
    yo = oracle.siddon_cone_f32(x[used].float().cpu().numpy().ravel(), small)
    assert bits_equal(y.ravel(), yo), first_mismatch(y, yo)
