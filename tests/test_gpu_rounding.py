"""The short square root and reciprocal return the bits of sqrtf and of division for
every float of the ranges they are used on."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["root", "reciprocal"])
def test_every_float(gpu, kind):
    from diag import diag
    bad = torch.ones(1, dtype=torch.int64, device=gpu)
    diag.check(diag.lib().fl_check_mid(["root", "reciprocal"].index(kind), bad.data_ptr(),
                                       torch.cuda.current_stream().cuda_stream), "fl_check_mid")
    assert int(bad.item()) == 0
