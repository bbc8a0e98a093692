"""The batch autotuner starts from the launch shape in force: a batch too small for
any grid to be cut keeps the default grids, and tuned batches return the same
bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _batch(n, k):
    from framelab_amd import geometry as G
    from framelab_amd.batch import ProjectorBatch
    return ProjectorBatch([G.fan_para(int(1.4 * n), n, N=(n, n), SO=4.0, OD=4.0, Ly=G.full_fan_width())] * k)


def test_small_batch_keeps_its_grids(gpu):
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    B = _batch(32, 2)
    for _ in range(2):
        tuned = B.autotune()
        assert (tuned["fwd_grid"], tuned["adj_grid"]) == (32 * cus, 16 * cus)


@pytest.mark.parametrize("n, k", [(32, 2), (130, 9)])
def test_same_bits(gpu, n, k):
    B = _batch(n, k)
    x = torch.randn(B.n_vol, generator=torch.Generator(gpu).manual_seed(n), device=gpu)
    y = B.forward(x)
    z = B.adjoint(y)
    B.autotune()
    assert torch.equal(B.forward(x), y) and torch.equal(B.adjoint(y), z)
