"""A batch holds no copies of its images: its forward reads the packed ones."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_no_image_copies(gpu):
    from framelab_amd import geometry as G
    from framelab_amd.batch import ProjectorBatch
    # 153 600 rays and 64 MiB of image each
    paras = [G.fan_para(512, 300, N=(4096, 4096), SO=4.0, OD=4.0, Ly=G.full_fan_width())] * 4
    ProjectorBatch([G.fan_para(24, 16, N=(16, 16), SO=4.0, OD=4.0, Ly=G.full_fan_width())])   # loads what batches load
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    B = ProjectorBatch(paras)
    torch.cuda.synchronize()
    used = free - torch.cuda.mem_get_info()[0]
    assert B.n_vol == 4 << 24 and used < 100 << 20   # the per-ray tables take 22 MB
