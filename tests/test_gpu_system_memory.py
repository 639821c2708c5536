"""Device memory of a system whose grid has far more cells than the counting sort
takes: two tables of the cells (start and end), no counters for that sort."""
import numpy as np
import pytest
import torch

from enjaparticles_amd import scenes
from enjaparticles_amd.rtps import RTPS

pytestmark = pytest.mark.gpu


def test_large_grids_have_no_counters(cuda):
    torch.cuda.empty_cache()
    free = torch.cuda.mem_get_info()[0]
    with RTPS.generateSystemInstance(scenes.dam_settings(23.0, 1000)) as s:
        cells = s.nb_cells
        assert cells > 190_000_000
        used = free - torch.cuda.mem_get_info()[0]
        pos = np.ones((1000, 4), np.float32)
        pos[:, :3] = np.random.default_rng(1).uniform(5.0, 5.3, (1000, 3))
        s.pushParticles(pos, np.zeros_like(pos))
        s.step(2)
        assert s.getNum() == 1000
    print(f"{used / cells:.2f} bytes a cell")
    assert used < 9 * cells + (256 << 20)
