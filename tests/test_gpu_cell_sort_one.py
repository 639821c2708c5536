"""The sort of small systems in one block (up to 4,096 particles on grids whose
counters fit its LDS) against the sort by digit passes (RTPS_OPT_BUCKET_SORT 0):
the same order, tables and states.  Sizes at the block's edges; free particles,
all in one cell, some outside the grid (then fewer than the launch has slots),
and a grid with too many cells for one block."""
import numpy as np
import pytest

from enjaparticles_amd import _native as N
from enjaparticles_amd import scenes
from enjaparticles_amd.rtps import RTPS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 1023, 1024, 1025, 4095, 4096, 4097])
@pytest.mark.parametrize("kind", ["free", "stacked", "leaving", "wide"])
def test_one_block_sort_equals_digit_passes(n, kind):
    rng = np.random.default_rng(n)
    box = 1.6 if kind == "wide" else 0.9      # 1.6: more than 60,000 cells
    pos = np.ones((n, 4), np.float32)
    pos[:, :3] = rng.uniform(0.05, box - 0.05, (n, 3))
    if kind == "stacked":
        pos[:, :3] = np.float32(0.4)
        pos[::3, 0] += np.float32(2e-3)
    if kind == "leaving":
        pos[::5, 1] = 50.0
    out = []
    for bucket in (1, 0):
        with RTPS.generateSystemInstance(scenes.dam_settings(box, n)) as s:
            s.setOption(15, bucket)      # RTPS_OPT_BUCKET_SORT
            s.pushParticles(pos, np.zeros_like(pos))
            got = []
            for _ in range(2):
                s.step(1)
                m = s.getNum()
                start, end = s.read("cell_start"), s.read("cell_end")
                got += [np.int64(m), start, end[start != 0xFFFFFFFF]]
                got += [s.read(f, m) for f in ("keys", "idx", "pos_s", "density", "pos", "vel")]
            out.append(got)
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
