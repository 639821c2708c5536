"""The colour field on lattices around the line between its two kernels, bricks of
nodes (from 28 nodes an axis, at most 1.8 cells apart along x and y) and a thread
per node: both against the brute-force sum, in boxes that are long along one axis;
and the cost of the coarsest lattice.

Bar: the field within 1e-4 of its maximum of the FP64 sum, as for the field in
general (FP32 sums over ~100 neighbours)."""
import time

import numpy as np
import pytest

import surface_oracle as SO
from enjaparticles_amd import _native as N
from enjaparticles_amd import scenes
from enjaparticles_amd.rtps import RTPS

pytestmark = pytest.mark.gpu

# res and the box's sides: 27 and 28 nodes at fine spacing; spacings of 1.8 cells
# of 0.04 and a little more, along each axis alone
LATTICES = [(27, (0.5, 0.5, 0.5)), (28, (0.5, 0.5, 0.5)), (28, (1.9, 0.3, 0.3)), (28, (1.99, 0.3, 0.3)),
            (28, (0.3, 1.9, 0.3)), (28, (0.3, 1.99, 0.3)), (28, (0.3, 0.3, 3.0)), (29, (2.6, 2.6, 0.3)), (4, (0.5, 1.1, 0.7))]


@pytest.mark.parametrize("res,box", LATTICES)
def test_field_around_the_line(cuda, res, box):
    rng = np.random.default_rng(7)
    n = 3000
    pos = np.ones((n, 4), np.float32)
    pos[:, :3] = rng.uniform(0.01, 0.99, (n, 3)) * box
    st = dict(scenes.dam_settings(1.0, n), domain_max=" ".join(str(b) for b in box) + " 0")
    with RTPS.generateSystemInstance(st) as s:
        s.pushParticles(pos, np.zeros_like(pos))
        s.step(1)
        f = s.colorField(res)
        sp, _, gs = s.params()
        m = s.getNum()
        lo, hi = ((b.x, b.y, b.z) for b in (gs.bnd_min, gs.bnd_max))
        ref = SO.color_field(s.read("pos_s")[:m].astype(np.float64), s.read("density")[:m], sp.mass,
                             sp.smoothing_distance, sp.EPSILON, lo, hi, res)
    assert (ref > 0).sum() > 20
    assert np.abs(f - ref).max() <= 1e-4 * ref.max()


def test_cost_of_the_coarsest_lattice(cuda):
    """Eight nodes in 262,144 particles, against a 128^3 lattice."""
    sc = scenes.dam_custom(80, 80, 41, seed=9)
    best = []
    with RTPS.generateSystemInstance(sc.settings) as s:
        s.pushParticles(sc.pos, sc.vel)
        s.step(2)
        for res in (2, 128):
            took = []
            for _ in range(9):
                s.synchronize()
                t = time.perf_counter()
                N.check(N.lib().rtps_sph_color_field(s._h, res, None))
                took.append(time.perf_counter() - t)
            best.append(min(took))
    print(f"2 nodes an axis {1e6 * best[0]:.0f} us, 128: {1e6 * best[1]:.0f} us")
    assert best[0] < 0.4 * best[1]
