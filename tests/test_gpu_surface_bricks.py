"""The colour field's bricks (32 x 2 x 1 nodes a wave) and the surface's tiles
(256 cubes a block) at their edges: lattices of one brick, one node more or
less, and many; a pool and a bar so dense that a row's candidates exceed the 256
of an LDS copy.

Bars: as for the field and the surface in general (the field within 1e-4 of its
maximum of the FP64 brute-force sum: FP32 sums of up to ~1,500 terms here, whose
rounding grows with the square root of their number to ~3e-6; the triangles
those of the GPU field, in order, vertices within 1e-5 of the box)."""
import numpy as np
import pytest

import surface_oracle as SO
from enjaparticles_amd import _native as N
from enjaparticles_amd import scenes
from enjaparticles_amd.rtps import RTPS

pytestmark = pytest.mark.gpu


def _pool():
    sc = scenes.dam_custom(12, 12, 8, seed=3)
    return sc.settings, sc.pos


def _bar():
    # 600 x 2 x 2 particles 0.0015 apart in x
    x, y, z = np.meshgrid(0.05 + 0.0015 * np.arange(600), [0.50, 0.51], [0.50, 0.51], indexing="ij")
    pos = np.stack([x, y, z, np.ones_like(x)], -1).reshape(-1, 4).astype(np.float32)
    return scenes.dam_settings(1.0, len(pos)), pos


@pytest.mark.parametrize("res", [2, 3, 31, 32, 33])
@pytest.mark.parametrize("scene", [_pool, _bar])
def test_field_and_surface_at_brick_edges(cuda, scene, res):
    st, pos = scene()
    s = RTPS.generateSystemInstance(st)
    s.pushParticles(pos, np.zeros_like(pos))
    s.step(1)
    f = s.colorField(res)
    sp, gp, gs = s.params()
    n = s.getNum()
    p = s.read("pos_s")[:n].astype(np.float64) * np.float64(np.float32(sp.simulation_scale))
    lo, hi = ((b.x, b.y, b.z) for b in (gs.bnd_min, gs.bnd_max))
    ref = SO.color_field(p, s.read("density")[:n], sp.mass, sp.smoothing_distance, sp.EPSILON, lo, hi, res)
    print(f"res {res}: {(ref > 0).sum()} nodes, max {ref.max():.4g}, off {np.abs(f - ref).max():.3g}", flush=True)
    assert np.abs(f - ref).max() <= 1e-4 * max(ref.max(), 1e-30)
    iso = 0.5 * float(f.max()) if f.max() > 0 else 0.5
    v, nn = s.surface(res, iso)
    tri, ntri = np.zeros((256, 16), np.int8), np.zeros(256, np.uint8)
    N.check(N.lib().rtps_mc_case_table(tri.ctypes.data, ntri.ctypes.data))
    wlo, whi = ((b.x, b.y, b.z) for b in (gp.bnd_min, gp.bnd_max))
    rv, _, _ = SO.marching_cubes(f, iso, (tri, ntri), wlo, whi)
    assert len(v) == len(nn) == len(rv)
    if len(v):
        assert np.abs(v - rv).max() <= 1e-5 * max(np.subtract(whi, wlo))
    s.close()
