"""rtps_collision_triangles on both sides of the lines between its two routes,
triangles listed per cell (few particles, many triangles) and blocks of particles
culled against the triangles: sets whose grid is hard to choose, particles in
random and in sorted order, against the restatement that tries every pair.

Bars: hit sets equal, forces within 1e-4 of the largest triangle force (FP32 with
fused multiply-adds on the GPU, one rounding per operation in the restatement)."""
import numpy as np
import pytest

import collision_tri_oracle as T
from enjaparticles_amd import ops, scenes
from enjaparticles_amd.rtps import RTPS

pytestmark = pytest.mark.gpu

FAR = np.float32([20, -12, 8])


def _sheet(n, count):
    x = np.linspace(0.05, 0.95, n + 1)
    g = np.stack([*np.meshgrid(x, x, indexing="ij"), np.full((n + 1, n + 1), 0.5)], -1)
    a, b, c, d = g[:-1, :-1], g[1:, :-1], g[1:, 1:], g[:-1, 1:]
    t = np.stack([np.stack([a, b, c], 2), np.stack([a, c, d], 2)], 2).reshape(-1, 3, 3).astype(np.float32)
    assert len(t) >= count
    return t[:count]


def _tris(kind, count):
    if kind == "huge":        # one triangle 400 times the others' size over all of them
        return np.concatenate([_sheet(24, count - 1), [[(-20, -20, 0.49), (40, -20, 0.49), (0, 60, 0.49)]]]).astype(np.float32)
    if kind == "far":         # a second cluster 25 m away
        t = _sheet(24, (count + 1) // 2)
        return np.concatenate([t, t + FAR])[:count]
    t = _sheet(24, count)
    if kind == "degenerate":  # no area, not a number, infinite: never hit
        t[0, 1] = t[0, 0]
        t[1, 0, 0] = np.nan
        t[2, 2, 1] = np.inf
    return t


@pytest.mark.parametrize("kind", ["plain", "huge", "far", "degenerate"])
@pytest.mark.parametrize("num,count", [(16384, 1024), (16385, 1024), (16384, 1023), (1, 1024), (257, 1025)])
def test_both_routes_match_the_restatement(cuda, kind, num, count):
    import torch
    tris = _tris(kind, count)
    rng = np.random.default_rng(6)
    pos = np.ones((num, 4), np.float32)
    pos[:, :2] = rng.uniform(-0.1, 1.1, (num, 2))
    pos[:, 2] = 0.495 + rng.uniform(-0.03, 0.03, num)
    if kind == "far":
        pos[::2, :3] += FAR
    if kind == "plain":
        pos = pos[np.lexsort((pos[:, 0], np.floor(pos[:, 1] / 0.04)))]
    vel = np.zeros((num, 4), np.float32)
    vel[:, :3] = rng.normal(0, 0.5, (num, 3))
    vel[::97] = 0.0
    force = rng.normal(0, 1, (num, 4)).astype(np.float32)
    with RTPS.generateSystemInstance(scenes.dam_custom(8, 8, 4, seed=1).settings) as s:
        sp, _, _ = s.params()
    got = ops.collision_triangles(*(torch.from_numpy(x).to(cuda) for x in (pos, vel, force)), tris, sp).cpu().numpy()
    with np.errstate(invalid="ignore"):
        want = T.collision_triangles(pos, vel, force, tris, sp.simulation_scale, sp.boundary_distance,
                                     sp.boundary_stiffness, sp.boundary_dampening)
    hit = np.abs((want - force)[:, :3]).max(1) > 0
    assert num < 1000 or hit.sum() > 300
    assert np.array_equal(np.abs((got - force)[:, :3]).max(1) > 0, hit)
    np.testing.assert_allclose(got, want, rtol=0, atol=1e-4 * max(np.abs(want - force).max(), 1e-30))
