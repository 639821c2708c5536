"""The nine-waves-per-tile kernels of small launches against the tile kernels
that look their rows up (RTPS_OPT_SHARED_ROWS 0): the same terms added in the
same order, so every state is bit-identical.

Sizes: one wave, its edges, the lines up to which density (40,960) and force
(24,576) take them.  States: free particles (windows of up to 20 candidates and
8 neighbours, which are worked out ahead of the turns), a clump (more of both,
several chunks of 32, more candidates than an LDS copy holds), short rows of
cells (waves that lie in several rows), particles outside the grid, positions
scaled by 0.31."""
import numpy as np
import pytest

import oracle as O
from enjaparticles_amd import _native as N
from enjaparticles_amd import scenes
from enjaparticles_amd.rtps import RTPS

pytestmark = pytest.mark.gpu


def _settings(n, kind):
    st = scenes.dam_settings(1.0, n)
    if kind == "scaled":
        for k in ("mass", "rest_distance", "smoothing_distance", "simulation_scale"):
            del st[k]
        sp, _, _ = O.derive_params(st)
        assert abs(sp.simulation_scale - 1.0) > 0.5
    return st


def _positions(n, kind):
    rng = np.random.default_rng(n)
    pos = np.ones((n, 4), np.float32)
    if kind == "clump":
        pos[:, :3] = 0.5 + 0.1 * (rng.random((n, 3)) - 0.5)
    elif kind == "short":      # a column: rows of cells of two or three particles' width
        pos[:, :3] = rng.random((n, 3)) * [0.08, 0.9, 0.9] + 0.05
    else:
        pos[:, :3] = 0.05 + 0.9 * rng.random((n, 3))
    if kind == "leaving":
        pos[::7, 2] = 40.0
    return pos


@pytest.mark.parametrize("n,kind", [(1, "free"), (2, "clump"), (63, "clump"), (64, "free"), (65, "clump"),
                                    (577, "short"), (2049, "clump"), (2049, "leaving"), (4097, "scaled"),
                                    (16384, "short"), (24576, "free"), (24577, "free"), (40960, "short"),
                                    (40961, "free"), (12000, "leaving")])
def test_row_kernels_equal_tile_kernels(n, kind):
    pos = _positions(n, kind)
    vel = np.zeros_like(pos)
    vel[:, :3] = 0.1 * np.random.default_rng(n + 1).standard_normal((n, 3))
    out = []
    for rows in (1, 0):
        with RTPS.generateSystemInstance(_settings(n, kind)) as s:
            s.setOption(N.OPT_SHARED_ROWS, rows)
            s.setOption(N.OPT_AUTOTUNE, 0)
            s.pushParticles(pos, vel)
            s.step(3)
            m = s.getNum()
            out.append((m, [s.read(f, m) for f in ("pos", "vel", "veleval", "density", "idx")]))
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1], out[1][1]):
        np.testing.assert_array_equal(a, b)
