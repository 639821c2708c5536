"""Runs of steps replayed as one graph: calls of any lengths give the states of
single launches, bit for bit, also after what makes the graphs void (a push, an
option, a changed setting) and in a batch."""
import numpy as np
import pytest

from enjaparticles_amd import _native as N
from enjaparticles_amd import scenes
from enjaparticles_amd.rtps import RTPS, BatchedSPH

pytestmark = pytest.mark.gpu

CALLS = (1, 3, 4, 5, 9, 8, 2)


def test_system_runs_equal_launches():
    sc = scenes.dam_custom(10, 10, 8, seed=5)
    more = sc.pos[:40].copy()
    more[:, 1] += 0.3
    states = []
    for graph in (1, 0):
        with RTPS.generateSystemInstance(dict(sc.settings, max_num_particles="900")) as s:
            s.setOption(N.OPT_GRAPH, graph)
            s.pushParticles(sc.pos, sc.vel)
            got = []
            for change in range(4):
                for n in CALLS:
                    s.step(n)
                    got.append(s.read("pos"))
                if change == 0:
                    s.pushParticles(more, np.zeros_like(more))
                elif change == 1:
                    s.setOption(N.OPT_COLLISION, 0)
                elif change == 2:
                    s.setSetting("viscosity", 0.4)
            states.append(got)
    for a, b in zip(*states):
        np.testing.assert_array_equal(a, b)


def test_batch_runs_equal_launches():
    sc = [scenes.dam_custom(6 + k, 6, 6, seed=k) for k in range(3)]
    states = []
    for graph in (1, 0):
        b = BatchedSPH([s.settings for s in sc])
        b.setOption(N.OPT_GRAPH, graph)
        for k, s in enumerate(sc):
            b.pushParticles(k, s.pos, s.vel)
        got = []
        for change in range(2):
            for n in CALLS:
                b.step(n)
                got += [b.read(k, "pos") for k in range(3)]
            b.setOption(N.OPT_COLLISION, 0)
        b.close()
        states.append(got)
    for a, c in zip(*states):
        np.testing.assert_array_equal(a, c)
