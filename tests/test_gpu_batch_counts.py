"""The scenes' particle counts that a step leaves in host memory: before the
first step, after pushes, and after steps that delete particles."""
import pytest

from enjaparticles_amd import _native as N
from enjaparticles_amd import scenes
from enjaparticles_amd.rtps import BatchedSPH

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [0, 1])
def test_scene_counts_follow_the_steps(graph):
    sc = [scenes.dam_custom(6, 6, 6, seed=k) for k in range(3)]
    b = BatchedSPH([s.settings for s in sc])
    b.setOption(N.OPT_GRAPH, graph)
    assert [b.getNum(k) for k in range(3)] == [0, 0, 0]
    for k, s in enumerate(sc):
        pos = s.pos.copy()
        if k == 1:   # one particle outside the grid: deleted by the first step
            pos[3, 0] = 1e4
        b.pushParticles(k, pos, s.vel)
    assert [b.getNum(k) for k in range(3)] == [216, 216, 216]
    for _ in range(3):
        b.step(2)
        assert [b.getNum(k) for k in range(3)] == [216, 215, 216]
        assert b.read(1, "pos").shape == (215, 4)
    b.close()
