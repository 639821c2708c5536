"""The autotuner's choices on both sides of the counts at which small launches go to
the row kernels (24,576 for the force, 40,960 for density), which ignore the block
size: a choice of its own on each side, made again when a push passes a line, and
never against a choice that the caller has fixed.  Read from the file of choices."""
import numpy as np
import pytest

from enjaparticles_amd import _native as N
from enjaparticles_amd import scenes
from enjaparticles_amd.rtps import RTPS

pytestmark = pytest.mark.gpu


def _system(tmp_path, monkeypatch, box, count=0):
    monkeypatch.setenv("RTPS_TUNE_CACHE", str(tmp_path / "choices"))
    rng = np.random.default_rng(3)
    pos = np.ones((48000, 4), np.float32)
    pos[:, :3] = rng.uniform(0.02, box - 0.02, (48000, 3))
    s = RTPS.generateSystemInstance(scenes.dam_settings(box, 48000))
    return s, pos


def _choices(tmp_path):
    f = tmp_path / "choices"
    return [line.split()[0] for line in f.read_text().splitlines()] if f.exists() else []


def test_a_choice_on_each_side_of_the_lines(cuda, tmp_path, monkeypatch):
    box = 2.12     # a grid of its own: nothing in the process's cache fits it
    s, pos = _system(tmp_path, monkeypatch, box)
    at = 0
    want = 0
    for upto, new in ((20000, 1), (24576, 0), (24577, 1), (32768, 0), (32769, 0), (40960, 0), (40961, 1), (48000, 0)):
        # (32,769 begins a size class, but is no line: the choice stays)
        s.pushParticles(pos[at:upto], np.zeros_like(pos[at:upto]))
        at = upto
        for _ in range(2):
            s.step(2)
        want += new
        assert len(_choices(tmp_path)) == want, upto
    s.close()
    assert len(set(_choices(tmp_path))) == 3
    for upto in (30000, 22000):               # other systems on the same grid: in the cache
        s, pos = _system(tmp_path, monkeypatch, box)
        s.pushParticles(pos[:upto], np.zeros_like(pos[:upto]))
        s.step(2)
        s.close()
    assert len(_choices(tmp_path)) == 3


def test_a_fixed_choice_stays(cuda, tmp_path, monkeypatch):
    s, pos = _system(tmp_path, monkeypatch, 2.16)
    s.setOption(N.OPT_BLOCK_DENSITY, 128)
    s.setOption(N.OPT_BLOCK_FORCE, 256)
    s.pushParticles(pos[:24000], np.zeros_like(pos[:24000]))
    s.step(2)
    s.pushParticles(pos[24000:], np.zeros_like(pos[24000:]))
    s.step(2)
    assert _choices(tmp_path) == []
    s.close()


def test_block_sizes_are_not_timed_where_they_have_no_effect(cuda, tmp_path, monkeypatch, capfd):
    s, pos = _system(tmp_path, monkeypatch, 2.2)
    monkeypatch.setenv("RTPS_TUNE_VERBOSE", "1")
    timed = []
    for a, b in ((0, 24576), (24576, 40960), (40960, 40961)):
        s.pushParticles(pos[a:b], np.zeros_like(pos[a:b]))
        capfd.readouterr()
        s.step(1)
        err = capfd.readouterr().err
        timed.append((err.count("density block"), err.count("force loop 5"), err.count("force loop 4")))
    s.close()
    assert timed == [(1, 1, 3), (1, 3, 3), (3, 3, 3)]


def test_the_lines_are_lower_where_particles_have_more_neighbours(cuda, tmp_path, monkeypatch):
    """A smoothing length of 2.5 spacings, 65 neighbours at rest: 40 / 65 of the
    counts (15,020 and 25,033); of four, 268 neighbours: no row kernels."""
    monkeypatch.setenv("RTPS_TUNE_CACHE", str(tmp_path / "choices"))
    rng = np.random.default_rng(5)
    pos = np.ones((30000, 4), np.float32)
    pos[:, :3] = rng.uniform(0.02, 1.3, (30000, 3))
    want = 0
    for h, steps in (("0.05", ((10000, 1), (15015, 0), (15030, 1), (25020, 0), (25050, 1))), ("0.08", ((2000, 1), (2040, 0)))):
        st = dict(scenes.dam_settings(1.32, 48000), smoothing_distance=h)
        with RTPS.generateSystemInstance(st) as s:
            at = 0
            for upto, new in steps:
                s.pushParticles(pos[at:upto], np.zeros_like(pos[at:upto]))
                at = upto
                s.step(1)
                want += new
                assert len(_choices(tmp_path)) == want, (h, upto)


@pytest.mark.parametrize("h,n", [("0.05", 15000), ("0.05", 15040), ("0.05", 25050), ("0.06", 8000), ("0.08", 2000)])
def test_both_kinds_of_kernel_give_the_same_bits(cuda, h, n):
    """The rows and, through the tile queues, the tiles (which the queues always take)."""
    out = []
    for queues in (0, 1):
        sc = scenes.dam_custom(32, 32, 32, seed=8)
        with RTPS.generateSystemInstance(dict(sc.settings, smoothing_distance=h)) as s:
            s.setOption(N.OPT_TILE_QUEUES, queues)
            s.setOption(N.OPT_BLOCK_DENSITY, 64)
            s.setOption(N.OPT_BLOCK_FORCE, 64)
            s.pushParticles(sc.pos[:n], sc.vel[:n])
            s.step(4)
            out.append([s.read(f) for f in ("pos", "vel", "density")])
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
