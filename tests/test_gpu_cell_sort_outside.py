"""Many particles outside the grid, in the counting sort by cell: the order and the
states of the digit passes (RTPS_OPT_BUCKET_SORT 0), in one block and in several
kernels, one system or the scenes of a batch, at the edges of waves and of the
words that count them; and at a cost that grows with their number, not its square."""
import time

import numpy as np
import pytest

from enjaparticles_amd import scenes
from enjaparticles_amd.rtps import RTPS, BatchedSPH

pytestmark = pytest.mark.gpu


def _leave(pos, share, seed):
    """A share of the particles (all of them: 1) put outside the grid, on both sides."""
    rng = np.random.default_rng(seed)
    out = rng.random(len(pos)) < share
    pos[out, 2] = np.where(rng.random(out.sum()) < 0.5, np.float32(500.0), np.float32(-500.0))
    return pos


def _free(n, seed, box=0.9):
    pos = np.ones((n, 4), np.float32)
    pos[:, :3] = np.random.default_rng(seed).uniform(0.05, box - 0.05, (n, 3))
    return pos


# outside: 64 and 65 at the line inside the one-block sort; nearly all; all
@pytest.mark.parametrize("n,share", [(640, 64 / 640), (640, 65 / 640), (1025, 0.9), (4096, 0.95), (4096, 1), (4097, 0.95),
                                     (4097, 1), (20011, 0.5), (327680, 0.95)])
def test_one_system(n, share):
    box = 0.9 if n < 10000 else 2.4
    pos = _free(n, n, box)
    if n == 640:
        pos[np.random.default_rng(2).permutation(n)[:round(share * n)], 2] = np.float32(500.0)
    else:
        pos = _leave(pos, share, n)
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
                got += [s.read(f, n) for f in ("keys", "idx")]
                got += [s.read(f, m) for f in ("pos_s", "density", "pos", "vel")]
            out.append(got)
    assert out[0][0] < n
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


def test_scenes_of_a_batch():
    """Scenes whose slots begin inside a wave, with unused slots, with one particle."""
    lots = [(1, 0, 1), (63, 1, 0.5), (5, 2, 1), (40, 0, 0.9), (700, 300, 0.95), (0, 100, 0), (1, 0, 0), (2049, 7, 1),
            (33000, 96, 0.95), (2, 0, 0.5)]
    pos = [_leave(_free(n, 20 + k), share, k) for k, (n, _, share) in enumerate(lots)]
    st = [scenes.dam_settings(0.9, n + spare) for n, spare, _ in lots]
    b = BatchedSPH(st)
    for k, p in enumerate(pos):
        if len(p):
            b.pushParticles(k, p, np.zeros_like(p))
    b.step(1)
    for k, (n, spare, _) in enumerate(lots):
        got_idx, got_keys = b.read(k, "idx", n + spare), b.read(k, "keys", n + spare)
        assert np.array_equal(got_idx[n:], np.arange(n, n + spare))
        if n == 0:
            continue
        with RTPS.generateSystemInstance(st[k]) as one:   # a system of its own, by digit passes
            one.setOption(15, 0)
            one.pushParticles(pos[k], np.zeros_like(pos[k]))
            one.step(1)
            assert np.array_equal(got_keys[:n], (np.uint32(k) << np.uint32(24)) | one.read("keys", n))
            assert np.array_equal(got_idx[:n], one.read("idx", n))
            m = one.getNum()
            assert b.getNum(k) == m
            assert np.array_equal(b.read(k, "pos_s", m), one.read("pos_s", m))
    b.close()


def _timed(step, sync):
    sync()
    t = time.perf_counter()
    step()
    sync()
    return time.perf_counter() - t


def test_cost_of_one_system():
    n = 327680
    sc = scenes.dam_custom(128, 128, 20, seed=3)
    assert sc.n == n
    far = sc.pos.copy()
    far[n // 20:, 2] = np.float32(500.0)
    took = []
    for bucket in (1, 0):
        best = []
        for _ in range(2):
            with RTPS.generateSystemInstance(sc.settings) as s:
                s.setOption(15, bucket)
                s.pushParticles(sc.pos, sc.vel)
                s.step(3)
                s.write("pos", far)
                best.append(_timed(lambda: s.step(1), s.synchronize))
                assert s.getNum() == n // 20
        took.append(min(best))
    print(f"step with 311,296 particles outside: {1e3 * took[0]:.2f} ms, by digit passes {1e3 * took[1]:.2f} ms")
    assert took[0] < 3 * took[1]


def test_cost_of_a_batch():
    n = 400000
    sc = scenes.dam_custom(128, 128, 25, seed=3)
    pos = np.concatenate([sc.pos, sc.pos])[:n]
    far = pos[n // 20:].copy()
    far[:, 2] = np.float32(500.0)
    b = BatchedSPH([dict(sc.settings, max_num_particles=str(n))])
    b.pushParticles(0, pos[:n // 20], np.zeros_like(pos[:n // 20]))
    b.step(3)
    inside = min(_timed(lambda: b.step(1), b.synchronize) for _ in range(5))
    b.pushParticles(0, far, np.zeros_like(far))
    outside = _timed(lambda: b.step(1), b.synchronize)
    assert b.getNum(0) == n // 20
    b.close()
    print(f"step of 20,000 particles: {1e3 * inside:.2f} ms, with 380,000 outside {1e3 * outside:.2f} ms")
    assert outside < 10 * inside
