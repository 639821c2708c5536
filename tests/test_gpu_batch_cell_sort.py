"""The order of a batch's slots after a step, sorted by cell for up to 2^20 slots
and by digit passes above: both the stable order of the reference's keys and the
16ths of a cell in x, scene by scene, unused slots in place at their scene's end.
Whole numbers: equal."""
import numpy as np
import pytest

from enjaparticles_amd import scenes
from enjaparticles_amd.rtps import RTPS, BatchedSPH

pytestmark = pytest.mark.gpu


def _scene(n, seed, kind):
    rng = np.random.default_rng(seed)
    pos = np.ones((n, 4), np.float32)
    pos[:, :3] = rng.uniform(0.05, 0.95, (n, 3))
    if kind == "stacked":       # one cell and equal positions
        pos[:, :3] = np.float32(0.5)
        pos[::3, 0] += np.float32(1e-3)
    if kind == "leaving":
        pos[::5, 1] = 50.0
    return pos


# (particles, unused slots, kind) of each scene; in the second batch the last scene takes it past 2^20 slots
BATCHES = {
    "small": [(1, 0, "free"), (63, 1, "free"), (700, 300, "stacked"), (0, 100, "free"), (2049, 0, "leaving"),
              (4000, 96, "free")],
    "large": [(500, 12, "leaving"), (3000, 1096, "free"), (2000, 1 << 20, "free")],
}


@pytest.mark.parametrize("batch", BATCHES)
def test_batch_order_is_the_stable_one(batch):
    lots = BATCHES[batch]
    pos = [_scene(n, 11 + k, kind) for k, (n, _, kind) in enumerate(lots)]
    st = [scenes.dam_settings(1.0, n + spare) for n, spare, _ in lots]
    b = BatchedSPH(st)
    for k, p in enumerate(pos):
        if len(p):
            b.pushParticles(k, p, np.zeros_like(p))
    b.step(1)
    for k, (n, spare, kind) in enumerate(lots):
        got_idx, got_keys = b.read(k, "idx", n + spare), b.read(k, "keys", n + spare)
        assert np.array_equal(got_idx[n:], np.arange(n, n + spare))
        if n == 0:
            continue
        with RTPS.generateSystemInstance(st[k]) as one:   # a system of its own, by digit passes
            one.setOption(15, 0)      # RTPS_OPT_BUCKET_SORT
            one.pushParticles(pos[k], np.zeros_like(pos[k]))
            one.step(1)
            keys = one.read("keys", n)
            assert np.array_equal(got_keys[:n], (np.uint32(k) << np.uint32(24)) | keys)
            assert np.array_equal(got_idx[:n], one.read("idx", n))
            assert np.array_equal(b.read(k, "pos_s", n), one.read("pos_s", n))
    b.close()
