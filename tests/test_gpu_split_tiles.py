"""The stage operators' split tiles (blocks of three waves over 64 particles,
one plane of the neighbourhood each) against the CPU oracle: particle counts
around a tile's edges and around the counts where the launches stop splitting
(3 * 2^16 for force, 2^20 for density).

Bars: those of the stage tests.  Density 1e-5 relative (FP32 sums of at most
about 60 positive terms: 60 roundings of 2^-24 are 3.6e-6); force and XSPH
1e-4 of each field's largest component.
"""
import numpy as np
import pytest

import oracle as O
from enjaparticles_amd import scenes

pytestmark = pytest.mark.gpu


def _sorted_state(n):
    nz = max(1, int(np.ceil((n / 4.0) ** (1.0 / 3.0))))
    while 4 * nz * nz * nz < n:
        nz += 1
    box = scenes.quarter_box(2 * nz, 2 * nz, nz)
    sp, gp, gs = O.derive_params(scenes.dam_settings(box, n))
    rng = np.random.default_rng(n)
    pos = scenes.lattice(2 * nz, 2 * nz, nz, seed=n, count=n, jitter=0.2)
    ve = np.zeros_like(pos)
    ve[:, :3] = rng.normal(scale=0.1, size=(n, 3)).astype(np.float32)
    k, i = O.sort_stable(*O.hash(pos, gp))
    start, end, _ = O.cellindices(k, gp.nb_cells)
    ps, _, es = O.permute(i, pos, ve, ve)
    return sp, gs, ps, es, start, end


@pytest.mark.parametrize("n", [1, 63, 64, 65, 200, 3 << 16, (3 << 16) + 1, 1 << 20, (1 << 20) + 1])
def test_density_and_force_at_the_edges_of_split_tiles(cuda, n):
    import torch
    from enjaparticles_amd import ops
    sp, gs, ps, es, start, end = _sorted_state(n)
    dev = [torch.from_numpy(np.ascontiguousarray(x)).to(cuda)
           for x in (ps, es, start.view(np.int32), end.view(np.int32))]
    od = O.density(ps, start, end, sp, gs)
    d = ops.density(dev[0], dev[2], dev[3], sp, gs)
    np.testing.assert_allclose(d.cpu().numpy(), od, rtol=1e-5, atol=0)
    if n > 1 << 18:
        return
    of, ox = O.force(ps, od, es, start, end, sp, gs)
    F, X = ops.force(dev[0], torch.from_numpy(od).to(cuda), dev[1], dev[2], dev[3], sp, gs)
    for a, b in ((F, of), (X, ox)):
        assert np.abs(a.cpu().numpy()[:, :3] - b[:, :3]).max() <= 1e-4 * max(np.abs(b[:, :3]).max(), 1e-20)
