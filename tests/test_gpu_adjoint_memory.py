"""What an adjoint handle leaves of the device's memory: half of what is free when it
allocates its step records, however many steps a segment holds."""
import pytest
import torch

from enjaparticles_amd import scenes
from enjaparticles_amd.adjoint import AdjointSPH, BatchedAdjointSPH

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [False, True])
def test_records_leave_half_of_the_free_memory(cuda, batch):
    steps = 300                                    # of 131,072 particles: 6.9 GB of records
    room = 8 << 30
    torch.cuda.empty_cache()
    spare = torch.empty(torch.cuda.mem_get_info()[0] - room, dtype=torch.uint8, device=cuda)
    before = torch.cuda.mem_get_info()[0]
    try:
        if batch:
            st = [scenes.dam_custom(64, 64, 16, seed=k).settings for k in range(2)]
            sim = BatchedAdjointSPH(st, checkpoint_every=steps, max_steps=steps)
        else:
            sim = AdjointSPH(scenes.dam_custom(64, 64, 32, seed=31).settings, 131072, checkpoint_every=steps,
                             max_steps=steps)
        after = torch.cuda.mem_get_info()[0]
        sim.close()
    finally:
        del spare
        torch.cuda.empty_cache()                   # give the memory back to the device
    print(f"{before / 2**30:.2f} GiB free before, {after / 2**30:.2f} after")
    assert after > 0.4 * before
    assert after < 0.6 * before                    # and uses the other half
