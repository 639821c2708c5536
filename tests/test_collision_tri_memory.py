"""Loading triangles without the memory for them: the call returns a status, and
a system that had triangles before steps on without any (its captured steps
name the freed ones)."""
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CALL = """
import ctypes as C, resource
from enjaparticles_amd import _native as N
lib = N.lib()
sp = N.SPHParams()
sp.simulation_scale, sp.boundary_distance = 1.0, 0.01
resource.setrlimit(resource.RLIMIT_AS, (8 << 30, 8 << 30))
# records of 2^31 - 1 triangles do not fit: the triangles themselves are never read
print("status", lib.rtps_collision_triangles(16, 4096, 4096, 4096, 4096, 2**31 - 1, C.byref(sp), None))
"""


def test_operator_without_host_memory():
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1", PYTHONPATH=ROOT)   # no device: nothing is launched
    r = subprocess.run([sys.executable, "-c", CALL], env=env, cwd=ROOT, capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    assert r.stdout.strip() == "status -1"


@pytest.mark.gpu
def test_system_without_device_memory(cuda):
    import torch
    from enjaparticles_amd import scenes
    from enjaparticles_amd._native import RTPSError
    from enjaparticles_amd.rtps import RTPS
    sc = scenes.dam_custom(12, 12, 8, seed=3)
    sheet = np.array([[[0, 0, 0.1], [1, 0, 0.1], [0, 1, 0.1]]], np.float32)
    many = np.random.default_rng(4).uniform(0, 1, (3000000, 3, 3)).astype(np.float32)   # 300 MB of records and lists
    out = []
    for fails in (True, False):
        with RTPS.generateSystemInstance(sc.settings) as s:
            s.pushParticles(sc.pos, sc.vel)
            s.loadTriangles(sheet)
            s.step(2)
            s.step(2)
            s.synchronize()
            if fails:
                torch.cuda.empty_cache()
                # the device filled but for 64 MB (it gives out somewhat more than it reports as free)
                spare = [torch.empty(torch.cuda.mem_get_info()[0] - (64 << 20), dtype=torch.uint8, device=cuda)]
                try:
                    while len(spare) < 64:
                        spare.append(torch.empty(32 << 20, dtype=torch.uint8, device=cuda))
                except torch.OutOfMemoryError:
                    pass
                del spare[-2:]
                torch.cuda.empty_cache()
                with pytest.raises(RTPSError):
                    s.loadTriangles(many)
                del spare
                torch.cuda.empty_cache()                       # give the memory back to the device
            else:
                s.loadTriangles(np.zeros((0, 3, 3), np.float32))
            s.step(4)
            out.append(s.read("pos"))
    np.testing.assert_array_equal(*out)
