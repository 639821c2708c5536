"""rtps_collision_triangles with boundary distances that allow no hit (negative,
zero, infinite, not a number): its host side ends, with a status.  Without a
device the status is the device's error, in a process of its own so that an
endless loop or an abort shows as one."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CALL = """
import ctypes as C, sys
import numpy as np
from enjaparticles_amd import _native as N
from enjaparticles_amd.rtps import triangles_array
rng = np.random.default_rng(1)
tri = rng.uniform(0, 1, (200, 1, 3)) + rng.uniform(-0.01, 0.01, (200, 3, 3))
t = triangles_array(tri.astype(np.float32))
sp = N.SPHParams()
sp.simulation_scale, sp.boundary_distance = 1.0, float(sys.argv[1])
# no particle array is read: num = 16 particles at an address that nothing touches without a device
rc = N.lib().rtps_collision_triangles(16, 4096, 4096, 4096, t.ctypes.data, len(t), C.byref(sp), None)
print("status", rc)
"""


@pytest.mark.parametrize("dist", ["0.01", "0", "-0.005", "-0.05", "-0.2", "-1", "-1e30", "nan", "inf", "-inf"])
def test_distances_without_a_hit_end(dist):
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1", PYTHONPATH=ROOT)   # no device: nothing is launched
    r = subprocess.run([sys.executable, "-c", CALL, dist], env=env, cwd=ROOT, capture_output=True, text=True,
                       timeout=20)
    assert r.returncode == 0, r.stderr
    assert "status" in r.stdout
