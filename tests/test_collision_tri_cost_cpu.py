"""What the host does in rtps_collision_triangles: it prepares each triangle (normal,
bounding sphere), and for few particles lists them by the cells of a grid.  The yardstick is numpy
doing the preparation on the same machine.  Without a device the call ends with
the device's error when that work is done."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CALL = """
import ctypes as C, sys, time
import numpy as np
from enjaparticles_amd import _native as N
from enjaparticles_amd.rtps import triangles_array
g = np.linspace(0, 1, 301)
x, y = np.meshgrid(g, g, indexing="ij")
p = np.stack([x, y, 0.3 + 0.05 * np.sin(7 * x) * np.cos(5 * y)], -1)
a, b, c, d = p[:-1, :-1], p[1:, :-1], p[1:, 1:], p[:-1, 1:]
tri = np.concatenate([np.stack(t, 2).reshape(-1, 3, 3) for t in ((a, b, c), (a, c, d))]).astype(np.float32)
t = triangles_array(tri)
sp = N.SPHParams()
sp.simulation_scale, sp.boundary_distance = 1.0, 0.01
lib = N.lib()

def call():
    return lib.rtps_collision_triangles(int(sys.argv[1]), 4096, 4096, 4096, t.ctypes.data, len(t), C.byref(sp), None)

def prepare():
    v = t[:, :3, :3]
    n = np.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0])
    u = n / np.linalg.norm(n, axis=1, keepdims=True)
    m = v.astype(np.float64).mean(1)
    r = np.sqrt(((v - m[:, None]) ** 2).sum(2).max(1)).astype(np.float32)
    return np.concatenate([v.reshape(-1, 9), n, u, m, r[:, None], r[:, None] ** 2], 1, dtype=np.float32)

def best(f):
    out = []
    for _ in range(7):
        s = time.perf_counter()
        f()
        out.append(time.perf_counter() - s)
    return min(out)

assert call() != 0
print(best(call), best(prepare))
"""


def _times(particles):
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1", PYTHONPATH=ROOT)   # no device: nothing is launched
    r = subprocess.run([sys.executable, "-c", CALL, str(particles)], env=env, cwd=ROOT, capture_output=True, text=True,
                       timeout=60)
    assert r.returncode == 0, r.stderr
    ours, numpys = (float(x) for x in r.stdout.split())
    print(f"{1e3 * ours:.1f} ms, numpy {1e3 * numpys:.1f} ms")
    return ours, numpys


def test_lists_cost_a_few_preparations():
    """180,000 triangles, 7.4 cells each: 21 ms where numpy prepares for 73."""
    ours, numpys = _times(16)
    assert ours < 0.5 * numpys


def test_many_particles_need_no_lists():
    """They are culled by block: the same triangles in 6 ms."""
    ours, numpys = _times(100000)
    assert ours < numpys / 5
