"""A program that ends with terrains still in device memory ends with its own exit
status: they are closed before the context that they are on."""
import os
import subprocess
import sys

import pytest

PROGRAM = """
import sys
from fastlem_amd import _native
from fastlem_amd.device import DeviceBatch, DeviceTerrain
from fastlem_amd.generator import context
from conftest import comb_terrain
a, b = comb_terrain(24, 6), comb_terrain(40, 2)
_native.check(_native.lib().fl_ctx_set_profiling(context(), 1))
terrain = DeviceTerrain(*(a[k] for k in ("row_ptr", "col", "length", "area", "erodibility", "uplift", "init_elevation",
                                         "outlets")))
batch = DeviceBatch([a, b])
print(terrain.solve(), batch.solve()[1], flush=True)
sys.exit(3)
"""


@pytest.mark.gpu
def test_terrains_alive_at_the_end():
    tests = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([os.path.dirname(tests), tests]))
    r = subprocess.run([sys.executable, "-c", PROGRAM], env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 3, (r.returncode, r.stdout, r.stderr[-2000:])
