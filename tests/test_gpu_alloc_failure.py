"""An allocation that fails when the particles' fourth components have to move
into arrays of their own leaves the simulation as it was."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))

PROGRAM = """
import ctypes, sys
oom = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # before the product library
import numpy as np
import gpusmoldyn_amd as smd
from gpusmoldyn_amd import configs
L = smd.lib()
vp = ctypes.c_void_p
L.smd_ps_create.restype = vp
L.smd_ps_create.argtypes = [vp, vp, vp, ctypes.c_uint, ctypes.c_int]
for f in ("smd_ps_update", "smd_ps_num_particles", "smd_ps_destroy"):
    getattr(L, f).argtypes = [vp]
L.smd_ps_get_positions.argtypes = [vp, vp, ctypes.c_uint]
L.smd_ps_set_positions.argtypes = [vp, vp, ctypes.c_int, ctypes.c_int]
spec, pos, types = configs.ref_test2(3000)
n = len(types)
ends = []
for fail in (0, 1, 2):
    ps = L.smd_ps_create(ctypes.byref(spec), pos.ctypes.data, types.ctypes.data, n, 0)
    assert ps
    for _ in range(3):
        assert L.smd_ps_update(ps) > 0
    if fail:
        other = np.full((1, 4), 0.3, np.float32)  # a component whose bits leave no room for a type
        oom.oom_arm(fail)
        assert L.smd_ps_set_positions(ps, other.ctypes.data, 0, 1) != 0
        print("allocation", fail, "failed:", smd.last_error(), flush=True)
    for _ in range(3):
        assert L.smd_ps_update(ps) > 0
    out = np.zeros((n, 4), np.float32)
    assert L.smd_ps_get_positions(ps, out.ctypes.data, n) == 0
    ends.append(out.copy())
    if fail:  # with memory at hand it works
        assert L.smd_ps_set_positions(ps, other.ctypes.data, 0, 1) == 0
        assert L.smd_ps_update(ps) > 0
        assert L.smd_ps_get_positions(ps, out.ctypes.data, n) == 0 and np.float32(0.3) in out[:, 3]
    L.smd_ps_destroy(ps)
assert all(np.array_equal(e, ends[0]) for e in ends)
"""


def test_failed_allocation_keeps_the_state(gpu, tmp_path):
    shim = os.path.join(HERE, "cpp", "liboom.so")
    assert os.path.exists(shim), "tests/cpp/liboom.so not built (run __graft_entry__.build())"
    r = subprocess.run([sys.executable, "-u", "-c", PROGRAM, shim], capture_output=True, text=True, timeout=100,
                       cwd=os.path.dirname(HERE))
    print(r.stdout, flush=True)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
    assert r.stdout.count("failed:") == 2
