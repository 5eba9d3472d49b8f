"""Device arrays handed out by ParticleSystem::getCudaPosVBO / getCudaTypesVBO
stay as they are until the next update() or VBO call, also when particles are
read back or set in between."""
import ctypes

import numpy as np
import pytest

from gpusmoldyn_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3000, 50000])
def test_view_outlives_reads(smd, gpu, n):
    L = ctypes.CDLL(smd.LIB_PATH)
    vp = ctypes.c_void_p
    L.smd_ps_create.restype = vp
    L.smd_ps_create.argtypes = [vp, vp, vp, ctypes.c_uint, ctypes.c_int]
    for f in ("smd_ps_update", "smd_ps_num_particles", "smd_ps_destroy"):
        getattr(L, f).argtypes = [vp]
    L.smd_ps_get_positions.argtypes = L.smd_ps_get_types.argtypes = [vp, vp, ctypes.c_uint]
    L.smd_ps_set_positions.argtypes = [vp, vp, ctypes.c_int, ctypes.c_int]
    pos_vbo = L["_ZNK14ParticleSystem13getCudaPosVBOEv"]
    types_vbo = L["_ZNK14ParticleSystem15getCudaTypesVBOEv"]
    pos_vbo.restype = types_vbo.restype = vp
    pos_vbo.argtypes = types_vbo.argtypes = [vp]
    L.hipMemcpy.argtypes = [vp, vp, ctypes.c_size_t, ctypes.c_int]

    spec, pos, types = configs.ref_test2(n)
    n = len(types)
    ps = L.smd_ps_create(ctypes.byref(spec), pos.ctypes.data, types.ctypes.data, n, 0)
    assert ps
    print(f"view of {n} particles", flush=True)
    assert L.smd_ps_update(ps) >= 0
    n = L.smd_ps_num_particles(ps)
    obj = ctypes.cast(ps, ctypes.POINTER(vp))[0]

    def device(ptr, like):
        out = np.empty_like(like)
        assert L.hipMemcpy(out.ctypes.data, ptr, out.nbytes, 2) == 0  # device to host
        return out

    now_p, now_t = np.empty((n, 4), np.float32), np.empty(n, np.int32)
    assert L.smd_ps_get_positions(ps, now_p.ctypes.data, n) == 0
    assert L.smd_ps_get_types(ps, now_t.ctypes.data, n) == 0
    dt = types_vbo(obj)
    dp = pos_vbo(obj)
    assert np.array_equal(device(dp, now_p), now_p) and np.array_equal(device(dt, now_t), now_t)
    moved = np.ascontiguousarray(now_p[::-1])
    assert L.smd_ps_set_positions(ps, moved.ctypes.data, 0, n) == 0
    back = np.empty_like(now_p)
    assert L.smd_ps_get_positions(ps, back.ctypes.data, n) == 0
    assert np.array_equal(back, moved)
    assert np.array_equal(device(dp, now_p), now_p) and np.array_equal(device(dt, now_t), now_t)
    L.smd_ps_destroy(ps)
