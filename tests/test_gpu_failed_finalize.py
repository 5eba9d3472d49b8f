"""Reading from an engine whose finalize failed is refused: nothing was
allocated, and no count has been published."""
import ctypes

import numpy as np
import pytest

from gpusmoldyn_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("replicas", [1, 2])
def test_reads_are_refused(smd, gpu, replicas):
    spec, pos, types = configs.c1(nA=500, nB=500, n_streams=64)
    e = smd.Engine(0)
    for _ in range(replicas):
        e.add_replica(spec, pos, types)
    with pytest.raises(smd.SmdError):
        e.finalize(0xF0000000)  # beyond the 2^31 slots
    print(f"failed finalize, {replicas} replicas", flush=True)
    L, n = smd.lib(), ctypes.c_uint(77)
    with pytest.raises(smd.SmdError):
        e.counts()
    with pytest.raises(smd.SmdError):
        e.step(1)
    out, ty = np.zeros((1000, 4), np.float32), np.zeros(1000, np.int32)
    for r in range(replicas):
        assert L.smd_engine_get(e._h, r, out.ctypes.data, ty.ctypes.data, 1000, ctypes.byref(n)) != 0
        assert L.smd_engine_get(e._h, r, None, None, 0, ctypes.byref(n)) != 0
        assert L.smd_engine_species_counts(e._h, r, ty.ctypes.data) != 0
    e.close()
