"""A job without particles has entered its slot once a step was taken, whether
that step was launched or replayed from a graph."""
import numpy as np
import pytest

from gpusmoldyn_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [1, 2, 3])
def test_empty_job_can_retire_after_replay(smd, gpu, steps):
    spec, pos, types = configs.c1(nA=600, nB=600, n_streams=256, grid_bits=(4, 4, 4))
    none = np.zeros((0, 4), np.float32), np.zeros(0, np.int32)
    e = smd.Engine(0)
    e.finalize_slots(2, 12, 1024, 1 << 14, 1 << 13)
    e.admit(0, spec, pos, types)
    e.step(9)  # graphs of this step count exist from here on
    e.step(steps)
    e.step(steps)
    e.admit(1, spec, *none)
    print(f"empty job, {steps} steps", flush=True)
    with pytest.raises(smd.SmdError):
        e.retire(1)  # not entered yet
    e.step(steps)
    e.retire(1)
    e.step(steps)
    assert e.counts()[1] == 0 and e.counts()[0] > 0
    e.close()
