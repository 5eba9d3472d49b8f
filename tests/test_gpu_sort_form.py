"""The sort form that an engine reports is the one its steps run."""
import numpy as np
import pytest

from gpusmoldyn_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,replicas,form", [(16384, 1, "replicas"), (200000, 1, "bins"), (4000, 5, "replicas")])
def test_reported_forms(smd, gpu, n, replicas, form):
    e = smd.Engine(0)
    for k in range(replicas):
        spec = configs.c1_spec(n_streams=256, seed=k + 1, grid_bits=configs.grid_bits_for(n))
        types = np.where(np.arange(n) < n // 2, 1, 2).astype(np.int32)
        e.add_replica(spec, configs.uniform_box(np.random.default_rng(k), n, 0.0, 20.0), types)
    with pytest.raises(smd.SmdError):
        e.sort_form()  # not before finalize
    e.finalize()
    assert e.sort_form() == form
    e.set_sort(0)
    assert e.sort_form() == "digits"
    e.close()
    s = smd.Engine(0)
    s.finalize_slots(2, 12, 256, 1 << 14, 1 << 12)
    assert s.sort_form() == "segments"
    s.close()
