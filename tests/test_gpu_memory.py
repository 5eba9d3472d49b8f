"""Device memory per particle of capacity, and systems that start a step at the
most particles their capacity allows."""
import ctypes

import numpy as np
import pytest

from gpusmoldyn_amd import configs, serving

pytestmark = pytest.mark.gpu


def _free(smd):
    L = ctypes.CDLL(smd.LIB_PATH)
    L.hipMemGetInfo.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    free, total = ctypes.c_size_t(0), ctypes.c_size_t(0)
    assert L.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def _spec(smd, split, n_streams=512):
    rx = [dict(order=2, reactants=[1, 2], products=[3], rate=1e-3)]
    if split:
        rx.append(dict(order=1, reactants=[3], products=[3, 3], rate=1e9))  # every C, in every step
    return configs.make_spec(D=[0.0, 1.0, 1.0, 0.5], dt=1e-3, reactions=rx, box_lo=[0.0] * 3, box_hi=[16.0] * 3,
                             faces=[smd.BC_REFLECT] * 6, grid_bits=(4, 4, 4), num_streams=n_streams, seed=3)


# kind: (network splits, fourth component), most bytes per particle
KINDS = {"bind": (False, 1.0, 96), "bind_apart": (False, 0.3, 96), "split": (True, 1.0, 96),
         "split_apart": (True, 0.3, 96), "slots": (None, 1.0, serving.BYTES_PER_PARTICLE)}


@pytest.mark.parametrize("kind", list(KINDS))
def test_bytes_per_particle(smd, gpu, kind):
    split, w, most = KINDS[kind]
    cap = 1 << 26
    pos = configs.uniform_box(np.random.default_rng(1), 4096, 0.0, 16.0)
    pos[:, 3] = w
    types = (np.arange(4096) % 3 + 1).astype(np.int32)
    smd.Engine(0).close()
    warm = smd.Engine(0)  # the first engine sets up what the process keeps
    warm.add_replica(_spec(smd, False), pos, types)
    warm.finalize()
    warm.step(2)
    warm.sync()
    before = _free(smd)
    e = smd.Engine(0)
    if split is None:
        e.finalize_slots(2, 12, 512, cap, 1 << 13)
    else:
        e.add_replica(_spec(smd, split), pos, types)
        e.finalize(cap)
    per = (before - _free(smd)) / cap
    e.close()
    warm.close()
    print(f"{kind}: {per:.1f} bytes per particle of capacity", flush=True)
    assert per < most + 1.5  # tiles' words and allocation granules


@pytest.mark.parametrize("n,cap", [(1000, 2000), (1000, 2001), (4096, 8192), (1023, 4092)])
def test_every_particle_splits(smd, orc, gpu, n, cap):
    """Exactly as many particles as can enter a step, all of which split; the
    next step has to grow first."""
    spec = _spec(smd, True)
    pos = configs.uniform_box(np.random.default_rng(2), n, 0.0, 16.0)
    types = np.full(n, 3, np.int32)
    print(f"{n} particles split, capacity {cap}", flush=True)
    e = smd.Engine(0)
    e.add_replica(spec, pos, types)
    e.finalize(cap)
    sim = orc.sim_for(smd, spec, pos, types, cap=64 * n)
    g = smd.gauss_table()
    for steps in (1, 1, 3):
        e.step(steps)
        sim.step(g, steps)
        gp, gt = e.get(0)
        rp, rt = sim.state()
        assert np.array_equal(gt, rt) and np.array_equal(gp.view(np.uint32), rp.view(np.uint32))
    assert len(gt) == 32 * n
    d = e.debug_stage(2, len(gt))  # more particles than could enter before
    assert d["n_total"] == len(gt)
    e.close()
