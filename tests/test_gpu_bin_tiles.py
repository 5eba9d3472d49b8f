"""The pass that bins one large system's keys, around the number of tiles whose
counts its second kernel adds up by itself (64 of 2048 keys), and with the few
particles that an absorbing box leaves: against the oracle, bit for bit."""
import numpy as np
import pytest

from gpusmoldyn_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [49153, 131071, 131072, 131073])
@pytest.mark.parametrize("absorb", [False, True])
def test_bins_match_oracle(smd, orc, gpu, n, absorb):
    spec = configs.make_spec(
        D=[0.0, 1.0, 1.0, 0.5], dt=40.0 if absorb else 1e-3,
        reactions=[dict(order=2, reactants=[1, 2], products=[3], rate=1e-3)],
        box_lo=[0.0] * 3, box_hi=[40.0] * 3, faces=[smd.BC_ABSORB if absorb else smd.BC_REFLECT] * 6,
        cell_size=[40.0 / 64] * 3 if not absorb else [40.0 / 8] * 3, grid_bits=(6, 6, 5) if not absorb else (3, 3, 3),
        num_streams=16384, seed=9)
    rng = np.random.default_rng(n)
    pos = configs.uniform_box(rng, n, 0.0, 40.0)
    types = rng.integers(1, 4, size=n).astype(np.int32)
    print(f"bin tiles {n} absorb {absorb}", flush=True)
    sim = orc.sim_for(smd, spec, pos, types, cap=n)
    e = smd.Engine(0)
    e.add_replica(spec, pos, types)
    e.finalize()
    g = smd.gauss_table()
    for k in (1, 2, 2):
        e.step(k)
        sim.step(g, k)
        gp, gt = e.get(0)
        rp, rt = sim.state()
        assert np.array_equal(gt, rt)
        assert np.array_equal(gp.view(np.uint32), np.ascontiguousarray(rp, np.float32).view(np.uint32))
    e.close()
