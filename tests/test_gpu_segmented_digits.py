"""The digit sort that goes replica by replica on local cells, in engines that
run it (11- and 4-bit digits: those do not count keys per cell)."""
import numpy as np
import pytest

from gpusmoldyn_amd import configs

pytestmark = pytest.mark.gpu


def _both(smd, reps, steps, radix):
    res = []
    for knob, form in ((1, "segments"), (0, "digits")):
        e = smd.Engine(0, radix)
        for spec, pos, types in reps:
            e.add_replica(spec, pos, types)
        e.finalize()
        e.set_knob(smd.KNOB_SEGMENTED_SORT, knob)
        assert e.sort_form() == form
        e.step(steps)
        assert e.sort_form() == form
        res.append([e.get(r) for r in range(len(reps))])
        e.close()
    for r, ((p1, t1), (p0, t0)) in enumerate(zip(*res)):
        assert np.array_equal(t1, t0) and np.array_equal(p1.view(np.uint32), p0.view(np.uint32)), r
    return res[0]


@pytest.mark.parametrize("radix", [4, 11])
@pytest.mark.parametrize("big", [(4, 4, 4), (5, 4, 4), (6, 5, 5), (6, 6, 5)])
def test_digit_widths(smd, gpu, big, radix):
    """Largest grids of 2^12 to 2^17 buckets, with births, deaths in pairs, an
    absorbing face, an empty replica and one below a tile."""
    reps = []
    for k, (n, gb) in enumerate(((30000, big), (3000, (4, 4, 4)), (0, (3, 3, 3)), (200, (4, 4, 4)), (45000, big))):
        spec, pos, types = configs.c3(n=max(n, 1), n_blobs=4, sigma=1.0, n_streams=1024, grid_bits=gb, cell=0.15,
                                      L=20.0, seed=300 + k)
        spec.sphere[0][3] = 6.0
        spec.rxn[0].rate = 2.0
        reps.append((spec, pos[:n], types[:n]))
    print(f"segmented digits, largest grid {big}, radix {radix}", flush=True)
    assert sum(len(t) for _, t in _both(smd, reps, 8, radix)) > 0


def test_long_segments(smd, gpu):
    """Replicas above 64 tiles, whose tile counts are scanned digit by digit,
    between short ones."""
    reps = [configs.c3(n=n, n_blobs=8, sigma=2.0, n_streams=4096, grid_bits=(6, 6, 5), cell=0.2, L=40.0, seed=700 + k)
            for k, n in enumerate((20000, 300000, 5000, 530000, 70000))]
    print("segmented digits, long segments", flush=True)
    assert len(_both(smd, reps, 4, 11)[3][1]) > 64 * 4096


def test_many_replicas(smd, gpu):
    """More replicas than a workgroup has lanes, some empty."""
    rng = np.random.default_rng(5)
    reps = []
    for k in range(1100):
        n = int(rng.integers(0, 160)) if k % 37 else 0
        reps.append(configs.c1(nA=n // 2, nB=n - n // 2, kf=50.0, n_streams=64, seed=1000 + k, rng_seed=2000 + k,
                               grid_bits=(3, 3, 3)))
    print("segmented digits, 1100 replicas", flush=True)
    assert sum(int((t == 3).sum()) for _, t in _both(smd, reps, 6, 11)) > 0


def test_against_oracle(smd, orc, gpu):
    reps = configs.c4(n_rep=12, nmin=2048, nmax=16384)
    print("segmented digits against the oracle", flush=True)
    got = _both(smd, reps, 8, 11)
    for r, (spec, pos, types) in enumerate(reps):
        sim = orc.sim_for(smd, spec, pos, types)
        sim.step(smd.gauss_table(), 8)
        rp, rt = sim.state()
        assert np.array_equal(got[r][1], rt) and np.array_equal(got[r][0].view(np.uint32), rp.view(np.uint32)), r
