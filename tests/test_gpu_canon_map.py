"""Steps read around the particles the step before removed, and find the ones
it gained behind the survivors: against the oracle bit for bit where many are
removed, few, all, where streams serve many particles, with fourth components
that do not fit the records, and with reads between steps."""
import numpy as np
import pytest

from gpusmoldyn_amd import configs

pytestmark = pytest.mark.gpu


def _system(smd, n, streams, decay, split, kf, seed, w="ones", absorb=False):
    rx = []
    if kf:
        rx.append(dict(order=2, reactants=[1, 2], products=[3], rate=kf))
    if decay:
        rx.append(dict(order=1, reactants=[1], products=[], rate=decay))
    if split:
        rx.append(dict(order=1, reactants=[2], products=[2, 1], rate=split))
    spec = configs.make_spec(
        D=[0.0, 1.0, 1.0, 0.5], dt=1e-2, reactions=rx, box_lo=[0.0] * 3, box_hi=[16.0] * 3,
        faces=[smd.BC_ABSORB if absorb else smd.BC_REFLECT] * 6, grid_bits=(5, 5, 4), num_streams=streams, seed=seed)
    rng = np.random.default_rng(seed)
    pos = configs.uniform_box(rng, n, 0.0, 16.0)
    if w == "any":
        pos[:, 3] = rng.uniform(-2.0, 2.0, size=n).astype(np.float32)
    types = rng.integers(1, 4, size=n).astype(np.int32)
    return spec, pos, types


# (n, streams, decay, split, kf, w, absorb)
CASES = {
    "few": (20000, 2500, 0.05, 0.0, 1e-3, "ones", False),
    "many": (30000, 4000, 30.0, 0.0, 1e-2, "ones", True),
    "all": (3000, 512, 1e6, 0.0, 1e-3, "ones", False),
    "deep_streams": (30011, 64, 2.0, 1.0, 1e-2, "ones", True),
    "births": (10000, 1250, 5.0, 8.0, 1e-2, "ones", False),
    "apart": (10000, 1250, 5.0, 8.0, 1e-2, "any", True),
    "one_stream": (700, 1, 3.0, 3.0, 1e-2, "any", False),
}


@pytest.mark.parametrize("name", list(CASES))
def test_steps_match_oracle(smd, orc, gpu, name):
    n, streams, decay, split, kf, w, absorb = CASES[name]
    spec, pos, types = _system(smd, n, streams, decay, split, kf, 77, w, absorb)
    print(f"canonical map {name}", flush=True)
    sim = orc.sim_for(smd, spec, pos, types, cap=40 * n)
    g = smd.gauss_table()
    e = smd.Engine(0)
    e.add_replica(spec, pos, types)
    e.finalize()
    counts = []
    for k in (1, 2, 3, 4, 1):  # single steps and captured pairs, read in between
        e.step(k)
        sim.step(g, k)
        gp, gt = e.get(0)
        rp, rt = sim.state()
        assert np.array_equal(gt, rt)
        assert np.array_equal(gp.view(np.uint32), rp.view(np.uint32))
        assert int(e.counts()[0]) == len(rt) and np.array_equal(
            e.species_counts(0), np.bincount(rt, minlength=spec.num_types).astype(np.uint32))
        counts.append(len(rt))
    e.close()
    assert len(set(counts)) > 1 or name == "all"


def test_ensemble_matches_replicas_alone(smd, orc, gpu):
    """Replicas with and without removals, births and fourth components of
    any value side by side, some empty."""
    reps = [_system(smd, n, max(64, n // 8), d, s, 1e-2, 90 + k, w)
            for k, (n, d, s, w) in enumerate(((5000, 0.0, 0.0, "ones"), (3000, 20.0, 5.0, "any"), (1, 1e6, 0.0, "ones"),
                                              (9000, 0.1, 0.0, "ones"), (130, 0.0, 60.0, "any"), (2049, 1e6, 0.0, "any")))]
    e = smd.Engine(0)
    for spec, pos, types in reps:
        e.add_replica(spec, pos, types)
    e.finalize()
    print("canonical map ensemble", flush=True)
    g = smd.gauss_table()
    sims = [orc.sim_for(smd, spec, pos, types, cap=40 * len(types) + 64) for spec, pos, types in reps]
    for k in (3, 4):
        e.step(k)
        for r, sim in enumerate(sims):
            sim.step(g, k)
            gp, gt = e.get(r)
            rp, rt = sim.state()
            assert np.array_equal(gt, rt) and np.array_equal(gp.view(np.uint32), rp.view(np.uint32)), r
    e.close()


def test_admitted_components_of_any_value(smd, orc, gpu):
    """A slot engine whose first job's fourth components fit the records takes
    a second one's that do not: both jobs equal the oracle alone."""
    e = smd.Engine(0)
    e.finalize_slots(3, 14, 4096, 1 << 17, 1 << 16)
    jobs = [_system(smd, 4000, 500, 1.0, 1.0, 1e-2, 21, "ones"), _system(smd, 3000, 400, 1.0, 1.0, 1e-2, 22, "any")]
    g = smd.gauss_table()
    print("canonical map admissions", flush=True)
    e.admit(0, *jobs[0])
    e.step(4)  # enters with the first step
    e.admit(1, *jobs[1])
    e.step(5)
    for slot, steps in ((0, 8), (1, 4)):
        spec, pos, types = jobs[slot]
        sim = orc.sim_for(smd, spec, pos, types, cap=40 * len(types))
        sim.step(g, steps)
        gp, gt = e.get(slot)
        rp, rt = sim.state()
        assert np.array_equal(gt, rt) and np.array_equal(gp.view(np.uint32), rp.view(np.uint32)), slot
    e.close()


@pytest.mark.parametrize("n,streams,kf,prob", [(3000, 1, 5.0, 0.0), (3000, 7, 5.0, 0.5), (3000, 3000, 5.0, 0.0),
                                               (30000, 1, 5.0, 0.0), (30000, 70, 5.0, 0.5), (30000, 30000, 5.0, 0.0)])
def test_pairs_of_one_stream_in_order(smd, orc, gpu, n, streams, kf, prob):
    """Reacting pairs drawn from few streams, worked off from the list of
    candidates (small systems) and by the walk over all particles (dense
    ones), with and without a coin per pair."""
    rx = dict(order=2, reactants=[1, 2], products=[3, 1], rate=kf)
    if prob:
        rx["prob"] = prob
    spec = configs.make_spec(
        D=[0.0, 1.0, 1.0, 0.5], dt=1e-3, reactions=[rx, dict(order=2, reactants=[1, 3], products=[2], rate=kf)],
        box_lo=[0.0] * 3, box_hi=[16.0] * 3, faces=[smd.BC_REFLECT] * 6, grid_bits=(4, 5, 5), num_streams=streams,
        seed=9)
    rng = np.random.default_rng(n + streams)
    pos = configs.uniform_box(rng, n, 0.0, 16.0)
    types = rng.integers(1, 4, size=n).astype(np.int32)
    print(f"pairs n={n} streams={streams} prob={prob}", flush=True)
    e = smd.Engine(0)
    e.add_replica(spec, pos, types)
    e.finalize()
    d = smd.Engine(0)
    d.add_replica(spec, pos, types)
    d.finalize()
    st = d.debug_stage(3, n)
    d.close()
    some = int((st["cand"] >= 0).sum())
    assert (some > 2200) == (n == 30000) and some > 40  # possible pairs: about half
    e.step(5)
    gp, gt = e.get(0)
    gs = e.get_streams(0)
    e.close()
    sim = orc.sim_for(smd, spec, pos, types)
    sim.step(smd.gauss_table(), 5)
    rp, rt = sim.state()
    assert np.array_equal(gt, rt) and np.array_equal(gp.view(np.uint32), rp.view(np.uint32))
    assert gs.shape[0] == streams and len(rt) < n
