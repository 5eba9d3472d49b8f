"""The counting cell sort: sorted keys, values and cell table of one step
against numpy's stable argsort of the keys the producer wrote, exactly, at the
edges of its slices, lists, windows and bins."""
import numpy as np
import pytest

from gpusmoldyn_amd import configs

pytestmark = pytest.mark.gpu


def _spec(smd, n_streams, grid_bits, L=16.0, faces=None, seed=11):
    # A + B -> C; most particles below are C, which pairs with nothing
    return configs.make_spec(
        D=[0.0, 1.0, 1.0, 0.5], dt=1e-3,
        reactions=[dict(order=2, reactants=[1, 2], products=[3], rate=1e-3)],
        box_lo=[0.0] * 3, box_hi=[L] * 3, faces=faces or [smd.BC_REFLECT] * 6, grid_bits=grid_bits,
        num_streams=n_streams, seed=seed)


def _particles(n, L, spread, rng):
    pos = np.empty((n, 4), np.float32)
    pos[:, :3] = rng.uniform(0.5 * L - 0.5 * spread, 0.5 * L + 0.5 * spread, size=(n, 3))
    pos[:, 3] = 1.0
    types = np.full(n, 3, np.int32)
    types[:: max(1, n // 50)] = 1
    types[1:: max(2, n // 50)] = 2
    return pos, types


# name: ([(n, grid bits, extent of the particles)], faces absorb)
CASES = {
    "one": ([(1, (2, 2, 2), 16.0)], False),
    "wave_edge": ([(65, (2, 2, 2), 16.0)], False),
    "ragged": ([(12347, (4, 5, 4), 16.0)], False),
    # sparse: many slices with hardly a particle
    "sparse_18_bits": ([(5003, (6, 6, 6), 16.0)], False),
    # every particle in one or two cells: several windows of one cell
    "point": ([(40000, (3, 3, 3), 0.01)], False),
    # dense middle cells beside empty slices, removed particles
    "dense_absorbing": ([(90001, (5, 5, 5), 15.99)], True),
    # one segment longer than a list entry's index
    "long_segment": ([((1 << 19) + 8193, (2, 2, 2), 16.0)], False),
    # few cells per slice, more cells than the list's first digit
    "cells_129_to_8192": ([(9001, (3, 3, 2), 16.0), (8192, (4, 4, 5), 16.0), (30000, (5, 4, 4), 16.0)], True),
    # an ensemble with empty and tiny replicas
    "ensemble": ([(0, (2, 2, 2), 16.0), (20011, (5, 5, 4), 16.0), (1, (3, 3, 3), 16.0), (0, (4, 4, 4), 16.0),
                  (11586, (5, 4, 4), 16.0), (70000, (6, 5, 5), 16.0)], True),
    # bins of the high key bits: 2^21 and 2^22 + 2^14 cells
    "bins": ([(300007, (7, 7, 7), 16.0)], True),
    "bins_point": ([(400000, (7, 7, 7), 0.02)], False),
    "bins_ensemble": ([(250000, (8, 7, 7), 16.0), (3000, (5, 5, 4), 16.0), (260000, (7, 7, 7), 4.0)], True),
}


@pytest.mark.parametrize("name", list(CASES))
def test_cell_sort_matches_argsort(smd, gpu, name):
    sizes, absorb = CASES[name]
    L = 16.0
    faces = [smd.BC_ABSORB] * 6 if absorb else None
    rng = np.random.default_rng(3)
    reps = []
    for k, (n, gb, spread) in enumerate(sizes):
        pos, types = _particles(max(n, 1), L, spread, rng)
        reps.append((_spec(smd, max(64, n // 8), gb, L, faces, seed=11 + k), pos[:n], types[:n]))
    total = sum(len(r[2]) for r in reps)
    print(f"cell sort {name}: {total} particles", flush=True)
    got = []
    for stage in (1, 2):
        e = smd.Engine(0)
        for spec, pos, types in reps:
            e.add_replica(spec, pos, types)
        e.finalize()
        got.append(e.debug_stage(stage, total))
        if stage == 2:
            first, lay = e.debug_first(), e.layout()
        e.close()
    keys = got[0]["keys"]
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(got[1]["keys"], keys[order])
    assert np.array_equal(got[1]["vals"], order.astype(np.uint32))
    dead = lay["total_buckets"]
    assert np.array_equal(first[: dead + 1], np.searchsorted(keys[order], np.arange(dead + 1, dtype=np.uint64)))
    assert first[dead + 1] == total
    assert got[1]["n_live"] == int((keys < dead).sum())
    if absorb:
        assert got[1]["n_live"] < total


@pytest.mark.parametrize("name", ["point", "long_segment", "ensemble", "bins_ensemble"])
def test_cell_sort_steps_match_digit_sort(smd, gpu, name):
    """Several steps (graph replays among them) with the counting sort equal
    those with the digit sort over all keys, bit for bit."""
    sizes, absorb = CASES[name]
    L = 16.0
    faces = [smd.BC_ABSORB] * 6 if absorb else None
    res = []
    for knob in (1, 0):
        rng = np.random.default_rng(3)
        e = smd.Engine(0)
        for k, (n, gb, spread) in enumerate(sizes):
            pos, types = _particles(max(n, 1), L, spread, rng)
            e.add_replica(_spec(smd, max(64, n // 8), gb, L, faces, seed=11 + k), pos[:n], types[:n])
        e.finalize()
        e.set_knob(smd.KNOB_SEGMENTED_SORT, knob)
        print(f"cell sort steps {name} knob {knob}", flush=True)
        e.step(5)
        res.append([e.get(r) for r in range(len(sizes))])
        e.close()
    for (p1, t1), (p0, t0) in zip(*res):
        assert np.array_equal(t1, t0) and np.array_equal(p1.view(np.uint32), p0.view(np.uint32))


def test_cell_sort_of_growing_system(smd, orc, gpu):
    """A system that doubles every few steps, past the size its slices were
    laid out for: the counting sort by replica, then by bins, equals the
    oracle bit for bit."""
    n, steps = 9000, 30
    spec = configs.make_spec(
        D=[0.0, 1.0, 1.0], dt=1e-2,
        reactions=[dict(order=1, reactants=[1], products=[1, 1], rate=10.0),
                   dict(order=2, reactants=[1, 2], products=[2], rate=1e-3)],
        box_lo=[0.0] * 3, box_hi=[16.0] * 3, faces=[smd.BC_REFLECT] * 6, grid_bits=(5, 5, 5), num_streams=2048, seed=5)
    rng = np.random.default_rng(8)
    pos = configs.uniform_box(rng, n, 0.0, 16.0)
    types = np.where(np.arange(n) < 8000, 1, 2).astype(np.int32)
    e = smd.Engine(0)
    e.add_replica(spec, pos, types)
    e.finalize()
    for k in range(0, steps, 5):
        print(f"growing system, {k} steps, {int(e.counts()[0])} particles", flush=True)
        e.step(5)
    gp, gt = e.get(0)
    e.close()
    sim = orc.sim_for(smd, spec, pos, types, cap=4 * len(gt))
    sim.step(smd.gauss_table(), steps)
    rp, rt = sim.state()
    assert len(gt) > 100000
    assert np.array_equal(gt, rt) and np.array_equal(gp.view(np.uint32), rp.view(np.uint32))
