"""Networks in which many particles are born and removed in each step: the
particles equal the oracle's bit for bit, and no stage of the step that only
keeps the books costs more than the stage that moves every particle."""
import math

import numpy as np
import pytest

from gpusmoldyn_amd import configs

pytestmark = pytest.mark.gpu


def _spec(smd, p, grid_bits, L, n_streams, seed, faces=None, offsets=0):
    """C splits in two or vanishes, each with probability p per step; A + B -> C."""
    rate = -math.log(1.0 - 2.0 * p) / 1e-3 / 2.0
    return configs.make_spec(
        D=[0.0, 1.0, 1.0, 0.5], dt=1e-3,
        reactions=[dict(order=2, reactants=[1, 2], products=[3], rate=1e-3),
                   dict(order=1, reactants=[3], products=[3, 3], rate=rate, pgem=0.2),
                   dict(order=1, reactants=[3], products=[], rate=rate)],
        box_lo=[0.0] * 3, box_hi=[L] * 3, faces=faces or [smd.BC_REFLECT] * 6, grid_bits=grid_bits,
        num_streams=n_streams, seed=seed, unbind_offsets=offsets)


def _system(smd, n, p, seed, w=1.0, **kw):
    L = max(4.0, (max(n, 1) / 2.048) ** (1.0 / 3.0))
    spec = _spec(smd, p, kw.pop("grid_bits", configs.grid_bits_for(max(n, 64))), L, max(64, n // 8), seed, **kw)
    pos = configs.uniform_box(np.random.default_rng(seed), n, 0.0, L)
    pos[:, 3] = w
    types = np.full(n, 3, np.int32)
    types[::16] = 1
    types[8::16] = 2
    return (spec, *configs.cell_order(spec, pos, types))


def _check(smd, orc, reps, steps):
    e = smd.Engine(0)
    for spec, pos, types in reps:
        e.add_replica(spec, pos, types)
    e.finalize()
    e.step(steps)
    got = [e.get(r) for r in range(len(reps))]
    e.close()
    g = smd.gauss_table()
    for r, (spec, pos, types) in enumerate(reps):
        sim = orc.sim_for(smd, spec, pos, types, cap=32 * len(types) + 4096)
        sim.step(g, steps)
        rp, rt = sim.state()
        assert np.array_equal(got[r][1], rt) and np.array_equal(got[r][0].view(np.uint32), rp.view(np.uint32)), r


@pytest.mark.parametrize("w", [1.0, 0.3])
@pytest.mark.parametrize("n", [1, 63, 1023, 1024, 1025, 4097, 70000])
def test_births_match_oracle(smd, orc, gpu, n, w):
    """One system around the edges of the 1024-slot tiles, fourth components in
    the records and apart."""
    print(f"births, {n} particles, w {w}", flush=True)
    _check(smd, orc, [_system(smd, n, 0.25, 5, w=w)], 5)


def test_births_of_replicas_match_oracle(smd, orc, gpu):
    """Replicas that start and end inside a tile, some within one tile."""
    print("births of replicas", flush=True)
    sizes = (700, 3, 40, 1024, 5000, 1, 281, 2000, 999)
    _check(smd, orc, [_system(smd, n, 0.05 + 0.04 * k, 30 + k) for k, n in enumerate(sizes)], 6)


def _stages(smd, n, p):
    e = smd.Engine(0)
    e.add_replica(*_system(smd, n, p, 7))
    e.finalize(8 * n)
    e.step(6)
    best = {}
    for _ in range(4):
        for k, v in e.profile(2).items():
            best[k] = min(best.get(k, 1e9), v)
    e.close()
    print(f"{n} particles, p {p}: " + " ".join(f"{k} {v:.1f}" for k, v in best.items()), flush=True)
    return best


def test_births_cost_less_than_the_move(smd, gpu):
    s = _stages(smd, 1 << 20, 0.05)
    assert s["scatter"] < 0.6 * s["producer"]


@pytest.mark.parametrize("n", [65535, 65536, 65537, 200000])
def test_holes_match_oracle(smd, orc, gpu, n):
    """Around the 64 tiles that a bookkeeping workgroup takes; most particles
    go in each step."""
    print(f"holes, {n} particles", flush=True)
    spec, pos, types = _system(smd, n, 0.3, 11)
    spec.rxn[1].rate *= 0.2
    _check(smd, orc, [(spec, pos, types)], 4)


def test_many_tiles_per_workgroup(smd, orc, gpu):
    """A capacity of more than 512 x 64 tiles: workgroups take several groups
    of tiles each."""
    print("holes, capacity 2^26", flush=True)
    spec, pos, types = _system(smd, 150000, 0.2, 12)
    e = smd.Engine(0)
    e.add_replica(spec, pos, types)
    e.finalize(1 << 26)
    e.step(4)
    gp, gt = e.get(0)
    e.close()
    sim = orc.sim_for(smd, spec, pos, types, cap=8 * len(types))
    sim.step(smd.gauss_table(), 4)
    rp, rt = sim.state()
    assert np.array_equal(gt, rt) and np.array_equal(gp.view(np.uint32), rp.view(np.uint32))


def test_holes_cost_less_than_the_move(smd, gpu):
    s = _stages(smd, 1 << 20, 0.25)
    assert s["finalize"] < 0.6 * s["producer"]


@pytest.mark.parametrize("n,p", [(4097, 0.5), (20000, 0.95), (20000, 0.995), (300, 1.0)])
def test_most_particles_vanish(smd, orc, gpu, n, p):
    """More holes than lanes between the particles of a wave."""
    print(f"{n} particles, {p} of the C vanish", flush=True)
    spec, pos, types = _system(smd, n, 0.25, 13)
    spec.rxn[1].rate = 0.0
    spec.rxn[2].rate = -math.log(max(1.0 - p, 1e-12)) / 1e-3
    _check(smd, orc, [(spec, pos, types)], 3)


def test_move_costs_the_same_with_many_holes(smd, gpu):
    few, many = _stages(smd, 100000, 0.01), _stages(smd, 100000, 0.45)
    assert many["producer"] < 1.6 * few["producer"]
