"""Where particles lie so that counting keys per cell is the slower sort, an
engine turns to the digit passes by itself, and turns back later; the particles
are the same throughout."""
import time

import numpy as np
import pytest

from gpusmoldyn_amd import configs

pytestmark = pytest.mark.gpu


def _system(smd, n, bits, part=None, where="box", D=1.0):
    """n particles, mostly C (which pairs with nothing), on a grid of 2^bits
    cells; where: all over the box, in a slab of 1/part of its height, or in a
    block of 1/part per axis."""
    L = max(4.0, (n / 2.048) ** (1.0 / 3.0))
    gb = [bits // 3 + (bits % 3 > d) for d in range(3)]
    spec = configs.make_spec(
        D=[0.0, D, D, D], dt=1e-3, reactions=[dict(order=2, reactants=[1, 2], products=[3], rate=1e-6)],
        box_lo=[0.0] * 3, box_hi=[L] * 3, faces=[smd.BC_REFLECT] * 6, grid_bits=gb,
        num_streams=max(64, min(n // 8, 262144) // 64 * 64), seed=1)
    pos = configs.uniform_box(np.random.default_rng(1), n, 0.0, L)
    for d in {"box": (), "slab": (2,), "block": (0, 1, 2)}[where]:
        pos[:, d] = np.float32(0.4 * L) + pos[:, d] / np.float32(part)
    types = np.full(n, 3, np.int32)
    types[::64] = 1
    types[32::64] = 2
    return (spec, *configs.cell_order(spec, pos, types))


# name: replicas of (n, grid bits, part, where), whether the digit passes take over
SHAPES = {
    "coarse_100k": ([(100003, 12, None, "box")], True),
    "coarse_1m": ([(1 << 20, 14, None, "box")], True),
    "slab_48k": ([(48000, 18, 32, "slab")], True),
    "slab_1m": ([(1 << 20, 20, 32, "slab")], True),
    "block_1m": ([(1 << 20, 20, 16, "block")], True),
    "slabs_8x100k": ([(100003, 17, 32, "slab")] * 8, True),
    "dense_20k": ([(20000, 9, None, "box")], False),
    "even_100k": ([(100003, 17, None, "box")], False),
    "even_1m": ([(1 << 20, 20, None, "box")], False),
}


@pytest.mark.parametrize("name", list(SHAPES))
def test_no_slower_than_digits(smd, gpu, name):
    shapes, digits = SHAPES[name]
    reps = [_system(smd, *s) for s in dict.fromkeys(shapes)]
    reps = [reps[list(dict.fromkeys(shapes)).index(s)] for s in shapes]
    took, got, forms = [], [], []
    for knob in (1, 0):
        e = smd.Engine(0)
        for r in reps:
            e.add_replica(*r)
        e.finalize()
        e.set_knob(smd.KNOB_SEGMENTED_SORT, knob)
        e.step(12)
        e.sync()
        best = 1e9
        for _ in range(6):
            t = time.perf_counter()
            e.step(20)
            e.sync()
            best = min(best, (time.perf_counter() - t) / 20)
        took.append(best * 1e6)
        forms.append(e.sort_form())
        got.append([e.get(r) for r in range(len(reps))])
        e.close()
    print(f"{name}: {took[0]:.1f} us/step ({forms[0]}), by digits {took[1]:.1f}", flush=True)
    for (p1, t1), (p0, t0) in zip(*got):
        assert np.array_equal(t1, t0) and np.array_equal(p1.view(np.uint32), p0.view(np.uint32))
    assert took[0] < 1.25 * took[1]  # 1.35 to 2.7 where the form did not change
    assert (forms[0] in ("digits", "segments")) == digits


@pytest.mark.parametrize("single", [False, True])
def test_counts_again_when_particles_have_spread(smd, gpu, single):
    """A block that spreads out within some hundred steps: the digit passes run
    for a while, then keys are counted per cell again."""
    spec, pos, types = _system(smd, 60000, 15, 8, "block", D=400.0)
    res = []
    for knob in (1, 0):
        e = smd.Engine(0)
        e.add_replica(spec, pos, types)
        e.finalize()
        e.set_knob(smd.KNOB_SEGMENTED_SORT, knob)
        seen = []
        for _ in range(40):
            if single:
                for _ in range(80):
                    e.step(1)
            else:
                e.step(80)
            e.sync()
            seen.append(e.sort_form())
        print(f"spreading block, knob {knob}: {seen}", flush=True)
        if knob:
            assert "digits" in seen[:2] and seen[-1] == "bins"
        res.append(e.get(0))
        e.close()
    assert np.array_equal(res[0][1], res[1][1])
    assert np.array_equal(res[0][0].view(np.uint32), res[1][0].view(np.uint32))


# ensembles: (particles, grid bits) of each replica, and the form
ENSEMBLES = {
    # most slices empty
    "sparse_512": ([(2048, 17)] * 512, "segments"),
    "sparse_256": ([(2048, 18)] * 256, "digits"),
    "half_sparse_200": ([(2048, 17)] * 200, "replicas"),
    # a replica above 131072 particles beside many, and with few
    "one_large_of_many": ([(20000, 14)] * 120 + [(140000, 17)], "replicas"),
    "large_16": ([(262140, 17)] * 16, "replicas"),
    "large_9": ([(200001, 17)] * 9, "bins"),
    "too_large": ([(262141, 17)] * 17, "bins"),
}


@pytest.mark.parametrize("name", list(ENSEMBLES))
def test_form_of_ensembles(smd, gpu, name):
    shapes, form = ENSEMBLES[name]
    made = {s: _system(smd, *s) for s in dict.fromkeys(shapes)}
    took, got = [], []
    for radix, knob in ((0, 1), (11, 1), (0, 0)):
        e = smd.Engine(0, radix)
        for s in shapes:
            e.add_replica(*made[s])
        e.finalize()
        e.set_knob(smd.KNOB_SEGMENTED_SORT, knob)
        e.step(6)
        e.sync()
        if (radix, knob) == (0, 1):
            assert e.sort_form() == form
        best = 1e9
        for _ in range(5):
            t = time.perf_counter()
            e.step(10)
            e.sync()
            best = min(best, (time.perf_counter() - t) / 10)
        took.append(best * 1e6)
        got.append([e.get(r) for r in (0, len(shapes) // 2, len(shapes) - 1)])
        e.close()
    print(f"{name}: {took[0]:.1f} us/step ({form}), 11-bit digits {took[1]:.1f}, digits {took[2]:.1f}", flush=True)
    for other in got[1:]:
        for (p1, t1), (p0, t0) in zip(got[0], other):
            assert np.array_equal(t1, t0) and np.array_equal(p1.view(np.uint32), p0.view(np.uint32))
    assert took[0] < 1.2 * min(took[1:])


def test_grown_ensemble_keeps_its_form(smd, gpu):
    """An ensemble that grows to several times its first size, bins of more
    than 8 slices: by replica throughout, as by digits bit for bit."""
    res = []
    for knob in (1, 0):
        e = smd.Engine(0)
        for r in range(64):
            spec, pos, types = _system(smd, 2000 + 97 * r, 18)
            spec.num_reactions = 2
            spec.rxn[1].order = 1
            spec.rxn[1].reactants[0], spec.rxn[1].reactants[1] = 3, -1
            spec.rxn[1].products[0], spec.rxn[1].products[1] = 3, 3
            spec.rxn[1].nprod = 2
            spec.rxn[1].rate = 100.0
            e.add_replica(spec, pos, types)
        e.finalize()
        e.set_knob(smd.KNOB_SEGMENTED_SORT, knob)
        n0 = int(e.counts().sum())
        e.step(20)
        n = int(e.counts().sum())
        print(f"64 replicas grown from {n0} to {n}, knob {knob}: {e.sort_form()}", flush=True)
        assert n > 4 * n0
        if knob:
            assert e.sort_form() == "replicas"
        res.append([e.get(r) for r in (0, 31, 63)])
        e.close()
    for (p1, t1), (p0, t0) in zip(*res):
        assert np.array_equal(t1, t0) and np.array_equal(p1.view(np.uint32), p0.view(np.uint32))
