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
        for _ in range(4):
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
    assert took[0] < 1.15 * took[1]
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
            assert seen[0] == "digits" and seen[-1] == "bins"
        res.append(e.get(0))
        e.close()
    assert np.array_equal(res[0][1], res[1][1])
    assert np.array_equal(res[0][0].view(np.uint32), res[1][0].view(np.uint32))
