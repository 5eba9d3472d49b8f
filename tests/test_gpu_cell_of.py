"""The cell a particle falls in and the faces that act on it, for particles
that do not move, within a few units in the last place of cell borders and
faces: the same as one float32 division and the plain face rules say, bit for
bit."""
import numpy as np
import pytest

from gpusmoldyn_amd import configs

pytestmark = pytest.mark.gpu

f32 = np.float32
LO, HI = (-1.3, 0.1, 2.0), (17.9, 9.7, 50.0)
RADIUS = 0.25
# (faces, cell size, origin, grid bits); the grid need not cover the box
CASES = {
    "reflect": ("R" * 6, (0.6, 0.3, 3.0), (-1.3, 0.1, 2.0), (5, 5, 4)),
    "clamp_absorb": ("CARACC", (0.7, 0.31, 0.97), (-2.17, 0.0, 1.3), (6, 4, 6)),
    "small_cells": ("AAAAAA", (0.3, 0.3, 0.3), (-1000.1, -333.3, 0.7), (9, 8, 7)),
    "far_origin": ("RRCCAR", (0.6, 0.6, 0.6), (1e6, -1e5, 3.3e3), (4, 4, 4)),
}
KIND = {"C": 0, "R": 1, "A": 2}


def _near(values, steps=4):
    out = [np.asarray(values, f32)]
    up = down = out[0]
    for _ in range(steps):
        up, down = np.nextafter(up, f32(np.inf)), np.nextafter(down, f32(-np.inf))
        out += [up, down]
    return np.concatenate(out)


def _axis(rng, n, lo, hi, c, o):
    k = np.arange(np.floor((lo - o) / c) - 1, np.ceil((hi - o) / c) + 2)
    if len(k) > 400:
        k = rng.choice(k, 400, replace=False)
    edge = [lo, hi, lo + RADIUS, hi - RADIUS, lo - 0.3, hi + 0.3, 0.0]
    v = np.concatenate([_near(f32(o) + k.astype(f32) * f32(c)), _near(edge), rng.uniform(lo, hi, 200).astype(f32)])
    return rng.choice(v, n).astype(f32)


def _faces(x, lo, hi, fl, fh):
    lo, hi, r = f32(lo), f32(hi), f32(RADIUS)
    x, alive = x.copy(), np.ones(len(x), bool)
    last = f32(hi - r) if fh == "C" else hi
    over = x > last
    x[over] = last if fh == "C" else hi + (hi - x[over]) if fh == "R" else x[over]
    alive &= ~over | (fh != "A")
    first = f32(lo + r) if fl == "C" else lo
    under = x < first
    x[under] = first if fl == "C" else lo + (lo - x[under]) if fl == "R" else x[under]
    alive &= ~under | (fl != "A")
    return x, alive


@pytest.mark.parametrize("name", list(CASES))
def test_cells_and_faces(smd, gpu, name):
    faces, cell, origin, bits = CASES[name]
    n = 20011
    rng = np.random.default_rng(len(name))
    spec = configs.make_spec(
        D=[0.0, 0.0, 1.0, 0.5], dt=1e-3, reactions=[dict(order=2, reactants=[1, 2], products=[3], rate=1e-3)],
        box_lo=LO, box_hi=HI, faces=[KIND[c] for c in faces], grid_bits=bits, cell_size=cell, origin=origin,
        num_streams=2500, seed=3, particle_radius=RADIUS)
    pos = np.ones((n, 4), f32)
    for d in range(3):
        pos[:, d] = _axis(rng, n, LO[d], HI[d], cell[d], origin[d])
    e = smd.Engine(0)
    e.add_replica(spec, pos, np.full(n, 1, np.int32))
    e.finalize()
    print(f"cells and faces {name}", flush=True)
    got = e.debug_stage(2, n)
    e.close()
    key, alive = np.zeros(n, np.int64), np.ones(n, bool)
    for d, shift in enumerate((0, bits[0], bits[0] + bits[1])):
        x, ok = _faces(pos[:, d], LO[d], HI[d], faces[2 * d], faces[2 * d + 1])
        alive &= ok
        assert np.array_equal(got["pos"][:, d].view(np.uint32), x.view(np.uint32))
        g = np.floor((x - f32(origin[d])) / f32(cell[d])).astype(np.int64)
        key += (g & ((1 << bits[d]) - 1)) << shift
    key[~alive] = 1 << sum(bits)
    assert got["n_live"] == alive.sum()
    have = np.empty(n, np.int64)
    have[got["vals"]] = got["keys"]
    assert np.array_equal(have, key)
