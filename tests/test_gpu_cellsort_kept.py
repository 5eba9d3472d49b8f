"""The counting cell sort with keys kept in registers, at the edges of what
they hold (24 vectors of four keys for each of 512 threads): whole and ragged
segments that just fit, ones a vector too long, and segments at odd offsets,
against numpy's stable argsort of the producer's keys, exactly."""
import numpy as np
import pytest

from test_gpu_cellsort import _particles, _spec

pytestmark = pytest.mark.gpu

FULL = 24 * 512 * 4
CASES = {
    "full": [FULL],
    "one_short": [FULL - 1],
    "odd_offset_fits": [3, FULL - 3],
    "odd_offset_a_vector_more": [1, FULL],
    "longer_beside_shorter": [5, 60001, 2049, 16383],
    "vector_edges": [2047, 2, 2048, 1, 2051],
}


@pytest.mark.parametrize("name", list(CASES))
def test_kept_keys_match_argsort(smd, gpu, name):
    rng = np.random.default_rng(5)
    total = sum(CASES[name])
    print(f"kept keys {name}: {total} particles", flush=True)
    reps = []
    for k, n in enumerate(CASES[name]):
        pos, types = _particles(n, 16.0, 16.0, rng)
        reps.append((_spec(smd, max(64, n // 8), (5, 5, 4) if n > 64 else (2, 2, 2), seed=21 + k), pos, types))
    got = []
    for stage in (1, 2):
        e = smd.Engine(0)
        for rep in reps:
            e.add_replica(*rep)
        e.finalize()
        got.append(e.debug_stage(stage, total))
        if stage == 2:
            first, dead = e.debug_first(), e.layout()["total_buckets"]
        e.close()
    keys = got[0]["keys"]
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(got[1]["keys"], keys[order])
    assert np.array_equal(got[1]["vals"], order.astype(np.uint32))
    assert np.array_equal(first[: dead + 1], np.searchsorted(keys[order], np.arange(dead + 1, dtype=np.uint64)))
