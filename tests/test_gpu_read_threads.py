"""Several threads read different replicas of one engine at the same time:
each gets its own replica's particles."""
import threading

import numpy as np
import pytest

from gpusmoldyn_amd import configs

pytestmark = pytest.mark.gpu


def test_threads_read_their_replicas(smd, gpu):
    e = smd.Engine(0)
    sizes = [2000 + 611 * k for k in range(8)]
    for k, n in enumerate(sizes):
        spec, pos, types = configs.c1(nA=n // 2, nB=n - n // 2, n_streams=256, seed=40 + k, rng_seed=50 + k)
        e.add_replica(spec, pos, types)
    e.finalize()
    e.step(4)
    want = [e.get(r) for r in range(len(sizes))]
    print("8 threads reading 8 replicas", flush=True)
    wrong = []

    def read(r):
        for _ in range(200):
            p, t = e.get(r)
            if not (np.array_equal(t, want[r][1]) and np.array_equal(p.view(np.uint32), want[r][0].view(np.uint32))):
                wrong.append(r)

    threads = [threading.Thread(target=read, args=(r,)) for r in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    e.close()
    assert not wrong
