"""Several launches whose workgroups wait for each other at once: batches with
more blocks of rings than the card has places, and contexts of long rings,
stepped from threads of their own.  Each ends with the bits that it has alone.
"""
import threading

import numpy as np
import pytest

import pimdb_amd as G
from test_gpu_exchanging_rings import ring

pytestmark = pytest.mark.gpu


def batch(N, R, seed):
    kw, x = ring(N, 4, 1)
    b = G.Batch([G.make_params(**dict(kw, seed=seed + r)) for r in range(R)])
    for r in range(R):
        b.set_state(r, x, 0.0 * x)

    def run():
        b.forces()
        for _ in range(3):
            b.step(4)
        return [v for r in range(0, R, 17) for v in b.state(r)]
    return b, run


def context(N, seed):
    kw, x = ring(N, 4, 1)
    c = G.Context(G.make_params(**dict(kw, seed=seed)))
    c.set_state(x, 0.0 * x)

    def run():
        c.forces()
        out = []
        for _ in range(3):
            c.step(4)
            out.append(c.observables())
        return out + list(c.state())
    return c, run


def test_threads():
    makes = [lambda: batch(130, 140, 1), lambda: batch(200, 110, 1000), lambda: context(1000, 5), lambda: context(1900, 6)]
    want = []
    for make in makes:
        o, run = make()
        want.append(run())
        o.close()
    objs = [make() for make in makes]
    got, errors = [None] * len(objs), []

    def work(i):
        try:
            got[i] = objs[i][1]()
        except Exception as e:   # (reported below)
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(objs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for o, _ in objs:
        o.close()
    assert not errors, errors
    for u, v in zip(got, want):
        for a, b in zip(u, v):
            assert np.array_equal(a, b)
