"""Rings that exchange strongly: bead P of a particle next to bead 1 of its
successor in a cycle of a given length, so that permutations are favoured by
many e^100 over one-particle cycles and the recursions leave the range of their
scaled form (exchange_wide.hpp), in all blocks or only in some.

Forces against the oracle.  An exchange probability's absolute error is about
beta~ eps |V|, 1e-12 at these sizes, times link energies of the ring's own size:
1e-10 of a bead's largest force.
"""
import numpy as np
import pytest

import oracle as O
import pimdb_amd as G
from helpers import AMU, ANGSTROM, FS, KELVIN, per_bead_err

pytestmark = pytest.mark.gpu


def ring(N, P, cycle, first=0):
    rng = np.random.default_rng(N + cycle)
    a = 3.6 * ANGSTROM
    side = int(np.ceil(N ** (1.0 / 3.0)))
    sites = np.indices((side,) * 3).reshape(3, -1).T[:N]
    L = side * a
    cen = (sites + 0.5) * a - 0.5 * L
    nxt = np.arange(N)
    for s in range(first, N, cycle):
        e = min(N, s + cycle)
        nxt[s:e] = np.roll(np.arange(s, e), -1)
    d = cen[nxt] - cen
    d -= L * np.floor(d / L + 0.5)
    x = cen[None] + (np.arange(P) / P)[:, None, None] * d[None] + rng.normal(0.0, 0.2, size=(P, N, 3))
    kw = dict(natoms=N, nbeads=P, ndim=3, mass=4.0026 * AMU, temperature=1.5 * KELVIN, dt=0.5 * FS, gamma=1.0 / (50.0 * FS),
              bosonic=1, pbc=1, size=L, ext_kind="free", int_kind="free", cutoff=-1.0, propagator="cartesian",
              thermostat="langevin", nmthermostat=0, fixcom=1, seed=7)
    return kw, x


@pytest.mark.parametrize("N,P,cycle,first", [(8, 8, 8, 0), (64, 32, 2, 0), (65, 16, 65, 0), (128, 32, 2, 64), (130, 16, 8, 0),
                                             (200, 32, 50, 100), (300, 16, 300, 0), (300, 32, 2, 0)])
def test_forces_of_exchanging_rings(N, P, cycle, first):
    kw, x = ring(N, P, cycle, first)
    want = O.update_forces(O.make_params(**kw), x)
    ctx = G.Context(G.make_params(**kw))
    b = G.Batch([G.make_params(**kw)] * 2)
    for _ in range(2):   # (again with the published values of the first)
        ctx.set_state(x, 0.0 * x)
        ctx.forces()
        e = per_bead_err(ctx.state()[2], want)
        print("N=%d cycle=%d %.2e" % (N, cycle, e), flush=True)
        assert e < 1e-10
    for r in range(2):
        b.set_state(r, x, 0.0 * x)
    b.forces()
    assert per_bead_err(b.state(1)[2], want) < 1e-10
    ctx.close()
    b.close()
