"""Pair forces of a single system by groups of 128 particles (slice_groups.hpp),
used above 128 particles: sizes around tiles of 64 and groups of 128, odd and
even numbers of groups, one to four parts per group (few beads take more),
every pair kind, image rule and dimension.

Each pair force is within a few 1e-14 of the oracle's and a sum of N of them is
rounded N times, so forces agree to 1e-11 of a bead's largest; a step adds
rounding of x and p alone (1e-12 over three steps) and f follows x.
"""
import numpy as np
import pytest

import oracle as O
import pimdb_amd as G
from helpers import AMU, ANGSTROM, FS, KELVIN, MEV, per_bead_err, rel_err

pytestmark = pytest.mark.gpu


def system(N, P, D, kind, **kw):
    rng = np.random.default_rng(7 * N + P + D)
    side = int(np.ceil(N ** (1.0 / D)))
    a = 3.6 * ANGSTROM
    L = side * a
    sites = np.indices((side,) * D).reshape(D, -1).T[rng.permutation(side ** D)[:N]]
    x = ((sites + 0.5) * a - 0.5 * L + rng.uniform(-0.4, 0.4, size=(N, D)))[None] + rng.normal(0.0, 0.3, size=(P, N, D))
    base = dict(natoms=N, nbeads=P, ndim=D, mass=4.0026 * AMU, temperature=1.5 * KELVIN, dt=0.5 * FS,
                gamma=1.0 / (50.0 * FS), bosonic=0, pbc=1, size=L, ext_kind="free", int_kind=kind, cutoff=0.5 * L,
                propagator="cartesian", thermostat="langevin", nmthermostat=0, fixcom=1, seed=31)
    if kind == "harmonic":
        base["int_omega"] = 0.1 * MEV
    if kind == "dipole":
        base["int_strength"] = 0.5
    return dict(base, **kw), x, rng.normal(0.0, 1.0, size=x.shape)


TRAP = dict(pbc=0, cutoff=-1.0, ext_kind="harmonic", ext_omega=3.0 * MEV)
CASES = [(N, 2, 3, "aziz", {}) for N in (128, 129, 191, 193, 256, 257, 320, 385, 513, 650, 1025)]
CASES += [(300, 40, 3, "aziz", {}), (300, 130, 2, "aziz", {}), (200, 3, 1, "harmonic", {}), (200, 3, 2, "dipole", {}),
          (270, 4, 3, "dipole", dict(cutoff=-1.0)), (260, 3, 3, "harmonic", dict(TRAP)), (390, 4, 2, "dipole", dict(TRAP)),
          (140, 4, 3, "aziz", dict(TRAP)), (300, 4, 3, "aziz", dict(bosonic=1)),
          (300, 4, 3, "aziz", dict(propagator="normal_modes")),
          (150, 6, 3, "aziz", dict(thermostat="nose_hoover_np", bosonic=1)),
          (150, 1, 3, "aziz", {}), (2100, 1, 3, "aziz", {})]


@pytest.mark.parametrize("N,P,D,kind,kw", CASES)
def test_forces(N, P, D, kind, kw):
    kw, x, p = system(N, P, D, kind, **kw)
    ctx = G.Context(G.make_params(**kw))
    ctx.set_state(x, p)
    ctx.forces()
    f = ctx.state()[2]
    ctx.close()
    e = per_bead_err(f, O.update_forces(O.make_params(**kw), x))
    print("N=%d P=%d %s %.2e" % (N, P, kind, e), flush=True)
    assert e < 1e-11


@pytest.mark.parametrize("N,P,D,kind,kw", [c for c in CASES if c[0] < 700 and "thermostat" not in c[4]])
def test_steps(N, P, D, kind, kw):
    """Three device-noise steps against the persistent batch kernel (pair forces by slices)."""
    kw, x, p = system(N, P, D, kind, **kw)
    ctx = G.Context(G.make_params(**kw))
    ctx.set_state(x, p)
    ctx.forces()
    ctx.step(2)
    ctx.step(1)
    got = ctx.state()
    ctx.close()
    b = G.Batch([G.make_params(**kw)])
    b.configure(256, 1)
    b.set_state(0, x, p)
    b.forces()
    b.step(3)
    ref = b.state(0)
    b.close()
    for name, u, v, tol in zip("xpf", got, ref, (1e-12, 1e-11, 1e-10)):
        e = rel_err(u, v)
        print("N=%d P=%d %s %s %.2e" % (N, P, kind, name, e), flush=True)
        assert e < tol
