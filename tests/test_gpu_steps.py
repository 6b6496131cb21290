"""Runs of device-noise steps of a single system, where consecutive steps share
one integration kernel, against the same steps taken one call at a time, where
each half step is a kernel of its own (the path the oracle tests cover).

The two evaluate the same sums in another order, so they agree to rounding:
each step adds a few ulp of each term to x and p (the combined update
c1^2 (p + h f) + H - shift + h f against four separate ones), and the forces
follow x through the springs, whose ulp-level change of x is at most
k / (typical force / x) ~ 1e2 times larger relative to f.  Over 6 steps that is
below 1e-11 of each array's norm at these sizes.
"""
import numpy as np
import pytest

import pimdb_amd as G
from helpers import AMU, ANGSTROM, FS, KELVIN, MEV, rel_err

pytestmark = pytest.mark.gpu


def system(N, P, D, seed, **kw):
    rng = np.random.default_rng(seed)
    L = (N / 0.02186) ** (1.0 / 3.0) * ANGSTROM
    side = int(np.ceil(N ** (1.0 / D)))
    sites = np.indices((side,) * D).reshape(D, -1).T[rng.permutation(side ** D)[:N]]
    centres = ((sites + 0.5) / side - 0.5) * L + rng.uniform(-0.3, 0.3, size=(N, D))
    x = centres[None] + rng.normal(0.0, 0.3, size=(P, N, D))
    p = rng.normal(0.2, 1.0, size=x.shape)
    base = dict(natoms=N, nbeads=P, ndim=D, mass=4.0026 * AMU, temperature=1.5 * KELVIN, dt=0.5 * FS,
                gamma=1.0 / (50.0 * FS), bosonic=1, pbc=1, size=L, ext_kind="free", int_kind="aziz",
                cutoff=0.5 * L, propagator="cartesian", thermostat="langevin", nmthermostat=0, fixcom=1, seed=99)
    return dict(base, **kw), x, p


TRAP = dict(pbc=0, ext_kind="harmonic", ext_omega=3.0 * MEV, int_kind="free", cutoff=-1.0)
CASES = [
    (4, 32, 3, dict(TRAP)),
    (1, 8, 3, dict(TRAP)),
    (13, 2, 2, dict(TRAP, int_kind="dipole", int_strength=0.5)),
    (13, 3, 2, dict(TRAP, int_kind="dipole", int_strength=0.5, nmthermostat=1)),
    (65, 5, 1, dict(TRAP, int_kind="harmonic", int_omega=1.0 * MEV, fixcom=0)),
    (64, 16, 3, dict(nmthermostat=1)),
    (65, 17, 3, dict(nmthermostat=1, fixcom=0)),
    (129, 64, 3, dict(nmthermostat=1)),
    (30, 65, 3, dict(nmthermostat=1)),          # modes beyond the matrix-core form
    (70, 6, 3, dict(thermostat="none")),
    (70, 6, 3, dict(thermostat="none", fixcom=0, bosonic=0)),
    (40, 12, 3, dict(bosonic=0)),
    (40, 1, 3, dict(bosonic=1)),                # one bead: no exchange
    (33, 7, 3, dict(pbc=1, ext_kind="cosine", ext_amplitude=1e-4, ext_phase=0.3)),
    (33, 7, 2, dict(TRAP, ext_kind="double_well", ext_strength=1e-9, ext_location=4.0)),
    (9, 8, 3, dict(TRAP, thermostat="nose_hoover_np", fixcom=0)),
    (21, 10, 3, dict(TRAP, bosonic=0, propagator="normal_modes")),
]


@pytest.mark.parametrize("N,P,D,kw", CASES)
def test_steps_together_and_apart(N, P, D, kw):
    kw, x, p = system(N, P, D, 5 * N + P, **kw)
    out = []
    for split in ((6,), (1,) * 6, (2, 3, 1)):
        ctx = G.Context(G.make_params(**kw))
        ctx.set_state(x, p)
        ctx.forces()
        for n in split:
            ctx.step(n)
        out.append(ctx.state())
        ctx.close()
    for other in out[1:]:
        for name, a, b in zip("xpf", out[0], other):
            e = rel_err(a, b)
            print("N=%d P=%d %s %.2e" % (N, P, name, e), flush=True)
            assert e < 1e-11
