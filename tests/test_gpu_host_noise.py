"""Steps with noise from the host: thousands of Langevin O-steps in Cartesian
coordinates, whose kernel stages a tile of momentum columns in LDS and updates
it by other threads than those that staged it.

Two runs from the same state with the same noise perform the same operations
in the same order, so they end with the same bits.
"""
import numpy as np
import pytest

import pimdb_amd as G
from helpers import AMU, KELVIN, MEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,P,bosonic", [(4, 32, 0), (9, 64, 0), (70, 3, 0), (5, 16, 1), (2, 300, 0)])
def test_same_noise_same_bits(N, P, bosonic):
    kw = dict(natoms=N, nbeads=P, ndim=3, mass=4.0026 * AMU, temperature=1.5 * KELVIN, dt=20.0, gamma=5e-4,
              bosonic=bosonic, pbc=0, size=60.0, ext_kind="harmonic", ext_omega=3.0 * MEV, int_kind="free", cutoff=-1.0,
              propagator="cartesian", thermostat="langevin", nmthermostat=0, fixcom=1, seed=5)
    rng = np.random.default_rng(N + P)
    x, p = rng.normal(0.0, 3.0, size=(P, N, 3)), rng.normal(0.0, 3.0, size=(P, N, 3))
    noise = [rng.normal(size=(500, 2, P, N, 3)) for _ in range(2)]
    ends = []
    for _ in range(2):
        ctx = G.Context(G.make_params(**kw))
        ctx.set_state(x, p)
        ctx.forces()
        for part in 4 * noise:
            ctx.step(len(part), part)
        ends.append(ctx.state())
        ctx.close()
    for name, u, v in zip("xpf", *ends):
        assert np.array_equal(u, v), name
