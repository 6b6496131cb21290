"""Device-noise steps of a single system (two kernels a step, steps.hpp) and of
few batched replicas (the same two kernels over many replicas), against the
persistent batch kernel, which integrates every half step by itself.

The forms evaluate the same sums in another order, so they agree to rounding:
a step adds a few ulp of each term to x and p, and f follows x through the
springs and, on beads 1 and P, through the exchange probabilities, whose
absolute error in double is about beta~ eps |V| (1e-13 at these sizes, times
link lengths up to 1e2 of the ring's own displacements).  Over 6 steps: x and
p below 1e-11 and f below 1e-10 of each array's norm.
"""
import numpy as np
import pytest

import pimdb_amd as G
from helpers import AMU, ANGSTROM, FS, KELVIN, MEV, rel_err

pytestmark = pytest.mark.gpu


def system(N, P, D, state, **kw):
    rng = np.random.default_rng(state)
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


def context_run(kw, x, p, split):
    ctx = G.Context(G.make_params(**kw))
    ctx.set_state(x, p)
    ctx.forces()
    for n in split:
        ctx.step(n)
    s = ctx.state()
    ctx.close()
    return s


def batch_run(systems, split, shape=None):
    b = G.Batch([G.make_params(**kw) for kw, _, _ in systems])
    if shape:
        b.configure(*shape)
    for r, (_, x, p) in enumerate(systems):
        b.set_state(r, x, p)
    b.forces()
    f0 = [b.state(r)[2] for r in range(len(systems))]
    for n in split:
        b.step(n)
    out = [b.state(r) for r in range(len(systems))]
    b.close()
    return out, f0


def close(a, b, label):
    for name, u, v, tol in zip("xpf", a, b, (1e-11, 1e-11, 1e-10)):
        e = rel_err(u, v)
        print("%s %s %.2e" % (label, name, e), flush=True)
        assert e < tol


@pytest.mark.parametrize("N,P,D,kw", CASES)
def test_single_system(N, P, D, kw):
    kw, x, p = system(N, P, D, 5 * N + P, **kw)
    together = context_run(kw, x, p, (6,))
    close(together, context_run(kw, x, p, (1, 2, 3)), "N=%d P=%d calls" % (N, P))
    ref, _ = batch_run([(kw, x, p)], (6,), (256, 1))
    close(together, ref[0], "N=%d P=%d persistent" % (N, P))


# mixes of replicas of one dimension and interaction: few beads (a slice on
# four waves), enough for two and for one wave a slice, ragged sizes
MIXES = {
    "helium": [(5, 2, {}), (64, 3, {}), (65, 16, dict(nmthermostat=1)), (130, 5, dict(fixcom=0)), (40, 1, {}),
               (33, 64, dict(nmthermostat=1, fixcom=0)), (70, 6, dict(thermostat="none")), (257, 4, dict(bosonic=0))],
    "dipole": [(N, P, dict(TRAP, int_kind="dipole", int_strength=0.5, nmthermostat=m))
               for N, P, m in ((1, 4, 0), (7, 33, 1), (64, 8, 0), (100, 12, 1), (129, 2, 0))],
    "many": [(8 + r % 5, 64, dict(TRAP, int_kind="harmonic", int_omega=1.0 * MEV, bosonic=r % 2)) for r in range(40)],
    "free": [(9, 7, dict(TRAP)), (66, 4, dict(TRAP, ext_kind="free"))],
}


@pytest.mark.parametrize("mix", sorted(MIXES))
@pytest.mark.parametrize("D", [2, 3])
def test_few_replicas(mix, D):
    systems = [system(N, P, D, 11 * r + N, **dict(kw, seed=50 + r)) for r, (N, P, kw) in enumerate(MIXES[mix])]
    ref, f0 = batch_run(systems, (6,), (1024, 256))
    for split in ((6,), (1, 4, 1)):
        got, g0 = batch_run(systems, split)
        for r in range(len(systems)):
            assert rel_err(g0[r], f0[r]) < 1e-11
            close(got[r], ref[r], "%s %d" % (mix, r))


def test_slices_beyond_lds():
    """A slice whose four force arrays exceed a workgroup's LDS (D=3: N > 1638) accumulates in device memory."""
    systems = [system(1700, 2, 3, 3, bosonic=0), system(30, 4, 3, 4)]
    ref, f0 = batch_run(systems, (2,), (1024, 256))
    got, g0 = batch_run(systems, (2,))
    for r in range(2):
        assert rel_err(g0[r], f0[r]) < 1e-11
        close(got[r], ref[r], "large %d" % r)


def test_forms_alternated():
    """The two-kernel form, then a launch shape (the persistent kernel with its owed half step), then the autotuner, on
    one batch: the trajectory is that of one form."""
    systems = [system(N, P, 3, N, nmthermostat=m, seed=N) for N, P, m in ((20, 8, 1), (48, 16, 0), (70, 4, 1))]
    ref, _ = batch_run(systems, (9,), (512, 256))
    b = G.Batch([G.make_params(**kw) for kw, _, _ in systems])
    for r, (_, x, p) in enumerate(systems):
        b.set_state(r, x, p)
    b.forces()
    b.step(2)
    b.configure(1024, 3)
    b.step(2)
    b.autotune(1)
    b.step(2)
    b.configure(256, 3)
    b.step(1)
    b.autotune(2)
    b.step(2)
    for r in range(3):
        close(b.state(r), ref[r], "alternated %d" % r)
    b.close()
