"""Steps of a handful of particles in one launch (small_steps.hpp: up to 8 with
exchange, 16 without) against the persistent batch kernel: one particle, the
most particles and one more, one to 64 beads (odd ones among them), the largest
state of one workgroup, each pair kind and external potential, more steps than a
launch takes.

Six steps agree to rounding, as in test_gpu_steps.  The long run compares the
forms over 520 steps, a trajectory without close pairs that contracts with the
friction: 1e-9.
"""
import pytest

from helpers import MEV, rel_err
from test_gpu_steps import TRAP, batch_run, close, context_run, system

pytestmark = pytest.mark.gpu

CASES = [(N, P, D, dict(TRAP, nmthermostat=m, fixcom=f, bosonic=b)) for N, P, D, m, f, b in
         ((4, 32, 3, 0, 1, 1), (1, 2, 3, 0, 1, 1), (1, 1, 1, 0, 0, 0), (2, 2, 3, 1, 1, 1), (8, 64, 3, 0, 1, 1),
          (8, 64, 3, 1, 0, 1), (9, 8, 3, 0, 1, 1), (7, 7, 1, 1, 0, 1), (9, 33, 3, 1, 1, 0), (3, 3, 2, 0, 0, 1),
          (16, 32, 3, 1, 1, 0), (16, 48, 2, 0, 1, 0), (17, 8, 3, 0, 1, 0), (5, 65, 3, 0, 1, 1))]
CASES += [(8, 5, 3, dict(TRAP, int_kind="harmonic", int_omega=1.0 * MEV)),
          (16, 8, 2, dict(TRAP, int_kind="dipole", int_strength=0.5, nmthermostat=1, bosonic=0)),
          (8, 9, 3, dict(int_kind="dipole", int_strength=0.5)),
          (12, 4, 3, dict(int_kind="dipole", int_strength=0.5, cutoff=-1.0, bosonic=0)),
          (7, 6, 3, dict(TRAP, thermostat="none")), (7, 6, 3, dict(TRAP, thermostat="none", fixcom=0)),
          (8, 7, 3, dict(pbc=1, int_kind="free", ext_kind="cosine", ext_amplitude=1e-4, ext_phase=0.3)),
          (8, 7, 2, dict(TRAP, ext_kind="double_well", ext_strength=1e-9, ext_location=4.0))]


@pytest.mark.parametrize("N,P,D,kw", CASES)
def test_small_steps(N, P, D, kw):
    kw, x, p = system(N, P, D, 5 * N + P, **kw)
    got = context_run(kw, x, p, (6,))
    close(got, context_run(kw, x, p, (1, 2, 3)), "N=%d P=%d calls" % (N, P))
    ref, _ = batch_run([(kw, x, p)], (6,), (256, 1))
    close(got, ref[0], "N=%d P=%d persistent" % (N, P))


def test_more_steps_than_a_launch():
    kw, x, p = system(5, 8, 3, 2, **dict(TRAP, gamma=0.02))
    got = context_run(kw, x, p, (520,))
    ref, _ = batch_run([(kw, x, p)], (520,), (256, 1))
    for u, v in zip(got, ref[0]):
        assert rel_err(u, v) < 1e-9
