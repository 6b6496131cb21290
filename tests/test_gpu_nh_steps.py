"""Nose-Hoover steps of a single system around the forces in one kernel
(nh_steps.hpp) against the persistent batch kernel: each kind of chain, with
and without zeroMomentum (one workgroup for the system or one per bead),
exchange forces inside (N <= 64) and beside it, chains of three, four and six
components, and systems too large for one workgroup.  Six steps agree to
rounding, as in test_gpu_steps.
"""
import pytest

from helpers import MEV
from test_gpu_steps import TRAP, batch_run, close, context_run, system

pytestmark = pytest.mark.gpu

KINDS = ["nose_hoover", "nose_hoover_np", "nose_hoover_np_dim"]
CASES = [(N, P, D, dict(TRAP, fixcom=f, bosonic=b)) for N, P, D, f, b in
         ((8, 16, 3, 0, 1), (8, 16, 3, 1, 1), (1, 4, 3, 1, 1), (64, 5, 2, 1, 1), (65, 4, 3, 1, 1), (65, 4, 3, 0, 1),
          (20, 1, 3, 1, 0), (33, 64, 1, 1, 0), (40, 64, 3, 1, 1), (150, 3, 3, 0, 0))]
CASES += [(30, 4, 3, dict(TRAP, nchains=3)), (30, 4, 3, dict(TRAP, nchains=6, fixcom=0)),
          (140, 2, 3, dict(fixcom=1)), (13, 6, 2, dict(TRAP, int_kind="dipole", int_strength=0.5)),
          (30, 40, 3, dict(TRAP, int_kind="harmonic", int_omega=1.0 * MEV))]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("N,P,D,kw", CASES)
def test_nose_hoover_steps(N, P, D, kw, kind):
    kw, x, p = system(N, P, D, 3 * N + P, **dict(kw, thermostat=kind))
    got = context_run(kw, x, p, (6,))
    close(got, context_run(kw, x, p, (1, 2, 3)), "N=%d P=%d calls" % (N, P))
    ref, _ = batch_run([(kw, x, p)], (6,), (256, 1))
    close(got, ref[0], "N=%d P=%d persistent" % (N, P))
