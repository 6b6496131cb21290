"""Device-noise steps of the normal-mode propagator in two kernels (steps.hpp),
against the persistent batch kernel: beads around the matrix cores' blocks of 16
(65 takes the four-kernel form), columns around tiles of 16, pairs by tiles and
by groups.  Six steps agree to rounding, as in test_gpu_steps.
"""
import pytest

from helpers import MEV
from test_gpu_steps import TRAP, batch_run, close, context_run, system

pytestmark = pytest.mark.gpu

CASES = [(N, P, 3, dict(TRAP)) for N, P in ((1, 2), (15, 3), (16, 8), (17, 15), (33, 16), (5, 17), (20, 33), (18, 48),
                                            (9, 63), (40, 64), (10, 65), (7, 1))]
CASES += [(101, 24, 2, dict(TRAP, int_kind="dipole", int_strength=0.5)), (30, 12, 1, dict(TRAP, int_kind="harmonic",
                                                                                         int_omega=1.0 * MEV)),
          (70, 32, 3, dict(nmthermostat=1)), (200, 6, 3, {}), (64, 20, 3, dict(fixcom=0)),
          (21, 10, 3, dict(TRAP, thermostat="none")), (21, 10, 2, dict(TRAP, thermostat="none", fixcom=0))]


@pytest.mark.parametrize("N,P,D,kw", CASES)
def test_normal_mode_steps(N, P, D, kw):
    kw, x, p = system(N, P, D, 3 * N + P, **dict(kw, bosonic=0, propagator="normal_modes"))
    got = context_run(kw, x, p, (6,))
    close(got, context_run(kw, x, p, (1, 2, 3)), "N=%d P=%d calls" % (N, P))
    ref, _ = batch_run([(kw, x, p)], (6,), (256, 1))
    close(got, ref[0], "N=%d P=%d persistent" % (N, P))
