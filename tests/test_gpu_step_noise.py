"""The deviates of the device noise of single systems: with friction so high
that c1 = 0, a free particle's momentum after a step is c2 times the deviate of
its last O-step, the same bits in every single-system form, whose draws have
the same keys and the same functions (one dimension and one bead: the key is the
particle).  The reference is the form of slices beyond a workgroup's LDS, which
draws in its O-step kernel.
"""
import numpy as np
import pytest

from test_gpu_steps import context_run, system

pytestmark = pytest.mark.gpu


def momenta(N, **kw):
    kw, x, p = system(70, 1, 1, 1, pbc=0, int_kind="free", cutoff=-1.0, bosonic=0, fixcom=0, **kw)
    kw.update(natoms=N, gamma=1e4 / kw["dt"])
    return context_run(kw, np.zeros((1, N, 1)), np.ones((1, N, 1)), (3,))[1][0, :, 0]


def test_same_deviates():
    ref = momenta(21000)
    for N, kw in ((16, {}), (3000, {}), (3000, dict(propagator="normal_modes"))):
        assert np.array_equal(momenta(N, **kw), ref[:N]), (N, kw)
