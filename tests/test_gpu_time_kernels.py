"""Kernel times of a single system: the forces that are timed are those a step
computes, so they take no longer than the step that contains them (up to the
separate launch that completes them and the clock's spread: 1.3), and the state
is left as it was.  The largest case is one where a step evaluates each pair
once and the other form every ordered pair (1.7 times as long as the step).
"""
import numpy as np
import pytest

import pimdb_amd as G
from test_gpu_steps import TRAP, system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,P,D,kw", [(1000, 4, 3, dict(bosonic=0)), (500, 16, 3, dict(bosonic=1)), (300, 8, 2, dict(TRAP, int_kind="dipole", int_strength=0.5)),
                                      (60, 8, 3, dict(bosonic=0)), (200, 6, 3, dict(bosonic=0, propagator="normal_modes"))])
def test_forces_within_a_step(N, P, D, kw):
    kw, x, p = system(N, P, D, N, **kw)
    ctx = G.Context(G.make_params(**kw))
    ctx.set_state(x, p)
    ctx.forces()
    want = ctx.state()
    forces, exchange, _ = ctx.time_kernels(reps=20, step=False)
    for u, v in zip(ctx.state(), want):
        assert np.array_equal(u, v)
    assert (exchange > 0.0) == bool(kw["bosonic"])
    step = min(ctx.time_kernels(reps=20, forces=False, exchange=False)[2] for _ in range(3))
    print("N=%d forces %.1f step %.1f us" % (N, 1e3 * forces, 1e3 * step), flush=True)
    assert 0.0 < forces < 1.3 * step
    ctx.close()
