"""A particle whose position is not finite, in systems with a cutoff: no distance
to it is below the cutoff, so the pair forces of the others are those of the
system without it, to the order of their sums (1e-11 of the bead's largest
force), and its own are not finite.
"""
import numpy as np
import pytest

import pimdb_amd as G
from test_gpu_steps import system

pytestmark = pytest.mark.gpu


def forces(kw, x):
    ctx = G.Context(G.make_params(**kw))
    ctx.set_state(x, np.zeros_like(x))
    ctx.forces()
    f = ctx.state()[2]
    ctx.close()
    return f


@pytest.mark.parametrize("N", [20, 130, 200, 400])
@pytest.mark.parametrize("kw", [dict(bosonic=0), dict(bosonic=0, pbc=0, cutoff=9.0, int_kind="dipole", int_strength=0.5)])
def test_others_unaffected(N, kw):
    kw, x, _ = system(N, 3, 3, N, **kw)
    for j, value in ((0, np.nan), (N // 2, np.inf), (N - 1, np.nan)):
        y = x.copy()
        y[1, j, 1] = value
        got = forces(kw, y)
        keep = np.arange(N) != j
        want = forces(dict(kw, natoms=N - 1), x[:, keep])
        e = np.abs(got[1, keep] - want[1]).max() / np.abs(want[1]).max()   # (in the other beads it takes part)
        assert e <= 1e-11, (j, value, e)
        assert not np.isfinite(got[1, j, 1])
