"""Potential energies at the ends of the range of a distance: coincident
particles (a dipole pair's energy is infinite, a harmonic one's 0, an Aziz one's
not a number, as its attraction is infinity times 0) and one so far away that the
distance's square overflows (it adds nothing to the dipole energy and the virial
of the others, 1e-13 of which is allowed for the order of the sum).
"""
import numpy as np
import pytest

import pimdb_amd as G
from test_gpu_steps import system

pytestmark = pytest.mark.gpu


def potential(N, P, D, x, **kw):
    kw, _, p = system(N, P, D, N, pbc=0, cutoff=-1.0, bosonic=0, **kw)
    ctx = G.Context(G.make_params(**kw))
    ctx.set_state(x, p)
    v = ctx.observables()
    ctx.close()
    return v[1], v[4]


@pytest.mark.parametrize("N,P,D", [(4, 3, 3), (70, 2, 2), (200, 2, 3)])
def test_extremes(N, P, D):
    _, x, _ = system(N, P, D, N)
    dipole = dict(int_kind="dipole", int_strength=0.5)
    far = x.copy()
    far[:, -1, 0] = 1e160
    d = far[:, :-1, None] - far[:, None, :-1]
    r = np.sqrt((d * d).sum(-1))[:, ~np.eye(N - 1, dtype=bool)]
    want = 0.5 * (0.5 / r ** 3).sum() / P
    pot, vir = potential(N, P, D, far, **dipole)
    assert abs(pot - want) <= 1e-13 * want
    # (r dV/dr = -3 V of a pair, half of it by either particle's forces: the sum over ordered i < j alone is taken)
    g = -1.5 / np.where(np.eye(N - 1, dtype=bool), 1.0, np.sqrt((d * d).sum(-1))) ** 5 * np.triu(np.ones((N - 1, N - 1)), 1)
    wantv = 0.5 * (far[:, :-1, None] * g[..., None] * d).sum() / P
    scale = 0.5 * np.abs(far[:, :-1, None] * g[..., None] * d).sum() / P
    assert abs(vir - wantv) <= 1e-13 * scale
    same = x.copy()
    same[0, 1] = same[0, 0]
    assert potential(N, P, D, same, **dipole)[0] == np.inf
    assert np.isnan(potential(N, P, D, same, int_kind="aziz")[0])
    same[:] = same[:, :1]
    assert potential(N, P, D, same, int_kind="harmonic", int_omega=1e-4)[0] == 0.0
