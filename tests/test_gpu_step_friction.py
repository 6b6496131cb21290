"""Thousands of Langevin steps of free particles with little friction, whose
momenta keep every step's rounding: the single-system forms and few batched
replicas against the persistent batch kernel, which applies the O-steps one by
one.

c1 = exp(-gamma dt / 2) is taken where c1^2 is farthest from a double.  A step
of either form rounds a momentum at most four times, by up to 2^-53 of it each
way at random: over n steps of two forms a spread of sqrt(8 n / 3) 2^-53, of
which six are allowed (n = 4000: 6.9e-14).  The two factors of a step rounded
into one would add n 2^-54 (2.2e-13), always the same way.
"""
import math
from fractions import Fraction

import numpy as np
import pytest

from test_gpu_steps import batch_run, context_run, system

pytestmark = pytest.mark.gpu

STEPS = 4000


def friction(dt):
    def off(g):
        c = math.exp(-0.5 * g * dt)
        return abs(Fraction(c) ** 2 - Fraction(c * c))
    return max((1e-6 * (1.0 + 0.01 * k) / dt for k in range(100)), key=off)


@pytest.mark.parametrize("N,kw", [(5, {}), (70, {}), (70, dict(propagator="normal_modes"))])
def test_free_particles(N, kw):
    kw, x, p = system(N, 1, 3, N, pbc=0, int_kind="free", cutoff=-1.0, bosonic=0, fixcom=0, **kw)
    kw["gamma"] = friction(kw["dt"])
    p = 1e3 * np.sign(p) * (1.0 + np.abs(p) % 1.0)   # (the noise adds a few percent)
    ref = batch_run([(kw, x, p)], (STEPS,), (256, 1))[0][0][1]
    tol = 6.0 * math.sqrt(8.0 * STEPS / 3.0) * 2.0 ** -53
    runs = [context_run(kw, x, p, (STEPS,))[1]]
    if kw["propagator"] == "cartesian":
        runs.append(batch_run([(kw, x, p)] * 2, (STEPS,))[0][0][1])
    for got in runs:
        e = np.max(np.abs(got - ref) / np.abs(ref))
        print("N=%d %.2e of %.2e" % (N, e, tol), flush=True)
        assert e <= tol
