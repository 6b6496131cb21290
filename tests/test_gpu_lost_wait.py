"""Recovery from a wait between workgroups that ran out: what such a call leaves
(published values of other positions, the flag) is put there from the host and
found as after a kernel; the calls after that agree with an untouched object's,
whose kernels and inputs are the same: equal bits.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")   # (before the library, so that both share a HIP runtime)

import pimdb_amd as G  # noqa: E402
from test_gpu_exchanging_rings import ring  # noqa: E402

pytestmark = pytest.mark.gpu

LOST = 3   # PIMDB_E_HIP


@pytest.mark.parametrize("N,P", [(5, 8), (130, 8), (1000, 4)])
def test_context(N, P):
    kw, x = ring(N, P, 1)
    ends = []
    for touched in (False, True):
        ctx = G.Context(G.make_params(**kw))
        ctx.set_state(x, 0.0 * x)

        def lose():
            if touched:
                assert G.lib().pimdb_test_lost_wait(ctx.h) == LOST

        lose()
        ctx.forces()
        f = ctx.state()[2]
        lose()
        obs = ctx.observables()
        lose()
        ctx.step(3)
        ends.append((f, obs) + ctx.state())
        ctx.close()
    for u, v in zip(*ends):
        assert np.array_equal(u, v)


def test_batch():
    kw, x = ring(200, 8, 1)
    ends = []
    for touched in (False, True):
        b = G.Batch([G.make_params(**kw)] * 3)
        for r in range(3):
            b.set_state(r, x, 0.0 * x)
        if touched:
            assert G.lib().pimdb_batch_test_lost_wait(b.h) == LOST
        b.forces()
        if touched:
            assert G.lib().pimdb_batch_test_lost_wait(b.h) == LOST
        b.step(2)
        ends.append([b.state(r) for r in range(3)])
        b.close()
    for s, t in zip(*ends):
        for u, v in zip(s, t):
            assert np.array_equal(u, v)


def test_plan():
    from pimdb_amd.autograd import exchange_potential
    from test_gpu_autograd_saved import plan_for, ring as beads
    x1, xP = beads(300, 3, 1)
    plan = plan_for(300, 3)
    x1.requires_grad_()
    xP.requires_grad_()

    def once():
        vb = exchange_potential(x1, xP, plan)
        return (vb,) + torch.autograd.grad(vb, (x1, xP))

    want = once()
    assert G.lib().pimdb_xplan_test_lost_wait(plan.h) == LOST
    for a, b in zip(once(), want):
        assert torch.equal(a, b)
    plan.close()
