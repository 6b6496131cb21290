"""The autograd harness on tensors whose memory does not hold their values:
lazily negated views (the imaginary part of a conjugate) as beads and as the
incoming gradient, and zeros without memory.  Against the same call on ordinary
tensors, whose kernels and inputs are the same: equal bits.
"""
import pytest

torch = pytest.importorskip("torch")

from test_gpu_autograd_saved import plan_for, ring  # noqa: E402

pytestmark = pytest.mark.gpu


def negated(t):
    """t as a view of the memory of -t with the negative bit."""
    z = torch.complex(torch.zeros_like(t), -t)
    v = torch.imag(z.conj())
    assert v.is_neg() and torch.equal(v, t)
    return v


def both(x1, xP, g, plan):
    from pimdb_amd.autograd import exchange_potential
    x1, xP = x1.detach().requires_grad_(), xP.detach().requires_grad_()
    vb = exchange_potential(x1, xP, plan)
    return (vb.detach(),) + torch.autograd.grad(vb, (x1, xP), grad_outputs=g)


@pytest.mark.parametrize("N,D", [(5, 3), (70, 2)])
def test_negated_views(N, D):
    x1, xP = ring(N, D, N)
    plan = plan_for(N, D)
    g = torch.tensor(1.7, dtype=torch.float64, device="cuda")
    want = both(x1, xP, g, plan)
    for u, v, w in ((negated(x1), xP, g), (x1, negated(xP), g), (negated(x1), negated(xP), g), (x1, xP, negated(g))):
        for a, b in zip(both(u, v, w, plan), want):
            assert torch.equal(a, b)
    plan.close()


def test_zeros_without_memory():
    x1, xP = ring(6, 3, 4)
    plan = plan_for(6, 3)
    zeros = torch._efficientzerotensor((6, 3), dtype=torch.float64, device="cuda")
    one = torch.ones((), dtype=torch.float64, device="cuda")
    for a, b in zip(both(zeros, xP, one, plan), both(torch.zeros_like(x1), xP, one, plan)):
        assert torch.equal(a, b)
    _, d1, dP = both(x1, xP, torch._efficientzerotensor((), dtype=torch.float64, device="cuda"), plan)
    assert torch.count_nonzero(d1) == 0 and torch.count_nonzero(dP) == 0
    plan.close()
