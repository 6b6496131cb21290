"""Batches of gradients at once through the autograd harness
(is_grads_batched, a vectorized jacobian) against one call for each: the
product with the incoming gradient is one rounding in either, 4 ulp.
"""
import pytest

torch = pytest.importorskip("torch")

from test_gpu_autograd_saved import agree, plan_for, ring  # noqa: E402

pytestmark = pytest.mark.gpu


def test_batched_gradients():
    from pimdb_amd.autograd import exchange_potential
    x1, xP = ring(11, 3, 9)
    plan = plan_for(11, 3)
    x1.requires_grad_()
    xP.requires_grad_()
    vb = exchange_potential(x1, xP, plan)
    w = torch.tensor([1.0, -2.5, 0.0], dtype=torch.float64, device="cuda")
    got = torch.autograd.grad(vb, (x1, xP), grad_outputs=w, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        for a, b in zip(got, torch.autograd.grad(vb, (x1, xP), grad_outputs=w[i], retain_graph=True)):
            agree(a[i], b)
    plan.close()


def test_vectorized_jacobian():
    from pimdb_amd.autograd import exchange_potential
    x1, xP = ring(9, 2, 3)
    plan = plan_for(9, 2)

    def pair(u):
        return torch.stack([exchange_potential(u, xP, plan), exchange_potential(2.0 * u, xP, plan)])

    got, want = (torch.autograd.functional.jacobian(pair, x1, vectorize=v) for v in (True, False))
    assert got.shape == (2, 9, 2)
    agree(got, want)
    plan.close()
