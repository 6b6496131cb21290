"""The autograd harness's forward and backward pair where its route depends on
the caller: strides, a ring beyond the block form's LDS, positions overwritten
between the passes, and a backward that is differentiated itself.  Against the
plan's forward / vb_grad calls on contiguous SoA copies (the same kernels'
arithmetic: V_B equal, gradients equal up to the product with g, 4 ulp)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

KELVIN, HE4 = 3.1668152e-06, 4.0026 * 1822.8885


def ring(N, D, seed):
    g = torch.Generator().manual_seed(seed)
    x1 = torch.rand(N, D, generator=g, dtype=torch.float64) * 30.0
    return x1.cuda(), (x1 + 0.3 * torch.randn(N, D, generator=g, dtype=torch.float64)).cuda()


def plan_for(N, D):
    from pimdb_amd.autograd import make_plan
    T, P = 1.5 * KELVIN, 16
    return make_plan(N, D, 1.0 / (T * P), HE4 * (P * T) ** 2, True, 30.0)


def reference(plan, x1, xP):
    N, D = x1.shape
    a, b = x1.t().contiguous(), xP.t().contiguous()
    vb = torch.empty(1, dtype=torch.float64, device="cuda")
    grad = torch.empty((2, D, N), dtype=torch.float64, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    plan.forward(a.data_ptr(), b.data_ptr(), vb.data_ptr(), None, None, s)
    plan.vb_grad(a.data_ptr(), b.data_ptr(), grad.data_ptr(), s)
    return vb[0], -grad[0].t(), -grad[1].t()


def agree(a, b):
    assert torch.all((a - b).abs() <= 4 * 2.0 ** -52 * b.abs())


@pytest.mark.parametrize("N,D", [(1, 3), (13, 2), (64, 1), (65, 3), (2050, 3)])
def test_strides_and_overwritten_inputs(N, D):
    from pimdb_amd.autograd import exchange_potential
    x1, xP = ring(N, D, N + D)
    plan = plan_for(N, D)
    vb0, g1, gP = reference(plan, x1, xP)
    wide = torch.zeros(N, 2 * D, dtype=torch.float64, device="cuda")
    views = [(x1.clone(), xP.clone()), (x1.t().contiguous().t(), xP.t().contiguous().t()),
             (wide[:, ::2].copy_(x1), torch.cat([xP, xP], 1)[:, :D])]
    for u, v in views:
        u, v = u.detach().requires_grad_(), v.detach().requires_grad_()
        vb = exchange_potential(u, v, plan)
        assert vb.shape == () and vb.item() == vb0.item()
        with torch.no_grad():
            u.zero_()
            v.zero_()
        (3.0 * vb).backward()
        agree(u.grad, 3.0 * g1)
        agree(v.grad, 3.0 * gP)
    plan.close()


def test_differentiated_backward():
    from pimdb_amd.autograd import exchange_potential
    x1, xP = ring(20, 3, 5)
    plan = plan_for(20, 3)
    _, g1, _ = reference(plan, x1, xP)
    x1.requires_grad_()
    w = torch.ones((), dtype=torch.float64, device="cuda", requires_grad=True)
    (d1,) = torch.autograd.grad(exchange_potential(x1, xP, plan), x1, grad_outputs=w, create_graph=True)
    agree(d1, g1)
    v = torch.randn_like(g1)
    (jv,) = torch.autograd.grad((d1 * v).sum(), w)   # the directional derivative
    assert abs(jv.item() - (g1 * v).sum().item()) <= 1e-12 * (g1 * v).abs().sum().item()
    plan.close()
