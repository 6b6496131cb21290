"""torch.autograd harness over the exchange kernels (test harness, not the
driver): the forward kernel computes V_B = V[N] from beads 1 and P
(quadratic_bosonic_exchange.cpp:34-132) and leaves both recursions for the
backward, the hand-written adjoint kernel: -dV_B/dx for both beads (the
exterior spring forces of :159-215 without the interior links).  Tensors are
float64 CUDA tensors of shape (N, D), read with whatever strides they have on
torch's current stream.
"""
import torch

from . import XPlan


class ExchangeVB(torch.autograd.Function):
    """V_B(x1, xP) with its gradient from the adjoint kernel."""

    @staticmethod
    def forward(ctx, x1, xP, plan):
        if not (x1.is_cuda and xP.is_cuda) or x1.dtype != torch.float64 or xP.dtype != torch.float64:
            raise TypeError("ExchangeVB takes float64 CUDA tensors")
        if x1.shape != xP.shape or x1.dim() != 2 or x1.shape != (plan.natoms, plan.ndim):
            raise ValueError("x1 and xP must both have shape (%d, %d)" % (plan.natoms, plan.ndim))
        # the values in memory: a lazily negated view (the imaginary part of a conjugate) holds the opposite ones
        # there, and zeros that autograd makes have no memory at all
        if x1.is_neg() or xP.is_neg() or not (x1.data_ptr() and xP.data_ptr()):
            x1, xP = x1.resolve_neg().clone(), xP.resolve_neg().clone()
        vb = torch.empty((), dtype=torch.float64, device=x1.device)
        saved = torch.empty(plan.saved_doubles, dtype=torch.float64, device=x1.device)
        stream = torch.cuda.current_stream(x1.device).cuda_stream
        plan.forward_saved(x1.data_ptr(), x1.stride(), xP.data_ptr(), xP.stride(), vb.data_ptr(), saved.data_ptr(), stream)
        ctx.plan = plan
        ctx.save_for_backward(saved)
        return vb

    @staticmethod
    def backward(ctx, g):
        (saved,) = ctx.saved_tensors
        plan = ctx.plan
        d1, dP = (torch.empty((plan.natoms, plan.ndim), dtype=torch.float64, device=saved.device) for _ in range(2))
        stream = torch.cuda.current_stream(saved.device).cuda_stream
        # the product with g stays a torch operation where it is to be differentiated itself, and where g's values are
        # not in memory as they are: lazily negated, zeros without memory, or many gradients at once
        # (is_grads_batched)
        scale = None
        if not (torch.is_grad_enabled() or g.is_neg()):
            try:
                scale = g.data_ptr() or None
            except RuntimeError:
                pass
        plan.backward_saved(saved.data_ptr(), scale, d1.data_ptr(), dP.data_ptr(), stream)
        return (d1, dP, None) if scale is not None else (d1 * g, dP * g, None)


def exchange_potential(x1, xP, plan):
    """V_B of beads 1 and P (differentiable in both)."""
    return ExchangeVB.apply(x1, xP, plan)


def make_plan(natoms, ndim, beta_t, spring_k, pbc=False, size=0.0):
    return XPlan(natoms, ndim, beta_t, spring_k, pbc, size)
