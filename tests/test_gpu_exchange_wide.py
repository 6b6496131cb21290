"""The exchange recursions with one workgroup per block of 64 targets, and
the device-memory form of larger rings, against the oracle (tolerances of
test_gpu_exchange.py: 1e-10, E 1e-12).

* Rings around the block edges (one block, an empty last backward block at
  N = 64 k + 1, several blocks) in every dimension with and without periodic
  boundaries, each evaluated twice on one context (the published values are
  put back to empty by the first evaluation).
* Rings whose one-particle cycles are suppressed by e^-300 each (the particles
  come in exchanged pairs), so that every block leaves the range of its
  one-particle gauge and takes the min-plus form.
* A ring above the LDS limit of the block form (D=3: N > 2015), judged against
  the exact exchange in extended precision as test_gpu_large_n.py does.
"""
import numpy as np
import pytest

import oracle as O
import pimdb_amd as G
from helpers import rel_err
from test_gpu_exchange import base_kw, check, run_both
from test_gpu_large_n import context_exchange, ring_args, thermal_ring

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [63, 64, 65, 128, 129, 193, 320])
@pytest.mark.parametrize("D,pbc", [(3, True), (2, False), (1, False)])
def test_block_edges_twice(N, D, pbc):
    rng = np.random.default_rng(7 * N + D)
    x = rng.uniform(-3.0, 3.0, size=(4, N, D))
    kw = base_kw(N, 4, D, pbc, L=6.0)
    g, f, o = run_both(kw, x)
    check(g, f, o, N)
    ctx = G.Context(G.make_params(**kw))
    ctx.set_state(x[::-1].copy())
    ctx.exchange_forward()
    ctx.set_state(x)
    again = ctx.exchange_forward()
    ctx.close()
    for k in ("V", "Vb", "prob"):
        assert np.array_equal(again[k], g[k])


@pytest.mark.parametrize("N", [10, 64, 130, 200])
def test_exchanged_pairs(N):
    P, D = 4, 3
    kw = base_kw(N, P, D, False)
    d = O.derived(O.make_params(**kw))
    a = np.sqrt(2.0 * 300.0 / (d["beta_t"] * d["k"]))   # beta~ k a^2 / 2 = 300
    rng = np.random.default_rng(N)
    x1 = rng.normal(0.0, 0.02 * a, size=(N, D))
    x1[1::2, 0] += a
    xP = x1.copy()
    xP[0::2], xP[1::2] = x1[1::2], x1[0::2]
    x = np.stack([x1, 0.5 * (x1 + xP), 0.5 * (x1 + xP), xP]) + rng.normal(0.0, 0.01 * a, size=(P, N, D))
    g, f, o = run_both(kw, x)
    check(g, f, o, N)


def test_device_memory_ring():
    N, P = 2100, 4
    kw, x = thermal_ring(N, P, 77)
    g, f = context_exchange(kw, x)
    args, _ = ring_args(kw, x)
    o, q = O.exchange(*args), O.exchange_quad(*args)
    assert rel_err(g["V"], q["V"]) <= max(1e-14, rel_err(o["V"], q["V"]))
    assert rel_err(g["Vb"], q["Vb"]) <= max(1e-14, rel_err(o["Vb"], q["Vb"]))
    for k, v in (("f_first", f[0]), ("f_last", f[1])):
        assert rel_err(v, q[k]) <= 1.05 * rel_err(o[k], q[k])
