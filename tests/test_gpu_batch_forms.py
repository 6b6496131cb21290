"""Which form a batch steps in (the persistent kernel or two kernels a step):
the default of batches far on either side of the choice, the waves per slice,
what configure and the autotuner leave, and both forms asked for by name, which
agree to rounding as in test_gpu_steps.  And single systems with a handful of
particles that the one-workgroup form does not take, in their two kernels.
"""
import pytest

import pimdb_amd as G
from test_gpu_steps import MIXES, TRAP, batch_run, close, context_run, system

pytestmark = pytest.mark.gpu


def make(systems):
    b = G.Batch([G.make_params(**kw) for kw, _, _ in systems])
    for r, (_, x, p) in enumerate(systems):
        b.set_state(r, x, p)
    b.forces()
    return b


def few(n=3, **kw):
    return [system(N, 8, 3, N, seed=N, **kw) for N in range(20, 20 + n)]


# waves per slice: enough slices for four, two or one on every SIMD
@pytest.mark.parametrize("systems,waves", [
    ([system(N, P, 3, 11 * r + N, **dict(kw, seed=50 + r)) for r, (N, P, kw) in enumerate(MIXES["helium"])], 4),
    ([system(N, P, 2, 11 * r + N, **dict(kw, seed=50 + r)) for r, (N, P, kw) in enumerate(MIXES["many"])], 1),
    ([system(30, 64, 3, r, seed=r) for r in range(20)], 2),
    ([system(1700, 2, 3, 3, bosonic=0), system(30, 4, 3, 4)], 1)])
def test_default_and_waves(systems, waves):
    b = make(systems)
    assert b.form() == (True, waves)
    b.close()


# (test_gpu_steps compares these with the persistent kernel)
@pytest.mark.parametrize("mix", sorted(MIXES))
@pytest.mark.parametrize("D", [2, 3])
def test_default_of_the_mixes(mix, D):
    b = make([system(N, P, D, 11 * r + N, **dict(kw, seed=50 + r)) for r, (N, P, kw) in enumerate(MIXES[mix])])
    assert b.form()[0]
    b.close()


# hundreds of rings of several blocks with few beads
@pytest.mark.parametrize("N,P,D,R", [(180, 8, 1, 400), (195, 8, 2, 500), (154, 2, 3, 500)])
def test_default_of_many_rings(N, P, D, R):
    kw, x, p = system(N, P, D, N, **TRAP)
    b = G.Batch([G.make_params(**kw)] * R)
    assert b.form() == (False, 1)
    b.close()


def test_refused():
    b = make(few(thermostat="nose_hoover_np"))
    assert b.form() == (False, 1)
    with pytest.raises(G.PimdbError):
        b.set_form(True)
    assert b.form() == (False, 1)
    b.close()


def test_configure_and_autotune():
    systems = few()
    b = make(systems)
    assert b.form()[0]
    b.configure()          # nothing asked for
    assert b.form()[0]
    with pytest.raises(G.PimdbError):
        b.configure(100, 0)
    assert b.form()[0]
    threads, resident = b.autotune(2)
    assert threads in (256, 512, 1024) and 0 < resident <= 4 * G.device_cus()
    b.configure(threads, resident)
    assert not b.form()[0]
    b.configure()
    assert not b.form()[0]
    b.set_form(True)
    assert b.form()[0]
    b.close()


@pytest.mark.parametrize("D,kw", [(3, dict(nmthermostat=1)), (2, dict(TRAP, int_kind="dipole", int_strength=0.5))])
def test_forms_agree(D, kw):
    systems = [system(N, P, D, N + P, seed=N, **kw) for N, P in ((8, 4), (64, 16), (70, 9), (129, 8))]
    ref, _ = batch_run(systems, (6,), (512, 256))
    for form in (True, False):
        b = make(systems)
        b.set_form(form)
        b.step(2)
        b.set_form(not form)
        b.step(3)
        b.set_form(form)
        b.step(1)
        for r in range(len(systems)):
            close(b.state(r), ref[r], "%s %d" % (form, r))
        b.close()


# (Aziz pairs; more coordinates than one workgroup holds)
@pytest.mark.parametrize("N,P,kw", [(1, 8, {}), (4, 32, {}), (8, 5, dict(nmthermostat=1)), (8, 70, dict(TRAP)), (3, 128, dict(TRAP, fixcom=0))])
def test_handful_in_two_kernels(N, P, kw):
    kw, x, p = system(N, P, 3, 5 * N + P, **kw)
    got = context_run(kw, x, p, (6,))
    close(got, context_run(kw, x, p, (1, 2, 3)), "N=%d P=%d calls" % (N, P))
    ref, _ = batch_run([(kw, x, p)], (6,), (256, 1))
    close(got, ref[0], "N=%d P=%d persistent" % (N, P))
