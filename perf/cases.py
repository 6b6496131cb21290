"""Performance cases of the framework: what its users have it do, through its
public entry points, over the range of systems they run.

A case is a dict of plain values; its "kind" names the entry point:

  md           one ring polymer (Context): device-noise MD steps from a captured
               graph, then the state, as a run does between two outputs
  observables  the observables of one ring polymer (Context.observables)
  exchange     V_B of beads 1 and P and its gradient (autograd harness) on
               device tensors
  batch        independent replicas (Batch): MD steps of all of them, then
               every replica's state

and its "system" the physics: "trap" (particles in a harmonic trap, no periodic
boundaries, with free, harmonic or dipole pairs) or "helium" (He-4 with Aziz
pairs in a periodic cube at 0.02186 A^-3, cutoff L/2).

exact() recomputes a case with plain numpy and torch in 64 bits (the exchange
in extended precision), without this repository's code.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pimd-b_amd"))

import pimdb_amd as G  # noqa: E402

# atomic units
KELVIN = 3.1668152e-06
ANGSTROM = 1.8897261
FS = 41.341373
HE4 = 4.0026 * 1822.8885
MEV = 0.036749326e-3
HELIUM_DENSITY = 0.02186   # per cubic angstrom

DEFAULTS = dict(kind="md", system="trap", pairs="free", natoms=4, nbeads=32, ndim=3, bosonic=True, propagator="cartesian",
                thermostat="langevin", nmthermostat=False, fixcom=True, temperature=1.5, steps=100, replicas=1,
                uneven=False)


def _case(**kw):
    return dict(DEFAULTS, **kw)


def listed():
    return [
        # a handful of trapped bosons, the usual first run and the reference's own regression size: launches and
        # latency count, not arithmetic
        _case(name="md_trap_few", natoms=4, nbeads=32, temperature=1.0),
        # Nose-Hoover chains on the particles of a small trapped system (the reference's dynamics regressions)
        _case(name="md_nose_hoover", natoms=8, nbeads=16, temperature=5.8, thermostat="nose_hoover_np", fixcom=False),
        # tens of trapped bosons with harmonic pairs: an ordinary production run
        _case(name="md_trap_pairs", natoms=64, nbeads=64, temperature=2.0, pairs="harmonic"),
        # distinguishable particles with the normal-mode propagator (odd sizes)
        _case(name="md_modes", natoms=101, nbeads=24, temperature=2.0, pairs="dipole", bosonic=False,
              propagator="normal_modes"),
        # liquid helium, the benchmark's replica as one system: pair forces, exchange and normal-mode Langevin
        _case(name="md_helium", system="helium", natoms=256, nbeads=64, nmthermostat=True, steps=50),
        # a large helium box (Cartesian Langevin): the exchange recursion is long, the pairs are many
        _case(name="md_helium_large", system="helium", natoms=1000, nbeads=32, steps=10),
        # the energies, estimators and exchange probabilities taken every few steps of a helium run
        _case(name="observables_helium", kind="observables", system="helium", natoms=256, nbeads=64),
        # the differentiable exchange of a small planar system: the smallest call
        _case(name="exchange_small", kind="exchange", natoms=13, nbeads=16, ndim=2),
        # the differentiable exchange of a large periodic ring
        _case(name="exchange_large", kind="exchange", system="helium", natoms=500, nbeads=32),
        # a few replicas of the helium system: fewer than the card has compute units (error bars, a temperature ladder)
        _case(name="batch_helium_few", kind="batch", system="helium", natoms=256, nbeads=64, nmthermostat=True,
              replicas=16, steps=100),
        # hundreds of uneven planar dipole replicas (N 8..128, P 16, 32 or 64, T 1..4 K): a parameter scan
        _case(name="batch_dipole_scan", kind="batch", pairs="dipole", natoms=128, nbeads=64, ndim=2, replicas=512,
              uneven=True, steps=200),
        # helium replicas that fill the card: the throughput workload
        _case(name="batch_helium", kind="batch", system="helium", natoms=256, nbeads=64, nmthermostat=True,
              replicas=256, steps=100),
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case: sizes over the logarithm of the range of the listed ones, options in the mix they are used in."""
    kind = rng.choice(["md", "md", "md", "md", "observables", "exchange", "exchange", "batch", "batch"])
    system = rng.choice(["trap", "helium"])
    c = _case(kind=kind, system=system, temperature=round(rng.uniform(1.0, 4.0), 3))
    if kind == "exchange":
        c.update(natoms=_log_int(rng, 4, 600 if system == "helium" else 128), nbeads=rng.choice([8, 16, 32, 64]),
                 ndim=3 if system == "helium" else rng.choice([1, 2, 3]))
        return c
    P = rng.choice([4, 8, 12, 16, 24, 32, 48, 64])
    c["nbeads"] = P
    c["nmthermostat"] = rng.random() < 0.5
    c["fixcom"] = rng.random() < 0.7
    c["bosonic"] = rng.random() < 0.8
    if system == "helium":
        c["natoms"] = _log_int(rng, 16, 1000 if kind != "batch" else 256)
    else:
        c["natoms"] = _log_int(rng, 3, 128)
        c["ndim"] = rng.choice([1, 2, 3, 3])
        c["pairs"] = rng.choice(["free", "harmonic", "dipole"])
        if c["ndim"] == 1 and c["pairs"] == "dipole":
            c["pairs"] = "harmonic"   # (1/r^3 pairs do not integrate in one dimension)
        if rng.random() < 0.2:
            c["thermostat"] = rng.choice(["nose_hoover", "nose_hoover_np", "nose_hoover_np_dim"])
    if kind == "batch":
        c["replicas"] = _log_int(rng, 4, 512 if system == "trap" else 256)
        c["uneven"] = rng.random() < 0.5
        c["steps"] = rng.choice([50, 100])
    elif kind == "md":
        if not c["bosonic"] and rng.random() < 0.4:
            c["propagator"] = "normal_modes"
        c["steps"] = 10 if c["natoms"] > 400 else 50
    return c


# ---------------------------------------------------------------- inputs

def _system(c, N, P, T, rng, seed):
    """The parameters of one ring polymer of a case and its state: a jittered lattice with the beads of a particle
    0.3 bohr apart (an equilibrated ring's local spread), Maxwell-Boltzmann momenta."""
    D = c["ndim"]
    kw = dict(natoms=N, nbeads=P, ndim=D, mass=HE4, temperature=T * KELVIN, bosonic=int(c["bosonic"]), cutoff=-1.0,
              propagator=c["propagator"], thermostat=c["thermostat"], nmthermostat=int(c["nmthermostat"]),
              fixcom=int(c["fixcom"]), seed=int(seed))
    side = 1
    while side ** D < N:
        side += 1
    sites = np.indices((side,) * D).reshape(D, -1).T[rng.permutation(side ** D)[:N]].astype(float)
    if c["system"] == "helium":
        L = (N / HELIUM_DENSITY) ** (1.0 / 3.0) * ANGSTROM
        kw.update(dt=0.5 * FS, pbc=1, size=L, ext_kind="free", int_kind="aziz", cutoff=0.5 * L)
        centres = ((sites + 0.5) / side - 0.5) * L + rng.uniform(-0.5, 0.5, size=sites.shape)
        centres -= L * np.floor(centres / L + 0.5)
    else:
        kw.update(dt=20.0, pbc=0, size=60.0, ext_kind="harmonic", ext_omega=3.0 * MEV, int_kind=c["pairs"])
        if c["pairs"] == "harmonic":
            kw["int_omega"] = 1.0 * MEV
        if c["pairs"] == "dipole":
            kw["int_strength"] = rng.uniform(0.5, 2.0)
        centres = (sites - 0.5 * (side - 1)) * 4.0 + rng.uniform(-0.5, 0.5, size=sites.shape)
    kw["gamma"] = 1.0 / (100.0 * kw["dt"])
    x = centres[None] + rng.normal(0.0, 0.3, size=(P, N, D))
    p = rng.normal(0.0, math.sqrt(HE4 * kw["temperature"] * P), size=(P, N, D))
    if c["fixcom"]:
        p -= p.mean(axis=(0, 1))
    return kw, x, p


def _sizes(c):
    """N, P and T of every replica: the case's own or, uneven, spread below it (the same for every seed)."""
    N, P, T, R = c["natoms"], c["nbeads"], c["temperature"], c["replicas"]
    if not c["uneven"]:
        return [(N, P, T)] * R
    rng = np.random.default_rng([N, P, R])
    step = max(1, N // 16)
    return [(step * int(rng.integers(1, N // step + 1)), max(4, P >> int(rng.integers(0, 3))), rng.uniform(1.0, 4.0))
            for _ in range(R)]


def _systems(c, seed):
    """Every ring polymer of a case."""
    rng = np.random.default_rng([seed, 77])
    return [_system(c, N, P, T, rng, int(rng.integers(1, 900000000))) for N, P, T in _sizes(c)]


def _ring(c, kw):
    """beta~ and the spring constant of a ring polymer (hbar = kB = 1)."""
    P, T = kw["nbeads"], kw["temperature"]
    return 1.0 / (T * P), kw["mass"] * (P * T) ** 2


def prepare(case, seed):
    if case["kind"] == "exchange":
        from pimdb_amd.autograd import make_plan
        kw, x, _ = _systems(case, seed)[0]
        bt, k = _ring(case, kw)
        plan = make_plan(kw["natoms"], kw["ndim"], bt, k, pbc=bool(kw["pbc"]), size=kw["size"])
        x1, xP = (torch.tensor(v, dtype=torch.float64, device="cuda", requires_grad=True) for v in (x[0], x[-1]))
        return dict(kind="exchange", plan=plan, x1=x1, xP=xP)
    systems = _systems(case, seed)
    if case["kind"] == "batch":
        b = G.Batch([G.make_params(**kw) for kw, _, _ in systems])
        for r, (_, x, p) in enumerate(systems):
            b.set_state(r, x, p)
        b.forces()
        return dict(kind="batch", batch=b, replicas=len(systems), steps=case["steps"])
    kw, x, p = systems[0]
    ctx = G.Context(G.make_params(**kw))
    ctx.set_state(x, p)
    ctx.forces()
    ctx.graph_capture()
    return dict(kind=case["kind"], ctx=ctx, steps=case["steps"])


def run(state):
    kind = state["kind"]
    if kind == "md":
        state["ctx"].step(state["steps"])
        x, p, f = state["ctx"].state()
        return dict(x=x, p=p, f=f)
    if kind == "observables":
        return state["ctx"].observables()
    if kind == "exchange":
        from pimdb_amd.autograd import exchange_potential
        vb = exchange_potential(state["x1"], state["xP"], state["plan"])
        g1, gP = torch.autograd.grad(vb, (state["x1"], state["xP"]))
        return dict(vb=vb.detach(), g1=g1, gP=gP)
    b = state["batch"]
    b.step(state["steps"])
    every = [b.state(r) for r in range(state["replicas"])]
    return [np.concatenate([s[k].ravel() for s in every]) for k in range(3)]


# ---------------------------------------------------------------- work

def _step_flops(c, N, P):
    """Operations of one MD step: +, -, *, compare, floor, divide, square root 1, a fused multiply-add 2, exp and log 1."""
    D = c["ndim"]
    pbc = c["system"] == "helium"
    pairs = P * N * (N - 1) / 2
    if pbc:
        f = pairs * 8 * D + pairs * (math.pi / 6) * 50
    elif c["pairs"] == "free":
        f = 0.0
    else:
        f = pairs * (6 * D + (7 if c["pairs"] == "dipole" else 0))
    f += N * P * D * (14 if pbc else 6)
    if c["bosonic"]:
        f += N * N * (2.5 * (8 * D if pbc else 3 * D) + 14)
    f += 15 * N * P * D
    if c["nmthermostat"]:
        f += 4 * P * P * N * D
    if c["propagator"] == "normal_modes":
        f += 8 * P * P * N * D
    return f


def work(case):
    N, P, D = case["natoms"], case["nbeads"], case["ndim"]
    if case["kind"] == "exchange":
        f = N * N * (2.5 * (8 * D if case["system"] == "helium" else 3 * D) + 14)
        return dict(bytes=8.0 * (4 * N * D + 1), flops=f)
    if case["kind"] == "observables":
        return dict(bytes=8.0 * (2 * N * P * D + 11), flops=_step_flops(case, N, P))
    if case["kind"] == "md":
        return dict(bytes=8.0 * 5 * N * P * D, flops=case["steps"] * _step_flops(case, N, P))
    sizes = _sizes(case)
    return dict(bytes=8.0 * 5 * D * sum(N * P for N, P, _ in sizes),
                flops=case["steps"] * sum(_step_flops(case, N, P) for N, P, _ in sizes))


# ---------------------------------------------------------------- exact values

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _image(d, L):
    return d - L * np.floor(d / L + 0.5) if L else d


def _exchange(x1, x2, xPm1, xP, bt, k, L, interior=True):
    """V, V backwards, cycle energies and the forces on beads 1 and P in extended precision."""
    one = np.longdouble
    x1, x2, xPm1, xP = (np.asarray(v, dtype=one) for v in (x1, x2, xPm1, xP))
    bt, k, L = one(bt), one(k), one(L)
    N = len(x1)
    d = _image(xP[None, :, :] - x1[:, None, :], L)        # [u][v]: from x1[u] to xP[v]
    link = (_image(x1[1:] - xP[:-1], L) ** 2).sum(-1)
    S = np.concatenate([np.zeros(1, dtype=one), np.cumsum(link)])
    E = 0.5 * k * (S[None, :] - S[:, None] + (d ** 2).sum(-1))
    V = np.zeros(N + 1, dtype=one)
    for m in range(1, N + 1):
        t = E[:m, m - 1] + V[:m]
        s = t.min()
        V[m] = s - np.log(np.exp(-bt * (t - s)).sum() / m) / bt
    Vb = np.zeros(N + 1, dtype=one)
    inv = 1 / np.arange(1, N + 1, dtype=one)
    for u in range(N - 1, 0, -1):
        t = E[u, u:] + Vb[u + 1:]
        s = t.min()
        Vb[u] = s - np.log((np.exp(-bt * (t - s)) * inv[u:]).sum()) / bt
    Vb[0] = V[N]
    prob = np.triu(np.exp(-bt * np.where(np.triu(np.ones((N, N), dtype=bool)), V[:N, None] + E + Vb[None, 1:] - V[N], 0)))
    prob = (prob * inv[None, :]).T                          # [l][u], u <= l
    direct = 1 - np.exp(-bt * (V[1:N] + Vb[1:N] - V[N]))   # [l] to l + 1
    f1 = np.einsum("vu,uva->ua", prob, d)
    fP = -np.einsum("vu,uva->va", prob, d)
    e = _image(x1[1:] - xP[:-1], L)
    f1[1:] -= direct[:, None] * e
    fP[:-1] += direct[:, None] * e
    if interior:
        f1 += _image(x2 - x1, L)
        fP += _image(xPm1 - xP, L)
    return V, E, k * f1, k * fP


AZ = dict(rm=5.60738, A=0.5448504e6, eps=3.42016e-5, alpha=13.353384, D=1.241314, C6=1.3732412, C8=0.4253785, C10=0.1781)


def _pair(kw, r, r2):
    """Pair energy and (1/r) dV/dr."""
    if kw["int_kind"] == "harmonic":
        kp = kw["mass"] * kw["int_omega"] ** 2
        return 0.5 * kp * r2, kp * torch.ones_like(r)
    if kw["int_kind"] == "dipole":
        return kw["int_strength"] / r ** 3, -3.0 * kw["int_strength"] / r ** 5
    z = r / AZ["rm"]
    rep = AZ["A"] * torch.exp(-AZ["alpha"] * z)
    t = AZ["D"] / z - 1.0
    near = z < AZ["D"]
    F = torch.where(near, torch.exp(-t * t), torch.ones_like(z))
    dF = torch.where(near, 2.0 * AZ["D"] / (z * z) * t * F, torch.zeros_like(z))
    att = AZ["C6"] / z ** 6 + AZ["C8"] / z ** 8 + AZ["C10"] / z ** 10
    datt = 6 * AZ["C6"] / z ** 7 + 8 * AZ["C8"] / z ** 9 + 10 * AZ["C10"] / z ** 11
    g = AZ["eps"] / AZ["rm"] * (-AZ["alpha"] * rep + datt * F - att * dF)
    return AZ["eps"] * (rep - att * F), g / r


def _physical(kw, x, energies=False):
    """Trap and pair forces [P][N][D]; with energies (forces, trap energy, pair energy, virial sum), each per bead."""
    P, N, D = x.shape
    xt = torch.tensor(x, dtype=torch.float64, device=_dev())
    f = torch.zeros_like(xt)
    ext, pot, vir = np.zeros(P), np.zeros(P), np.zeros(P)
    if kw["ext_kind"] == "harmonic":
        a = kw["mass"] * kw["ext_omega"] ** 2
        f -= a * xt
        if energies:
            ext += 0.5 * a * (x ** 2).sum((1, 2))
            vir += a * (x ** 2).sum((1, 2))
    if kw["int_kind"] != "free":
        eye = torch.eye(N, dtype=torch.bool, device=xt.device)
        chunk = max(1, int(2 ** 24 // (N * N)))
        for b in range(0, P, chunk):
            q = xt[b:b + chunk]
            d = q[:, :, None, :] - q[:, None, :, :]
            if kw["pbc"]:
                d = d - kw["size"] * torch.floor(d / kw["size"] + 0.5)
            r2 = (d * d).sum(-1)
            r = torch.sqrt(torch.where(eye, torch.ones_like(r2), r2))
            out = eye if kw["cutoff"] < 0 else eye | (r >= kw["cutoff"])
            e, g = _pair(kw, r, r2)
            g = torch.where(out, torch.zeros_like(g), g)
            fp = -(g[..., None] * d).sum(2)
            f[b:b + chunk] += fp
            if energies:
                up = torch.triu(torch.ones_like(eye), 1)
                pot[b:b + chunk] = torch.where(up & ~out, e, torch.zeros_like(e)).sum((1, 2)).cpu().numpy()
                gd = torch.where(up, g, torch.zeros_like(g))[..., None] * d
                vir[b:b + chunk] += (q[:, :, None, :] * gd).sum((1, 2, 3)).cpu().numpy()
    f = f.cpu().numpy()
    return (f, ext, pot, vir) if energies else f


def _forces(kw, x):
    """(all forces, physical forces) of every bead."""
    P = kw["nbeads"]
    bt = 1.0 / (kw["temperature"] * P)
    k = kw["mass"] * (P * kw["temperature"]) ** 2
    L = kw["size"] if kw["pbc"] else 0.0
    phys = _physical(kw, x)
    spring = k * (_image(np.roll(x, 1, 0) - x, L) + _image(np.roll(x, -1, 0) - x, L))
    if kw["bosonic"] and P > 1:
        _, _, f1, fP = _exchange(x[0], x[1], x[-2], x[-1], bt, k, L)
        spring[0], spring[-1] = f1, fP
    return spring + phys, phys


def _modes(P):
    """Cartesian to normal modes, [mode][bead]."""
    b, j = np.arange(P)[:, None], np.arange(P)[None, :]
    w = 2 * math.pi / P * b * j
    C = np.where(b < 0.5 * P, math.sqrt(2.0 / P) * np.cos(w), -math.sqrt(2.0 / P) * np.sin(w))
    C[0] = 1 / math.sqrt(P)
    if P % 2 == 0:
        C[P // 2] = (1 - 2 * (np.arange(P) % 2)) / math.sqrt(P)
    return C


def _noise(seed, step, ostep, P, N, D):
    """The device noise of one O-step, [bead or mode][particle][axis]: Philox4x32-10 and Box-Muller."""
    half = (P + 1) // 2
    c = [np.arange(half * D * N, dtype=np.uint64), np.full(half * D * N, step, dtype=np.uint64),
         np.full(half * D * N, ostep, dtype=np.uint64), np.zeros(half * D * N, dtype=np.uint64)]
    k0, k1 = seed & 0xFFFFFFFF, 0x5EEDB05E
    low = np.uint64(0xFFFFFFFF)
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & low, (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & low]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    a = (c[0] << np.uint64(21)) ^ (c[1] >> np.uint64(11))
    b = (c[2] << np.uint64(21)) ^ (c[3] >> np.uint64(11))
    mask = np.uint64((1 << 53) - 1)
    u1 = ((a & mask).astype(float) + 1.0) / 2.0 ** 53
    u2 = (b & mask).astype(float) / 2.0 ** 53
    r = np.sqrt(-2.0 * np.log(u1))
    g = np.stack([r * np.cos(2 * math.pi * u2), r * np.sin(2 * math.pi * u2)])
    g = g.reshape(2, half, D, N).transpose(1, 0, 3, 2).reshape(2 * half, N, D)
    return g[:P]


class _Chains:
    """Nose-Hoover chains of four components, one per bead, per particle or per degree of freedom of a bead (or mode)."""

    def __init__(self, kw):
        P, N, D = kw["nbeads"], kw["natoms"], kw["ndim"]
        self.axes = {"nose_hoover": (1, 2), "nose_hoover_np": (2,), "nose_hoover_np_dim": ()}[kw["thermostat"]]
        ndof = {"nose_hoover": N * D, "nose_hoover_np": D, "nose_hoover_np_dim": 1}[kw["thermostat"]]
        shape = {"nose_hoover": (P, 1, 1), "nose_hoover_np": (P, N, 1), "nose_hoover_np_dim": (P, N, D)}[kw["thermostat"]]
        self.v, self.a = np.zeros((4,) + shape), np.zeros((4,) + shape)
        self.kT = kw["temperature"] * P
        self.Q = 1.0 / self.kT
        self.Q1, self.want = ndof * self.Q, ndof * self.kT
        self.dt, self.m = kw["dt"], kw["mass"]

    def scale(self, p):
        v, a, h, q = self.v, self.a, 0.25 * self.dt, 0.125 * self.dt
        e = (p * p).sum(self.axes, keepdims=True) / self.m if self.axes else p * p / self.m
        a[0] = (e - self.want) / self.Q1
        v[3] += a[3] * h
        for i in (2, 1, 0):
            f = np.exp(-q * v[i + 1])
            v[i] = (v[i] * f + a[i] * h) * f
        s = np.exp(-0.5 * self.dt * v[0])
        a[0] = (e * s * s - self.want) / self.Q1
        v[0] = (v[0] * f + a[0] * h) * f
        former = self.Q1
        for i in (1, 2):
            f = np.exp(-q * v[i + 1])
            v[i] = v[i] * f
            a[i] = (former * v[i - 1] ** 2 - self.kT) / self.Q
            v[i] = (v[i] + a[i] * h) * f
            former = self.Q
        a[3] = (self.Q * v[2] ** 2 - self.kT) / self.Q
        v[3] += a[3] * h
        return p * s


def _md(c, kw, x, p, steps):
    """OBABO steps from valid forces; the state after them."""
    P, N, D, dt, m = kw["nbeads"], kw["natoms"], kw["ndim"], kw["dt"], kw["mass"]
    c1 = math.exp(-0.5 * kw["gamma"] * dt)
    c2 = math.sqrt((1 - c1 * c1) * m * kw["temperature"] * P)
    C = _modes(P)
    nm = bool(kw["nmthermostat"])
    chains = _Chains(kw) if kw["thermostat"].startswith("nose") else None
    to_modes = lambda v: np.tensordot(C, v, 1)      # noqa: E731
    to_beads = lambda v: np.tensordot(C.T, v, 1)    # noqa: E731

    def ostep(p, step, o):
        if nm:
            p = to_modes(p)
        p = chains.scale(p) if chains else c1 * p + c2 * _noise(kw["seed"], step, o, P, N, D)
        if nm:
            p = to_beads(p)
        return p - p.mean(axis=(0, 1)) if kw["fixcom"] else p

    f, phys = _forces(kw, x)
    modes = kw["propagator"] == "normal_modes"
    w = 2 * P * kw["temperature"] * np.sin(np.arange(P) * math.pi / P)[:, None, None]
    for s in range(steps):
        p = ostep(p, s, 0)
        if modes:
            p = p + 0.5 * dt * phys
            q, pn = to_modes(x), to_modes(p)
            sn, cs = np.sin(w * dt), np.cos(w * dt)
            over = np.where(w == 0, dt / m, sn / np.where(w == 0, 1.0, m * w))
            x, p = to_beads(cs * q + over * pn), to_beads(cs * pn - m * w * sn * q)
        else:
            p = p + 0.5 * dt * f
            x = x + dt * p / m
        f, phys = _forces(kw, x)
        p = ostep(p + 0.5 * dt * (phys if modes else f), s + 1, 1)
    return x, p, f


def _observables(kw, x, p):
    P, N, D = kw["nbeads"], kw["natoms"], kw["ndim"]
    beta = 1.0 / kw["temperature"]
    bt, k = beta / P, kw["mass"] * (P / beta) ** 2
    L = kw["size"] if kw["pbc"] else 0.0
    _, ext, pot, vir = _physical(kw, x, energies=True)
    spring = 0.5 * k * (_image(x - np.roll(x, 1, 0), L) ** 2).sum((1, 2))
    kin = np.full(P, 0.5 * D * N / beta) - spring / P
    dist = whole = 0.0
    boson = kw["bosonic"] and P > 1
    if boson:
        V, E, _, _ = _exchange(x[0], x[1], x[-2], x[-1], bt, k, L)
        prim = np.zeros(N + 1, dtype=np.longdouble)
        for m in range(1, N + 1):
            e = E[:m, m - 1]
            prim[m] = ((prim[:m] - e) * np.exp(-np.longdouble(bt) * (e + V[:m] - V[m]))).sum() / m
        kin[0] = 0.5 * D * N / beta + float(prim[N]) / P
        spring[0] = float(V[N])
        dist = float(np.exp(-np.longdouble(bt) * (np.trace(E) - V[N]) - math.lgamma(N + 1.0)))
        whole = float(np.exp(-np.longdouble(bt) * (E[0, N - 1] - V[N])))
    both = kw["ext_kind"] != "free" and kw["int_kind"] != "free"
    ke = (p * p).sum() * 0.5 / kw["mass"]
    return np.array([kin.sum(), (ext + pot).sum() / P, ext.sum() / P if both else 0.0, pot.sum() / P if both else 0.0,
                     vir.sum() * 0.5 / P, 2.0 * ke / (D * N * P) / P, ke, spring.sum(), dist, whole, 0.0])


def _seconds(c):
    """About how long exact() takes."""
    N, P, D = c["natoms"], c["nbeads"], c["ndim"]
    one = P * N * N * 2.5e-8 + (P * N * D * 6e-7) + 1e-3 + P * P * N * D * 2e-9
    if c["bosonic"]:
        one += N * 9e-5 + N * N * 6e-7
    return one * (c["steps"] if c["kind"] in ("md", "batch") else 1) * c["replicas"]


def exact(case, seed):
    if _seconds(case) > 15.0:
        return None   # (batches and long runs)
    if case["kind"] == "exchange":
        kw, x, _ = _systems(case, seed)[0]
        bt, k = _ring(case, kw)
        V, _, f1, fP = _exchange(x[0], x[0], x[-1], x[-1], bt, k, kw["size"] if kw["pbc"] else 0.0, interior=False)
        return dict(vb=np.asarray(V[-1], dtype=float), g1=-f1.astype(float), gP=-fP.astype(float))
    systems = _systems(case, seed)
    if case["kind"] == "observables":
        return _observables(*systems[0])
    ends = [_md(case, kw, x, p, case["steps"]) for kw, x, p in systems]
    if case["kind"] == "md":
        return dict(zip("xpf", ends[0]))
    return [np.concatenate([e[k].ravel() for e in ends]) for k in range(3)]
