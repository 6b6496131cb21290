// pimdb_ctx.hip -- the single-system ("plain" per-kernel) form of the C ABI in
// include/pimdb_gpu.h.
//
// One MD step (Simulation::run body, src/simulation.cpp:246-259) is
//   K1 k_momenta      O-step (+ deferred zeroMomentum of the previous step)
//   K2 k_kick_drift   zeroMomentum, B, A          (or k_nm_propagate)
//   K3 k_step_forces  exchange recursions beside the bead forces, then
//                     k_exchange_forces (beads 1 and P)
//   K4 k_momenta      B, O-step, partial sums for zeroMomentum
// but device-noise Langevin (or NVE) steps take k_step_forces and one
// k_step_integrate (normal-mode propagator: k_step_modes) per step (steps.hpp),
// or a handful of particles one k_small_steps for many (small_steps.hpp), and
// Nose-Hoover ones k_step_forces and k_nh_steps (nh_steps.hpp).  Rings and
// slices beyond a workgroup's LDS take the recursions and the bead forces as
// two kernels on two streams.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <utility>
#include <vector>

#include "pimdb_gpu.h"
#include "ctx_common.hpp"
#include "exchange.hpp"
#include "factorial.hpp"
#include "forces.hpp"
#include "nose_hoover.hpp"
#include "integrator.hpp"
#include "observables.hpp"
#include "steps.hpp"
#include "nh_steps.hpp"
#include "small_steps.hpp"

using namespace pimdb;

struct pimdb_ctx {
    pimdb_params prm{};
    Derived dv{};
    int N = 0, P = 0, D = 0;
    size_t nbd = 0;
    char* arena = nullptr;         // holds every device buffer but E, ET, prob and noise
    hipStream_t s0 = nullptr, s1 = nullptr;
    hipEvent_t ev_fork = nullptr, ev_join = nullptr, t0 = nullptr, t1 = nullptr;
    double *x = nullptr, *p = nullptr, *f = nullptr, *fext = nullptr;
    double *E = nullptr, *ET = nullptr, *V = nullptr, *Vb = nullptr, *prob = nullptr, *fex = nullptr;
    double *Shi = nullptr, *Slo = nullptr;   // link prefix sums of the ring (exterior forces)
    unsigned long long* pub = nullptr;   // the recursions' published values (k_exchange_wide)
    double* xws = nullptr;   // the recursions' workspace in device memory, when it exceeds LDS
    double *C = nullptr, *CT = nullptr, *rot = nullptr, *com0 = nullptr, *com1 = nullptr;
    double *noise = nullptr, *obs = nullptr;
    size_t noise_cap = 0;
    int* status = nullptr;
    unsigned long long* ctr = nullptr;
    bool merged = false;           // recursions and bead forces in one k_step_forces
    PairGroups pg{};               // pair forces by groups of 128 (slice_groups.hpp)
    bool small = false;            // split steps, many in one k_small_steps
    bool nh_whole = false;         // consecutive Nose-Hoover steps by k_step_forces and k_nh_steps
    bool nh_close = false;         // closing halves with the exchange forces by k_nh_steps
    bool split = false;            // consecutive steps by k_step_forces and k_step_integrate
    double *xc = nullptr, *H = nullptr, *fpart = nullptr, *hpart = nullptr;   // their workspace (StepArgs)
    int tc = 1, ntiles = 1;
    int ncom = 1;                  // rows of the partial momentum sums (com0 / com1)
    NhArgs nh{};                   // Nose-Hoover chains (thermostat >= 2)
    double* modes = nullptr;       // normal modes of p, [k][a][i] (Nose-Hoover with nmthermostat)
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    double* pinned = nullptr;
    size_t pinned_cap = 0;
    std::string err;
    int fail(int code, const std::string& msg) {
        err = msg;
        return code;
    }
};

#define CK(expr)                                                                                   \
    do {                                                                                           \
        hipError_t e_ = (expr);                                                                    \
        if (e_ != hipSuccess) return ctx->fail(PIMDB_E_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

// ------------------------------------------------------------------ launches

template <int D>
static void launch_bead_forces_d(pimdb_ctx* ctx, hipStream_t s, double* f, double* fext) {
    ForceArgs fa = make_force_args(ctx->prm, ctx->dv);
    dim3 grid((ctx->N + FORCE_TILE - 1) / FORCE_TILE, ctx->P);
    const size_t red = sizeof(double) * (size_t)(FORCE_WAVES - 1) * D * FORCE_TILE;
    const size_t lds = sizeof(double) * (size_t)D * ctx->N + red;
    const dim3 blk(FORCE_TILE * FORCE_WAVES);
    if (lds > device_lds_limit()) {   // the slice read in place
        switch (ctx->prm.int_kind) {
        case POT_HARMONIC: hipLaunchKernelGGL((k_bead_forces<D, POT_HARMONIC, true>), grid, blk, red, s, fa, ctx->x, f, fext); break;
        case POT_DIPOLE: hipLaunchKernelGGL((k_bead_forces<D, POT_DIPOLE, true>), grid, blk, red, s, fa, ctx->x, f, fext); break;
        case POT_AZIZ: hipLaunchKernelGGL((k_bead_forces<D, POT_AZIZ, true>), grid, blk, red, s, fa, ctx->x, f, fext); break;
        default: hipLaunchKernelGGL((k_bead_forces<D, POT_FREE, true>), grid, blk, red, s, fa, ctx->x, f, fext); break;
        }
        return;
    }
    switch (ctx->prm.int_kind) {
    case POT_HARMONIC: hipLaunchKernelGGL((k_bead_forces<D, POT_HARMONIC>), grid, blk, lds, s, fa, ctx->x, f, fext); break;
    case POT_DIPOLE: hipLaunchKernelGGL((k_bead_forces<D, POT_DIPOLE>), grid, blk, lds, s, fa, ctx->x, f, fext); break;
    case POT_AZIZ: hipLaunchKernelGGL((k_bead_forces<D, POT_AZIZ>), grid, blk, lds, s, fa, ctx->x, f, fext); break;
    default: hipLaunchKernelGGL((k_bead_forces<D, POT_FREE>), grid, blk, lds, s, fa, ctx->x, f, fext); break;
    }
}

static void launch_bead_forces(pimdb_ctx* ctx, hipStream_t s) {
    double* fext = ctx->prm.propagator == PIMDB_PROP_NORMAL_MODES ? ctx->fext : nullptr;
    switch (ctx->D) {
    case 1: launch_bead_forces_d<1>(ctx, s, ctx->f, fext); break;
    case 2: launch_bead_forces_d<2>(ctx, s, ctx->f, fext); break;
    default: launch_bead_forces_d<3>(ctx, s, ctx->f, fext); break;
    }
}

// Both recursions (cycle energies recomputed from the ring's prefix sums,
// which are also left in Shi/Slo for the exterior forces).
static void launch_exchange_forward(pimdb_ctx* ctx, hipStream_t s) {
    launch_exchange_recursions(ctx->D, ctx->N, ctx->dv.bt, ctx->dv.k, ctx->prm.pbc, ctx->prm.size, ctx->x,
                               ctx->x + (size_t)(ctx->P - 1) * ctx->D * ctx->N, ctx->V, ctx->Vb, ctx->Shi, ctx->Slo,
                               ctx->pub, ctx->xws, ctx->status, s);
}

// Buffers of the outputs that take the energies or probabilities themselves,
// allocated when first asked for.
static int need_buffer(pimdb_ctx* ctx, double** buf, size_t n) {
    if (!*buf) CK(hipMalloc((void**)buf, sizeof(double) * n));
    return PIMDB_OK;
}

// The stored triangle E (and its row-major copy).
static void launch_cycle_energies_ctx(pimdb_ctx* ctx, hipStream_t s) {
    const int N = ctx->N, P = ctx->P;
    const double* x1 = ctx->x;
    const double* xP = ctx->x + (size_t)(P - 1) * ctx->D * N;
    launch_cycle_energies(ctx->D, N, x1, xP, ctx->dv.k, ctx->prm.pbc, ctx->prm.size, ctx->E, ctx->ET, s);
}

template <int D>
static void launch_exchange_forces_d(pimdb_ctx* ctx, hipStream_t s, double* f, double* fex) {
    const int N = ctx->N;
    hipLaunchKernelGGL((k_exchange_forces<D>), dim3((2 * N + 3) / 4), dim3(256), 0, s, N, ctx->P, ctx->dv.bt,
                       ctx->dv.k, ctx->prm.pbc, ctx->prm.size, ctx->Shi, ctx->Slo, ctx->V, ctx->Vb, ctx->x, f, fex);
}

static void launch_exchange_forces(pimdb_ctx* ctx, hipStream_t s, double* f, double* fex) {
    switch (ctx->D) {
    case 1: launch_exchange_forces_d<1>(ctx, s, f, fex); break;
    case 2: launch_exchange_forces_d<2>(ctx, s, f, fex); break;
    default: launch_exchange_forces_d<3>(ctx, s, f, fex); break;
    }
}

static bool factorial(const pimdb_ctx* ctx) {
    return ctx->dv.bosonic && ctx->prm.exchange_algo == PIMDB_EXCHANGE_FACTORIAL;
}

// The factorial exchange (one wave): forces added into f1 / fP, or written to
// fex; V_eff to VN; the estimator triple to est.
static void launch_factorial(pimdb_ctx* ctx, hipStream_t s, double* f, double* fex, double* VN, double* est) {
    const int N = ctx->N, P = ctx->P, D = ctx->D;
    const size_t bs = (size_t)D * N;
    const double* x1 = ctx->x;
    const double* x2 = ctx->x + bs * (1 % P);
    const double* xPm1 = ctx->x + bs * ((P - 2 + P) % P);
    const double* xP = ctx->x + bs * (P - 1);
    double* f1 = f ? f : nullptr;
    double* fP = f ? f + bs * (P - 1) : nullptr;
    const size_t lds = sizeof(double) * factorial_lds_doubles(N, D);
    const double bt = ctx->dv.bt, k = ctx->dv.k, L = ctx->prm.size;
    const int pbc = ctx->prm.pbc;
    switch (D) {
    case 1: hipLaunchKernelGGL(k_factorial_exchange<1>, dim3(1), dim3(FACT_LANES), lds, s, N, P, bt, k, pbc, L, x1, x2, xPm1, xP, f1, fP, fex, VN, est); break;
    case 2: hipLaunchKernelGGL(k_factorial_exchange<2>, dim3(1), dim3(FACT_LANES), lds, s, N, P, bt, k, pbc, L, x1, x2, xPm1, xP, f1, fP, fex, VN, est); break;
    default: hipLaunchKernelGGL(k_factorial_exchange<3>, dim3(1), dim3(FACT_LANES), lds, s, N, P, bt, k, pbc, L, x1, x2, xPm1, xP, f1, fP, fex, VN, est); break;
    }
}

// How the pair forces of a merged step are cut (PairGroups; G = 0 for one tile
// of 64 rows per workgroup).  nx, nn: workgroups of the recursions, which hold a
// compute unit each for as long as they take (8 us and 4.6 us per 100
// particles), and of the noise.
//
// A workgroup takes about 4 us and 1 us per 16 steps (Aziz).  Whole rounds over
// the card take groups whole (or in q1 parts); the beads that are left over
// would take as long again on a part of the card and are cut finer (N=400, P=64
// 56.7 -> 46.1 us a step, N=1000, P=32 85 -> 79.5, P=64 133 -> 119; too few
// workgroups to fill the card: N=1000, P=4 without exchange 44.0, 28.6, 25.0, 21.3
// with 1 .. 4 parts).  Finer only for a tenth less, since the integration reads
// the sums of every part.
static PairGroups plan_pair_groups(const pimdb_params& p, const Derived& d, int nx, int nn) {
    PairGroups pg{};
    const int N = p.natoms, P = p.nbeads;
    if (p.int_kind == PIMDB_POT_FREE || d.cutoff == 0.0 || N <= GROUP_MIN) return pg;
    const int G = (N + GROUP - 1) / GROUP;
    const int steps = GROUP_OWN + group_seg_start(G, group_segments(G)), cus = std::max(1, device_cus() - nx);
    const double rec = nx ? 8.0 + 0.046 * N : 0.0;
    auto us = [&](int q) { return 4.0 + steps / (16.0 * q); };
    double best = 0.0;
    for (int q1 = 1; q1 <= GROUP_PARTS; ++q1) {
        for (int q2 = q1; q2 <= GROUP_PARTS; ++q2) {
            const int k = std::max(group_kslots(G, q1), group_kslots(G, q2));
            if (sizeof(double) * group_lds_doubles(p.ndim, k) > device_lds_limit()) continue;
            const int rounds = P * G * q1 / cus;
            const int b1 = q1 == q2 ? 0 : std::min(P, std::max(0, rounds * cus - nn) / (G * q1));
            const int left = (P - b1) * G * q2;
            const double t = std::max((b1 ? rounds * us(q1) : 0.0) + (left + cus - 1) / cus * us(q2), rec);
            if (!pg.G || t < 0.9 * best) {
                best = t;
                pg.G = G; pg.kslots = k;
                pg.b1 = b1; pg.q1 = q1; pg.q2 = q2;
            }
        }
    }
    return pg;
}

static StepArgs step_args(pimdb_ctx* ctx) {
    StepArgs a{};
    a.fa = make_force_args(ctx->prm, ctx->dv);
    a.bt = ctx->dv.bt;
    a.thermostat = ctx->prm.thermostat;
    a.nm = ctx->prm.nmthermostat;
    a.fixcom = ctx->prm.fixcom;
    a.x = ctx->x; a.p = ctx->p; a.f = ctx->f;
    a.fext = ctx->prm.propagator == PIMDB_PROP_NORMAL_MODES ? ctx->fext : nullptr;
    a.V = ctx->V; a.Vb = ctx->Vb; a.Shi = ctx->Shi; a.Slo = ctx->Slo; a.xc = ctx->xc;
    a.pub = ctx->pub; a.status = ctx->status;
    a.c1 = a.thermostat ? ctx->dv.c1 : 1.0;
    a.c2 = ctx->dv.c2;
    a.half_dt = 0.5 * ctx->prm.dt;
    a.dt_m = ctx->prm.dt / ctx->prm.mass;
    a.Ct = ctx->C; a.CTt = ctx->CT; a.rot = ctx->rot;
    a.H = ctx->H; a.hpart = ctx->hpart;
    a.frows = ctx->P * ((ctx->N + FORCE_TILE - 1) / FORCE_TILE);
    a.fpart = ctx->prm.ext_kind != PIMDB_POT_FREE && a.fixcom ? ctx->fpart : nullptr;
    a.pg = ctx->pg;
    a.ctr = ctx->ctr;
    a.seed = ctx->prm.seed;
    return a;
}

static size_t tile_lds_bytes(int N, int D) {
    return sizeof(double) * ((size_t)D * N + (size_t)(FORCE_WAVES - 1) * D * FORCE_TILE);
}

template <int D>
static void launch_step_forces_d(pimdb_ctx* ctx, bool forces, bool noise, int mode, bool ring) {
    const StepArgs a = step_args(ctx);
    const int nx = forces && ring && ctx->dv.bosonic ? xw_grid(ctx->N) : 0, nf = !forces ? 0 : a.pg.G ? a.pg.groups_of(ctx->P) : a.frows;
    const int nn = noise ? step_noise_groups(a, D) : 0;
    if (nx + nf + nn == 0) return;
    size_t lds = 0;
    if (nf) lds = a.pg.G ? sizeof(double) * group_lds_doubles(D, a.pg.kslots) : tile_lds_bytes(ctx->N, D);
    if (nx) lds = std::max(lds, xw_lds_bytes(ctx->N, D));
    if (nn) lds = std::max(lds, sizeof(double) * step_noise_lds_doubles<XW_THREADS>(ctx->P, a.thermostat && a.nm));
    const dim3 grid(nx + nf + nn), blk(XW_THREADS);
    const hipStream_t s = ctx->s0;
    switch (ctx->prm.int_kind) {
    case POT_HARMONIC: hipLaunchKernelGGL((k_step_forces<D, POT_HARMONIC>), grid, blk, lds, s, a, nx, nn, mode); break;
    case POT_DIPOLE: hipLaunchKernelGGL((k_step_forces<D, POT_DIPOLE>), grid, blk, lds, s, a, nx, nn, mode); break;
    case POT_AZIZ: hipLaunchKernelGGL((k_step_forces<D, POT_AZIZ>), grid, blk, lds, s, a, nx, nn, mode); break;
    default: hipLaunchKernelGGL((k_step_forces<D, POT_FREE>), grid, blk, lds, s, a, nx, nn, mode); break;
    }
}

// The recursions and bead forces (forces: all but the exterior forces of beads
// 1 and P) and the noise of the integration of this mode (noise).  ring false:
// without the recursions.
static void launch_step_forces(pimdb_ctx* ctx, bool forces, bool noise, int mode, bool ring = true) {
    switch (ctx->D) {
    case 1: launch_step_forces_d<1>(ctx, forces, noise, mode, ring); break;
    case 2: launch_step_forces_d<2>(ctx, forces, noise, mode, ring); break;
    default: launch_step_forces_d<3>(ctx, forces, noise, mode, ring); break;
    }
}

// f (and fext) completed with the group pair forces' slots.
static void launch_pair_sum(pimdb_ctx* ctx) {
    if (ctx->pg.G)
        hipLaunchKernelGGL(k_pair_sum, dim3((unsigned)((ctx->nbd + 255) / 256)), dim3(256), 0, ctx->s0, ctx->nbd,
                           (size_t)ctx->D * ctx->N, ctx->pg, ctx->f, ctx->prm.propagator == PIMDB_PROP_NORMAL_MODES ? ctx->fext : nullptr);
}

static void launch_step_integrate(pimdb_ctx* ctx, int mode) {
    StepArgs a = step_args(ctx);
    if (ctx->prm.propagator == PIMDB_PROP_NORMAL_MODES) {
        if (mode != STEP_CLOSE) {
            const dim3 mgrid(step_modes_groups(ctx->N, ctx->D));
            const size_t lds = sizeof(double) * step_modes_lds_doubles(ctx->P);
            switch (ctx->D) {
            case 1: hipLaunchKernelGGL(k_step_modes<1>, mgrid, dim3(256), lds, ctx->s0, a, mode); break;
            case 2: hipLaunchKernelGGL(k_step_modes<2>, mgrid, dim3(256), lds, ctx->s0, a, mode); break;
            default: hipLaunchKernelGGL(k_step_modes<3>, mgrid, dim3(256), lds, ctx->s0, a, mode); break;
            }
            return;
        }
        a.f = a.fext;   // the closing kick (f and fext are complete)
        a.pg = PairGroups{};
    }
    const dim3 grid(step_integrate_groups(a.fa, ctx->D, mode));
    switch (ctx->D) {
    case 1: hipLaunchKernelGGL(k_step_integrate<1>, grid, dim3(256), 0, ctx->s0, a, mode); break;
    case 2: hipLaunchKernelGGL(k_step_integrate<2>, grid, dim3(256), 0, ctx->s0, a, mode); break;
    default: hipLaunchKernelGGL(k_step_integrate<3>, grid, dim3(256), 0, ctx->s0, a, mode); break;
    }
}

// Forces of every bead (updateForces on all ranks); f and (NM propagator) fext.
static int enqueue_forces(pimdb_ctx* ctx) {
    if (ctx->merged) {
        launch_step_forces(ctx, true, false, STEP_CLOSE);
        launch_pair_sum(ctx);
        if (ctx->dv.bosonic) launch_exchange_forces(ctx, ctx->s0, ctx->f, nullptr);
    } else if (factorial(ctx)) {
        launch_bead_forces(ctx, ctx->s0);
        launch_factorial(ctx, ctx->s0, ctx->f, nullptr, nullptr, nullptr);
    } else if (ctx->dv.bosonic) {
        CK(hipEventRecord(ctx->ev_fork, ctx->s0));
        CK(hipStreamWaitEvent(ctx->s1, ctx->ev_fork, 0));
        launch_exchange_forward(ctx, ctx->s1);
        CK(hipEventRecord(ctx->ev_join, ctx->s1));
        launch_bead_forces(ctx, ctx->s0);
        CK(hipStreamWaitEvent(ctx->s0, ctx->ev_join, 0));
        launch_exchange_forces(ctx, ctx->s0, ctx->f, nullptr);
    } else {
        launch_bead_forces(ctx, ctx->s0);
    }
    CK(hipGetLastError());
    return PIMDB_OK;
}

static MomentaArgs momenta_args(pimdb_ctx* ctx, int ostep, const double* noise) {
    MomentaArgs m{};
    m.N = ctx->N; m.P = ctx->P; m.D = ctx->D; m.tc = ctx->tc;
    m.half_dt = 0.5 * ctx->prm.dt;
    m.c1 = ctx->dv.c1; m.c2 = ctx->dv.c2;
    m.thermostat = ctx->prm.thermostat;
    m.nm = ctx->prm.nmthermostat;
    m.Ct = ctx->C; m.CTt = ctx->CT;
    m.noise = noise;
    m.step_ctr = ctx->ctr;
    m.ostep = (uint32_t)ostep;
    m.seed = ctx->prm.seed;
    m.replica = 0;
    return m;
}

static size_t momenta_lds(pimdb_ctx* ctx) {
    return sizeof(double) * (2 * (size_t)ctx->P * ctx->tc + 256 / WAVE);
}

// One Nose-Hoover O-step: the pending zeroMomentum (com_in), the half kick
// (kick_f), the chains, the partial sums of the result (com_out).  Under
// normal-mode coupling the chains act on the modes: transform (k_momenta
// stage 1), chains, back-transform with the partial sums (stage 2).
static void enqueue_nh_ostep(pimdb_ctx* ctx, const double* com_in, const double* kick_f, double* com_out) {
    NhArgs h = ctx->nh;
    h.half_dt = 0.5 * ctx->prm.dt;
    if (!ctx->prm.nmthermostat) {
        h.com_in = com_in;
        h.ncom_in = ctx->ncom;
        h.kick_f = kick_f;
        h.com_out = com_out;
        hipLaunchKernelGGL(k_nh_ostep, dim3(ctx->P), dim3(256), 0, ctx->s0, h, ctx->p);
        return;
    }
    dim3 tgrid(ctx->ntiles, ctx->D);
    MomentaArgs m = momenta_args(ctx, 0, nullptr);
    m.thermostat = 0;
    m.stage = 1;
    m.modes = ctx->modes;
    m.com_in = com_in;
    m.ncom_in = ctx->ncom;
    m.kick_f = kick_f;
    hipLaunchKernelGGL(k_momenta, tgrid, dim3(256), momenta_lds(ctx), ctx->s0, m, ctx->p);
    h.com_in = nullptr;
    h.kick_f = nullptr;
    h.com_out = nullptr;
    hipLaunchKernelGGL(k_nh_ostep, dim3(ctx->P), dim3(256), 0, ctx->s0, h, ctx->modes);
    m.stage = 2;
    m.com_in = nullptr;
    m.kick_f = nullptr;
    m.com_out = com_out;
    hipLaunchKernelGGL(k_momenta, tgrid, dim3(256), momenta_lds(ctx), ctx->s0, m, ctx->p);
}

// Up to the drift: K1 and K2.
static void enqueue_open(pimdb_ctx* ctx, const double* noise0) {
    const bool fixcom = ctx->prm.fixcom != 0;
    const int N = ctx->N, P = ctx->P, D = ctx->D;
    dim3 tgrid(ctx->ntiles, D);
    // K1: deferred zeroMomentum + O-step
    if (ctx->prm.thermostat >= PIMDB_THERMO_NOSE_HOOVER) {
        enqueue_nh_ostep(ctx, fixcom ? ctx->com1 : nullptr, nullptr, fixcom ? ctx->com0 : nullptr);
    } else {
        MomentaArgs m1 = momenta_args(ctx, 0, noise0);
        m1.com_in = fixcom ? ctx->com1 : nullptr;
        m1.ncom_in = ctx->ncom;
        m1.com_out = fixcom ? ctx->com0 : nullptr;
        hipLaunchKernelGGL(k_momenta, tgrid, dim3(256), momenta_lds(ctx), ctx->s0, m1, ctx->p);
    }
    // K2: zeroMomentum + B + A   (or the normal-mode propagator)
    if (ctx->prm.propagator == PIMDB_PROP_NORMAL_MODES) {
        NmPropArgs a{};
        a.N = N; a.P = P; a.D = D; a.tc = ctx->tc;
        a.half_dt = 0.5 * ctx->prm.dt; a.dt = ctx->prm.dt; a.mass = ctx->prm.mass;
        a.Ct = ctx->C; a.CTt = ctx->CT; a.rot = ctx->rot;
        a.com_in = fixcom ? ctx->com0 : nullptr; a.ncom_in = ctx->ncom;
        a.fext = ctx->fext; a.step_ctr = ctx->ctr;
        hipLaunchKernelGGL(k_nm_propagate, tgrid, dim3(256), sizeof(double) * 4 * (size_t)P * ctx->tc, ctx->s0, a,
                           ctx->x, ctx->p);
    } else {
        DriftArgs d{};
        d.N = N; d.P = P; d.D = D;
        d.half_dt = 0.5 * ctx->prm.dt; d.dt = ctx->prm.dt; d.mass = ctx->prm.mass;
        d.com_in = fixcom ? ctx->com0 : nullptr; d.ncom_in = ctx->ncom;
        d.step_ctr = ctx->ctr;
        hipLaunchKernelGGL(k_kick_drift, dim3((unsigned)((ctx->nbd + 255) / 256)), dim3(256), 0, ctx->s0, d, ctx->x,
                           ctx->p, ctx->f);
    }
}

template <int D>
static void launch_nh_steps_d(pimdb_ctx* ctx, int mode) {
    const StepArgs a = step_args(ctx);
    NhArgs h = ctx->nh;
    h.half_dt = 0.5 * ctx->prm.dt;
    if (!ctx->nh_whole && ctx->prm.fixcom) h.com_out = ctx->com1;
    const int nb = ctx->prm.fixcom && ctx->nh_whole ? ctx->P : 1;
    const bool ext = ctx->dv.bosonic && ctx->N <= NH_EXT;
    hipLaunchKernelGGL(k_nh_steps<D>, dim3(ctx->P / nb), dim3(NH_THREADS),
                       sizeof(double) * nh_step_lds_doubles(ctx->N, D, nb, ext), ctx->s0, a, h, nb, ext ? 1 : 0, mode);
}

static void launch_nh_steps(pimdb_ctx* ctx, int mode) {
    switch (ctx->D) {
    case 1: launch_nh_steps_d<1>(ctx, mode); break;
    case 2: launch_nh_steps_d<2>(ctx, mode); break;
    default: launch_nh_steps_d<3>(ctx, mode); break;
    }
}

// The closing half: K4 (B + O-step + partial COM sums).
static void enqueue_close(pimdb_ctx* ctx, const double* noise1) {
    const bool fixcom = ctx->prm.fixcom != 0;
    dim3 tgrid(ctx->ntiles, ctx->D);
    const double* kick = ctx->prm.propagator == PIMDB_PROP_NORMAL_MODES ? ctx->fext : ctx->f;
    if (ctx->prm.thermostat >= PIMDB_THERMO_NOSE_HOOVER) {
        enqueue_nh_ostep(ctx, nullptr, kick, fixcom ? ctx->com1 : nullptr);
    } else {
        MomentaArgs m2 = momenta_args(ctx, 1, noise1);
        m2.kick_f = kick;
        m2.com_out = fixcom ? ctx->com1 : nullptr;
        hipLaunchKernelGGL(k_momenta, tgrid, dim3(256), momenta_lds(ctx), ctx->s0, m2, ctx->p);
    }
}

// One OBABO step; noise0/noise1: host noise of the two O-steps, on the device, or
// null for device noise.
static int enqueue_step(pimdb_ctx* ctx, const double* noise0, const double* noise1) {
    enqueue_open(ctx, noise0);
    if (ctx->nh_close) {
        launch_step_forces(ctx, true, false, STEP_CLOSE);
        launch_nh_steps(ctx, STEP_CLOSE);
    } else {
        const int rc = enqueue_forces(ctx);
        if (rc) return rc;
        enqueue_close(ctx, noise1);
    }
    CK(hipGetLastError());
    return PIMDB_OK;
}

// nsteps Nose-Hoover steps by k_step_forces and k_nh_steps.
static int enqueue_nh_steps(pimdb_ctx* ctx, int nsteps) {
    if (nsteps == 0) return PIMDB_OK;
    launch_nh_steps(ctx, STEP_OPEN);
    for (int s = 1; s <= nsteps; ++s) {
        launch_step_forces(ctx, true, false, STEP_CLOSE);
        launch_pair_sum(ctx);
        if (ctx->dv.bosonic && ctx->N > NH_EXT) launch_exchange_forces(ctx, ctx->s0, ctx->f, nullptr);
        launch_nh_steps(ctx, s < nsteps ? STEP_FULL : STEP_CLOSE);
    }
    CK(hipGetLastError());
    return PIMDB_OK;
}

template <int D>
static void launch_small_steps_d(pimdb_ctx* ctx, int nsteps) {
    const StepArgs a = step_args(ctx);
    const size_t lds = sizeof(double) * small_lds_doubles(ctx->N, ctx->P, D, a.thermostat && a.nm);
    const dim3 grid(1), blk(SMALL_THREADS);
    switch (ctx->prm.int_kind) {
    case POT_HARMONIC: hipLaunchKernelGGL((k_small_steps<D, POT_HARMONIC>), grid, blk, lds, ctx->s0, a, nsteps); break;
    case POT_DIPOLE: hipLaunchKernelGGL((k_small_steps<D, POT_DIPOLE>), grid, blk, lds, ctx->s0, a, nsteps); break;
    default: hipLaunchKernelGGL((k_small_steps<D, POT_FREE>), grid, blk, lds, ctx->s0, a, nsteps); break;
    }
}

static int enqueue_small_steps(pimdb_ctx* ctx, int nsteps) {
    for (int s = 0; s < nsteps; s += SMALL_STEPS) {
        const int n = std::min(SMALL_STEPS, nsteps - s);
        switch (ctx->D) {
        case 1: launch_small_steps_d<1>(ctx, n); break;
        case 2: launch_small_steps_d<2>(ctx, n); break;
        default: launch_small_steps_d<3>(ctx, n); break;
        }
    }
    CK(hipGetLastError());
    return PIMDB_OK;
}

// nsteps device-noise steps.
static int enqueue_steps(pimdb_ctx* ctx, int nsteps) {
    if (ctx->small) return enqueue_small_steps(ctx, nsteps);
    if (ctx->nh_whole) return enqueue_nh_steps(ctx, nsteps);
    if (!ctx->split) {
        for (int s = 0; s < nsteps; ++s) {
            if (ctx->gexec) {
                CK(hipGraphLaunch(ctx->gexec, ctx->s0));
            } else {
                const int rc = enqueue_step(ctx, nullptr, nullptr);
                if (rc) return rc;
            }
        }
        return PIMDB_OK;
    }
    if (nsteps == 0) return PIMDB_OK;
    launch_step_forces(ctx, false, true, STEP_OPEN);
    launch_step_integrate(ctx, STEP_OPEN);
    for (int s = 1; s <= nsteps; ++s) {
        const int mode = s < nsteps ? STEP_FULL : STEP_CLOSE;
        launch_step_forces(ctx, true, true, mode);
        if (ctx->prm.propagator == PIMDB_PROP_NORMAL_MODES) launch_pair_sum(ctx);
        launch_step_integrate(ctx, mode);
    }
    CK(hipGetLastError());
    return PIMDB_OK;
}

// Apply the pending zeroMomentum of the last O-step and clear the partials.
// (Split and whole Nose-Hoover steps leave neither.)
static int finish_steps(pimdb_ctx* ctx, bool host_noise) {
    if (ctx->prm.fixcom && (host_noise || !(ctx->split || ctx->nh_whole))) {
        hipLaunchKernelGGL(k_com_subtract, dim3((unsigned)((ctx->nbd + 255) / 256)), dim3(256), 0, ctx->s0, ctx->N,
                           ctx->P, ctx->D, ctx->com1, ctx->ncom, ctx->p);
        CK(hipMemsetAsync(ctx->com1, 0, sizeof(double) * (size_t)ctx->ncom * ctx->D, ctx->s0));
    }
    CK(hipGetLastError());
    return PIMDB_OK;
}

// Layout of ctx->obs: bead sums [P][2], energies [P][tiles][3], then the
// estimators: k_ring_estimator's 2N + 2 values, or of the factorial exchange
// the triple (and V_eff at 2N + 1); then the Nose-Hoover energy.
static size_t obs_tail(int N, int P) { return 2 * (size_t)P + 3 * (size_t)P * ((N + FORCE_TILE - 1) / FORCE_TILE); }
static size_t obs_doubles(int N, int P) { return obs_tail(N, P) + std::max<size_t>(2 * (size_t)N + 2, 5) + 1; }

// Copies n doubles of ctx->obs from offset `from` to h (may be larger than a
// pinned buffer) and waits.
static hipError_t read_obs(pimdb_ctx* ctx, size_t from, std::vector<double>& h) {
    const Stage st(h.size());
    if (!st.b.first) return hipErrorOutOfMemory;
    for (size_t o = 0; o < h.size(); o += st.b.second) {
        const size_t n = std::min(st.b.second, h.size() - o);
        hipError_t e = hipMemcpyAsync(st.b.first, ctx->obs + from + o, n * sizeof(double), hipMemcpyDeviceToHost, ctx->s0);
        const hipError_t w = hipStreamSynchronize(ctx->s0);
        if (e == hipSuccess) e = w;
        if (e != hipSuccess) return e;
        std::memcpy(h.data() + o, st.b.first, n * sizeof(double));
    }
    return hipSuccess;
}

static void launch_estimators(pimdb_ctx* ctx) {
    const int N = ctx->N, D = ctx->D;
    const double* xP = ctx->x + (size_t)(ctx->P - 1) * D * N;
    double* out = ctx->obs + obs_tail(N, ctx->P);
    const dim3 grid((N + 3) / 4), blk(256);
    switch (D) {
    case 1: hipLaunchKernelGGL(k_ring_estimator<1>, grid, blk, 0, ctx->s0, N, ctx->dv.bt, ctx->dv.k, ctx->prm.pbc, ctx->prm.size, ctx->x, xP, ctx->Shi, ctx->Slo, ctx->V, ctx->Vb, out); break;
    case 2: hipLaunchKernelGGL(k_ring_estimator<2>, grid, blk, 0, ctx->s0, N, ctx->dv.bt, ctx->dv.k, ctx->prm.pbc, ctx->prm.size, ctx->x, xP, ctx->Shi, ctx->Slo, ctx->V, ctx->Vb, out); break;
    default: hipLaunchKernelGGL(k_ring_estimator<3>, grid, blk, 0, ctx->s0, N, ctx->dv.bt, ctx->dv.k, ctx->prm.pbc, ctx->prm.size, ctx->x, xP, ctx->Shi, ctx->Slo, ctx->V, ctx->Vb, out); break;
    }
}

// The exchange estimators' limit on natoms (about 20,000): what the workgroup of
// their first form held.  The present kernels have none; larger rings stay
// refused.
static bool estimator_fits(int N) { return sizeof(double) * ((size_t)N + 1 + 16) <= device_lds_limit(); }

template <int D>
static void launch_observe_d(pimdb_ctx* ctx) {
    ObserveArgs o{};
    const int N = ctx->N, P = ctx->P;
    o.fa = make_force_args(ctx->prm, ctx->dv);
    o.bt = ctx->dv.bt;
    o.nx = ctx->dv.bosonic ? xw_grid(N) : 0;
    o.nf = P * ((N + FORCE_TILE - 1) / FORCE_TILE);
    o.x = ctx->x; o.p = ctx->p;
    o.V = ctx->V; o.Vb = ctx->Vb; o.Shi = ctx->Shi; o.Slo = ctx->Slo;
    o.pub = ctx->pub; o.status = ctx->status;
    o.sums = ctx->obs;
    o.epart = ctx->obs + 2 * (size_t)P;
    const size_t red = std::max<size_t>(3 * FORCE_WAVES, 2 * XW_THREADS / WAVE);
    size_t lds = sizeof(double) * ((size_t)D * N + red);
    if (o.nx) lds = std::max(lds, xw_lds_bytes(N, D));
    const dim3 grid(o.nx + o.nf + P), blk(XW_THREADS);
    switch (ctx->prm.int_kind) {
    case POT_HARMONIC: hipLaunchKernelGGL((k_observe<D, POT_HARMONIC>), grid, blk, lds, ctx->s0, o); break;
    case POT_DIPOLE: hipLaunchKernelGGL((k_observe<D, POT_DIPOLE>), grid, blk, lds, ctx->s0, o); break;
    case POT_AZIZ: hipLaunchKernelGGL((k_observe<D, POT_AZIZ>), grid, blk, lds, ctx->s0, o); break;
    default: hipLaunchKernelGGL((k_observe<D, POT_FREE>), grid, blk, lds, ctx->s0, o); break;
    }
}

// Waits for the stream.  The flag is pinned host memory that the kernels write
// through, so looking at it takes no copy.
static int check_status(pimdb_ctx* ctx) {
    CK(hipStreamSynchronize(ctx->s0));
    if (const int st = *(volatile int*)ctx->status) {
        *(volatile int*)ctx->status = 0;
        CK(empty_published(ctx->pub, xw_pub_words(ctx->N), ctx->s0));
        if (lost_wait(st)) return ctx->fail(PIMDB_E_HIP, LOST_WAIT_MESSAGE);
        return ctx->fail(PIMDB_E_NONFINITE, "Invalid sig_denom in bosonic exchange potential (non-finite V)");
    }
    return PIMDB_OK;
}

static double* pinned_buffer(pimdb_ctx* ctx, size_t n) {
    if (ctx->pinned_cap < n) {
        if (ctx->pinned) (void)hipHostFree(ctx->pinned);
        ctx->pinned = nullptr;
        ctx->pinned_cap = 0;
        if (hipHostMalloc((void**)&ctx->pinned, n * sizeof(double), hipHostMallocDefault) != hipSuccess) return nullptr;
        ctx->pinned_cap = n;
    }
    return ctx->pinned;
}

// ------------------------------------------------------------------ C ABI

extern "C" {

int pimdb_ctx_create(const pimdb_params* prm, pimdb_ctx** out) {
    if (!prm || !out) return PIMDB_E_ARG;
    *out = nullptr;
    std::string why;
    if (!validate_params(*prm, &why)) {
        set_create_error(why);
        return PIMDB_E_ARG;
    }
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) {
        set_create_error("no HIP device available");
        return PIMDB_E_HIP;
    }
    pimdb_ctx* ctx = new pimdb_ctx();
    ctx->prm = *prm;
    ctx->dv = derive(*prm);
    ctx->N = prm->natoms; ctx->P = prm->nbeads; ctx->D = prm->ndim;
    ctx->nbd = (size_t)ctx->N * ctx->P * ctx->D;
    ctx->tc = column_tile(ctx->P);
    ctx->ntiles = (ctx->N + ctx->tc - 1) / ctx->tc;
    const int N = ctx->N, P = ctx->P, D = ctx->D;
    int rc = PIMDB_OK;
    // one device allocation for all buffers (each of its own costs 10 us or more)
    std::vector<std::pair<void**, size_t>> want;   // pointer, offset
    size_t arena = 0;
    auto alloc = [&](auto** ptr, size_t bytes) {
        want.push_back({(void**)ptr, arena});
        arena += (bytes + 255) & ~(size_t)255;
    };
    alloc(&ctx->x, sizeof(double) * ctx->nbd);
    alloc(&ctx->p, sizeof(double) * ctx->nbd);
    alloc(&ctx->f, sizeof(double) * ctx->nbd);
    alloc(&ctx->fext, sizeof(double) * ctx->nbd);
    alloc(&ctx->V, sizeof(double) * (N + 1));
    alloc(&ctx->Vb, sizeof(double) * (N + 1));
    alloc(&ctx->Shi, sizeof(double) * N);
    alloc(&ctx->Slo, sizeof(double) * N);
    // the recursions' published values, or both workspaces in device memory
    // when the ring exceeds the LDS of a workgroup
    const bool ring = ctx->dv.bosonic && prm->exchange_algo != PIMDB_EXCHANGE_FACTORIAL;
    const bool wide = ring && exchange_wide(N, D);
    if (wide) alloc(&ctx->pub, 8 * xw_pub_words(N));
    else if (ring) alloc(&ctx->xws, 2 * rec_lds_bytes(N, D));
    const bool slice_fits = tile_lds_bytes(N, D) <= device_lds_limit();
    ctx->merged = slice_fits && (!ctx->dv.bosonic || wide);
    ctx->split = ctx->merged && prm->thermostat <= PIMDB_THERMO_LANGEVIN &&
                 (P <= STEP_NM_MAXP || (prm->propagator == PIMDB_PROP_CARTESIAN &&
                                        (prm->thermostat == PIMDB_THERMO_NONE || !prm->nmthermostat)));
    ctx->small = ctx->split && prm->propagator == PIMDB_PROP_CARTESIAN && prm->int_kind != PIMDB_POT_AZIZ &&
                 N <= (ctx->dv.bosonic ? SMALL_RING : SMALL_N) && ctx->nbd <= SMALL_E && P <= STEP_NM_MAXP;
    if (ctx->merged && prm->thermostat >= PIMDB_THERMO_NOSE_HOOVER && !prm->nmthermostat &&
        prm->propagator == PIMDB_PROP_CARTESIAN) {
        const int groups = prm->thermostat == PIMDB_THERMO_NOSE_HOOVER ? 1 : prm->thermostat == PIMDB_THERMO_NOSE_HOOVER_NP ? N : N * D;
        const bool fits = sizeof(double) * nh_step_lds_doubles(N, D, prm->fixcom ? P : 1, ctx->dv.bosonic && N <= NH_EXT) + 1024 <=
                          device_lds_limit();
        // with zeroMomentum one workgroup: two chains a thread or beads a wave
        // in turn already cost more than the kernels they replace (nh_steps.hpp)
        const bool few = groups == 1 ? P <= NH_WAVES && ctx->nbd <= NH_THREADS : (size_t)P * groups <= NH_THREADS / 2;
        ctx->nh_whole = fits && (!prm->fixcom || few);
        ctx->nh_close = !ctx->nh_whole && ctx->dv.bosonic && N <= NH_EXT / 2;
    }
    if (ctx->merged) {
        ctx->pg = plan_pair_groups(*prm, ctx->dv, wide ? xw_grid(N) : 0, D * step_noise_tiles(N));
        if (ctx->pg.G && ctx->pg.max_slots(P)) alloc(&ctx->pg.cpart, sizeof(double) * ctx->nbd * ctx->pg.max_slots(P));
    }
    if (ctx->merged && ctx->dv.bosonic) alloc(&ctx->xc, sizeof(double) * 4 * (size_t)D * N);
    if (ctx->split) {
        alloc(&ctx->H, sizeof(double) * ctx->nbd);
        alloc(&ctx->fpart, sizeof(double) * D * (size_t)P * ((N + FORCE_TILE - 1) / FORCE_TILE));
        alloc(&ctx->hpart, sizeof(double) * D * (size_t)step_noise_tiles(N));
    }
    alloc(&ctx->fex, sizeof(double) * 2 * (size_t)D * N);
    alloc(&ctx->C, sizeof(double) * (size_t)P * P);
    alloc(&ctx->CT, sizeof(double) * (size_t)P * P);
    alloc(&ctx->rot, sizeof(double) * 4 * (size_t)P);
    // partial momentum sums: one row per k_momenta tile, or per bead when the
    // Cartesian Nose-Hoover O-step (one workgroup per bead) produces them
    const bool nh = prm->thermostat >= PIMDB_THERMO_NOSE_HOOVER;
    ctx->ncom = (nh && !prm->nmthermostat) ? P : ctx->ntiles;
    alloc(&ctx->com0, sizeof(double) * (size_t)ctx->ncom * D);
    alloc(&ctx->com1, sizeof(double) * (size_t)ctx->ncom * D);
    if (nh) {
        NhArgs& h = ctx->nh;
        h.N = N; h.P = P; h.D = D; h.nc = prm->nchains;
        h.kind = prm->thermostat;
        h.groups = prm->thermostat == PIMDB_THERMO_NOSE_HOOVER ? 1 : prm->thermostat == PIMDB_THERMO_NOSE_HOOVER_NP ? N : N * D;
        const int ndof = prm->thermostat == PIMDB_THERMO_NOSE_HOOVER ? D * N : prm->thermostat == PIMDB_THERMO_NOSE_HOOVER_NP ? D : 1;
        h.mass = prm->mass; h.dt = prm->dt;
        h.thermo_beta = ctx->dv.thermo_beta;   // beta / P
        h.Qi = 1.0 * 1.0 * ctx->dv.beta / P;    // hbar^2 beta / P, nose_hoover.cpp:17
        h.Q1 = ndof * h.Qi;
        h.required = ndof / h.thermo_beta;
        const size_t nch = (size_t)P * h.groups * h.nc;
        alloc(&h.eta, sizeof(double) * nch);
        alloc(&h.eta_dot, sizeof(double) * nch);
        alloc(&h.eta_dot_dot, sizeof(double) * nch);
        if (prm->nmthermostat) alloc(&ctx->modes, sizeof(double) * ctx->nbd);
    }
    alloc(&ctx->obs, sizeof(double) * obs_doubles(N, P));
    alloc(&ctx->ctr, sizeof(unsigned long long));
    if (hipMalloc((void**)&ctx->arena, arena) != hipSuccess || hipMemset(ctx->arena, 0, arena) != hipSuccess)
        rc = ctx->fail(PIMDB_E_HIP, "device allocation failed");
    if (!rc)
        for (auto& w : want) *w.first = ctx->arena + w.second;
    if (!rc && wide && hipMemset(ctx->pub, 0xFF, 8 * xw_pub_words(N)) != hipSuccess)
        rc = ctx->fail(PIMDB_E_HIP, "device initialisation failed");
    if (!rc && !(ctx->status = status_pool().take())) rc = ctx->fail(PIMDB_E_HIP, "pinned allocation failed");
    if (!rc && (hipStreamCreateWithFlags(&ctx->s0, hipStreamNonBlocking) != hipSuccess ||
                hipEventCreate(&ctx->t0) != hipSuccess || hipEventCreate(&ctx->t1) != hipSuccess))
        rc = ctx->fail(PIMDB_E_HIP, "stream/event creation failed");
    // the second stream of steps whose recursions are a kernel of their own
    if (!rc && ring && !ctx->merged &&
        (hipStreamCreateWithFlags(&ctx->s1, hipStreamNonBlocking) != hipSuccess ||
         hipEventCreateWithFlags(&ctx->ev_fork, hipEventDisableTiming) != hipSuccess ||
         hipEventCreateWithFlags(&ctx->ev_join, hipEventDisableTiming) != hipSuccess))
        rc = ctx->fail(PIMDB_E_HIP, "stream/event creation failed");
    if (!rc) {
        std::vector<double> C0((size_t)P * P), CT0((size_t)P * P), Cm((size_t)P * P), CTm((size_t)P * P),
            rot(4 * (size_t)P);
        nm_matrices(P, C0.data(), CT0.data());
        transpose_square(P, C0.data(), Cm.data());    // device holds C^T: [j][k]
        transpose_square(P, CT0.data(), CTm.data());  // and CT^T: [k][b]
        nm_rotation(*prm, ctx->dv, rot.data());
        if (hipMemcpy(ctx->C, Cm.data(), sizeof(double) * Cm.size(), hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(ctx->CT, CTm.data(), sizeof(double) * CTm.size(), hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(ctx->rot, rot.data(), sizeof(double) * rot.size(), hipMemcpyHostToDevice) != hipSuccess)
            rc = ctx->fail(PIMDB_E_HIP, "upload of normal-mode tables failed");
    }
    if (!rc && ctx->dv.bosonic && prm->exchange_algo == PIMDB_EXCHANGE_FACTORIAL &&
        sizeof(double) * factorial_lds_doubles(N, D) > device_lds_limit())
        rc = ctx->fail(PIMDB_E_ARG, "natoms too large for the factorial exchange workgroup");
    if (rc) {
        set_create_error(ctx->err);
        pimdb_ctx_destroy(ctx);
        return rc;
    }
    *out = ctx;
    return PIMDB_OK;
}

void pimdb_ctx_destroy(pimdb_ctx* ctx) {
    if (!ctx) return;
    if (ctx->s0) (void)hipStreamSynchronize(ctx->s0);
    if (ctx->s1) (void)hipStreamSynchronize(ctx->s1);
    if (ctx->gexec) (void)hipGraphExecDestroy(ctx->gexec);
    if (ctx->graph) (void)hipGraphDestroy(ctx->graph);
    void* bufs[] = {ctx->arena, ctx->E, ctx->ET, ctx->prob, ctx->noise};
    for (void* b : bufs)
        if (b) (void)hipFree(b);
    status_pool().give(ctx->status);
    if (ctx->pinned) (void)hipHostFree(ctx->pinned);
    if (ctx->ev_fork) (void)hipEventDestroy(ctx->ev_fork);
    if (ctx->ev_join) (void)hipEventDestroy(ctx->ev_join);
    if (ctx->t0) (void)hipEventDestroy(ctx->t0);
    if (ctx->t1) (void)hipEventDestroy(ctx->t1);
    if (ctx->s0) (void)hipStreamDestroy(ctx->s0);
    if (ctx->s1) (void)hipStreamDestroy(ctx->s1);
    delete ctx;
}

const char* pimdb_last_error(const pimdb_ctx* ctx) { return ctx ? ctx->err.c_str() : create_error(); }

int pimdb_test_lost_wait(pimdb_ctx* ctx) {
    if (!ctx) return PIMDB_E_ARG;
    CK(fill_published(ctx->pub, xw_pub_words(ctx->N), ctx->s0));
    *(volatile int*)ctx->status = LOST_WAIT;
    return check_status(ctx);
}

int pimdb_set_state(pimdb_ctx* ctx, const double* x, const double* p) {
    if (!ctx) return PIMDB_E_ARG;
    const double* src[2] = {x, p};
    double* dst[2] = {ctx->x, ctx->p};
    StateArrays a{{nullptr, nullptr, nullptr}, 0, ctx->N, ctx->D, ctx->nbd, nullptr, 0};
    double* host[3];
    for (int k = 0; k < 2; ++k)
        if (src[k]) {
            host[a.count] = const_cast<double*>(src[k]);
            a.dev[a.count++] = dst[k];
        }
    if (a.count) CK(copy_state<true>(a, host, ctx->s0));
    return PIMDB_OK;
}

int pimdb_get_state(pimdb_ctx* ctx, double* x, double* p, double* f) {
    if (!ctx) return PIMDB_E_ARG;
    double* dst[3] = {x, p, f};
    double* src[3] = {ctx->x, ctx->p, ctx->f};
    StateArrays a{{nullptr, nullptr, nullptr}, 0, ctx->N, ctx->D, ctx->nbd, nullptr, 0};
    double* host[3];
    for (int k = 0; k < 3; ++k)
        if (dst[k]) {
            host[a.count] = dst[k];
            a.dev[a.count++] = src[k];
        }
    if (a.count) CK(copy_state<false>(a, host, ctx->s0));
    return PIMDB_OK;
}

int pimdb_forces(pimdb_ctx* ctx) {
    if (!ctx) return PIMDB_E_ARG;
    int rc = enqueue_forces(ctx);
    if (rc) return rc;
    return check_status(ctx);
}

int pimdb_exchange_forward(pimdb_ctx* ctx, double* VB, double* V, double* Vb, double* prob, double* E) {
    if (!ctx) return PIMDB_E_ARG;
    if (!ctx->dv.bosonic) return ctx->fail(PIMDB_E_STATE, "exchange requires bosonic=true and nbeads > 1");
    const int N = ctx->N;
    if (factorial(ctx)) {
        if (V || Vb || prob || E)
            return ctx->fail(PIMDB_E_ARG, "the factorial exchange has no V, Vb, E or connection probabilities");
        launch_factorial(ctx, ctx->s0, nullptr, nullptr, ctx->V + N, nullptr);
        CK(hipGetLastError());
        const int rc = check_status(ctx);   // waits for the stream
        if (rc) return rc;
        if (VB) CK(hipMemcpy(VB, ctx->V + N, sizeof(double), hipMemcpyDeviceToHost));
        return PIMDB_OK;
    }
    const size_t tri = (size_t)N * (N + 1) / 2;
    int rc = PIMDB_OK;
    if (prob || E) {
        rc = need_buffer(ctx, &ctx->E, tri);
        if (!rc) rc = need_buffer(ctx, &ctx->ET, tri);
    }
    if (!rc && prob) rc = need_buffer(ctx, &ctx->prob, (size_t)N * N);
    if (rc) return rc;
    launch_exchange_forward(ctx, ctx->s0);
    if (prob || E) launch_cycle_energies_ctx(ctx, ctx->s0);
    if (prob) {
        const size_t nn = (size_t)N * N;
        hipLaunchKernelGGL(k_exchange_probabilities, dim3((unsigned)((nn + 255) / 256)), dim3(256), 0, ctx->s0, N,
                           ctx->dv.bt, ctx->E, ctx->V, ctx->Vb, ctx->prob);
    }
    CK(hipGetLastError());
    rc = check_status(ctx);
    if (rc) return rc;
    if (VB) CK(hipMemcpy(VB, ctx->V + N, sizeof(double), hipMemcpyDeviceToHost));
    if (V) CK(hipMemcpy(V, ctx->V, sizeof(double) * (N + 1), hipMemcpyDeviceToHost));
    if (Vb) CK(hipMemcpy(Vb, ctx->Vb, sizeof(double) * (N + 1), hipMemcpyDeviceToHost));
    if (prob) CK(hipMemcpy(prob, ctx->prob, sizeof(double) * (size_t)N * N, hipMemcpyDeviceToHost));
    if (E) CK(hipMemcpy(E, ctx->E, sizeof(double) * (size_t)N * (N + 1) / 2, hipMemcpyDeviceToHost));
    return PIMDB_OK;
}

int pimdb_exchange_adjoint(pimdb_ctx* ctx, double* f_first, double* f_last) {
    if (!ctx) return PIMDB_E_ARG;
    if (!ctx->dv.bosonic) return ctx->fail(PIMDB_E_STATE, "exchange requires bosonic=true and nbeads > 1");
    if (factorial(ctx)) {
        launch_factorial(ctx, ctx->s0, nullptr, ctx->fex, nullptr, nullptr);
    } else {
        launch_exchange_forward(ctx, ctx->s0);
        launch_exchange_forces(ctx, ctx->s0, nullptr, ctx->fex);
    }
    CK(hipGetLastError());
    int rc = check_status(ctx);
    if (rc) return rc;
    const int N = ctx->N, D = ctx->D;
    std::vector<double> h(2 * (size_t)D * N);
    CK(hipMemcpy(h.data(), ctx->fex, sizeof(double) * h.size(), hipMemcpyDeviceToHost));
    for (int w = 0; w < 2; ++w) {
        double* dst = w == 0 ? f_first : f_last;
        if (!dst) continue;
        for (int i = 0; i < N; ++i)
            for (int a = 0; a < D; ++a) dst[(size_t)i * D + a] = h[((size_t)w * D + a) * N + i];
    }
    return PIMDB_OK;
}

int pimdb_step(pimdb_ctx* ctx, int nsteps, const double* host_noise) {
    if (!ctx || nsteps < 0) return PIMDB_E_ARG;
    const size_t per = 2 * ctx->nbd;   // noise of one step
    if (host_noise) {
        const int chunk = (int)std::max<size_t>(1, std::min<size_t>((size_t)nsteps, (64u << 20) / (per * 8) + 1));
        const size_t need = per * (size_t)chunk;
        if (ctx->noise_cap < need) {
            if (ctx->noise) (void)hipFree(ctx->noise);
            ctx->noise = nullptr;
            ctx->noise_cap = 0;
            CK(hipMalloc((void**)&ctx->noise, need * sizeof(double)));
            ctx->noise_cap = need;
        }
        for (int s0 = 0; s0 < nsteps; s0 += chunk) {
            const int n = std::min(chunk, nsteps - s0);
            CK(hipStreamSynchronize(ctx->s0));   // previous chunk's copy and kernels are done
            double* st = pinned_buffer(ctx, per * n);
            if (!st) return ctx->fail(PIMDB_E_HIP, "pinned allocation failed");
            for (size_t blk = 0; blk < 2 * (size_t)n; ++blk)
                to_soa(host_noise + ((size_t)s0 * 2 + blk) * ctx->nbd, st + blk * ctx->nbd, ctx->N, ctx->P, ctx->D);
            CK(hipMemcpyAsync(ctx->noise, st, sizeof(double) * per * n, hipMemcpyHostToDevice, ctx->s0));
            for (int s = 0; s < n; ++s) {
                const double* nz = ctx->noise + per * s;
                int rc = enqueue_step(ctx, nz, nz + ctx->nbd);
                if (rc) return rc;
            }
        }
    } else {
        const int rc = enqueue_steps(ctx, nsteps);
        if (rc) return rc;
    }
    int rc = finish_steps(ctx, host_noise != nullptr);
    if (rc) return rc;
    return check_status(ctx);
}

int pimdb_graph_capture(pimdb_ctx* ctx) {
    if (!ctx) return PIMDB_E_ARG;
    // A step of one stream is launched faster than its graph is replayed (N=256,
    // P=64 helium 36.9 against 41.1 us a step, N=8 Nose-Hoover 29.3 against
    // 31.9): only the two-stream steps are captured.
    if (ctx->gexec || ctx->merged || !ctx->dv.bosonic || factorial(ctx)) return PIMDB_OK;
    CK(hipStreamSynchronize(ctx->s0));
    CK(hipStreamBeginCapture(ctx->s0, hipStreamCaptureModeThreadLocal));
    int rc = enqueue_step(ctx, nullptr, nullptr);
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(ctx->s0, &g);
    if (rc) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    if (e != hipSuccess) return ctx->fail(PIMDB_E_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
    ctx->graph = g;
    CK(hipGraphInstantiate(&ctx->gexec, ctx->graph, nullptr, nullptr, 0));
    return PIMDB_OK;
}

int pimdb_observables(pimdb_ctx* ctx, double* out) {
    if (!ctx || !out) return PIMDB_E_ARG;
    const int N = ctx->N, P = ctx->P, D = ctx->D;
    const int nt = (N + FORCE_TILE - 1) / FORCE_TILE;
    const size_t tail = obs_tail(N, P), all = obs_doubles(N, P);
    double* est = ctx->obs + tail;
    const bool ring = ctx->dv.bosonic && !factorial(ctx);
    if (ring && !estimator_fits(N)) return ctx->fail(PIMDB_E_ARG, "natoms too large for the exchange estimators");
    if (ctx->merged) {
        switch (D) {
        case 1: launch_observe_d<1>(ctx); break;
        case 2: launch_observe_d<2>(ctx); break;
        default: launch_observe_d<3>(ctx); break;
        }
    } else {
        launch_bead_sums(D, N, P, ctx->dv.k, ctx->prm.pbc, ctx->prm.size, ctx->x, ctx->p, ctx->obs, ctx->s0);
        launch_bead_energies(D, ctx->prm, ctx->dv, ctx->x, ctx->obs + 2 * (size_t)P, ctx->s0);
        if (ring) launch_exchange_forward(ctx, ctx->s0);
    }
    if (ring) launch_estimators(ctx);
    if (factorial(ctx)) launch_factorial(ctx, ctx->s0, nullptr, nullptr, est + std::max(2 * N + 1, 4), est);
    if (ctx->prm.thermostat >= PIMDB_THERMO_NOSE_HOOVER) {
        const int ndof = ctx->nh.kind == PIMDB_THERMO_NOSE_HOOVER ? D * N : ctx->nh.kind == PIMDB_THERMO_NOSE_HOOVER_NP ? D : 1;
        hipLaunchKernelGGL(k_nh_energy, dim3(1), dim3(256), 0, ctx->s0, ctx->nh, ndof, ctx->obs + all - 1);
    }
    CK(hipGetLastError());
    std::vector<double> obs(all);
    CK(read_obs(ctx, 0, obs));
    const double* h = obs.data();
    int rc = check_status(ctx);
    if (rc) return rc;
    double prim[3] = {0.0, 0.0, 0.0}, VN = 0.0;
    if (ring) {
        combine_estimators(N, P, ctx->dv.bt, h + tail, prim);
        VN = h[tail + 2 * (size_t)N + 1];
    } else if (factorial(ctx)) {
        std::copy(h + tail, h + tail + 3, prim);
        VN = h[tail + std::max(2 * N + 1, 4)];
    }
    combine_observables(ctx->prm, ctx->dv, h, h + 2 * (size_t)P, nt, prim, VN, out);
    out[10] = ctx->prm.thermostat >= PIMDB_THERMO_NOSE_HOOVER ? h[all - 1] : 0.0;
    return PIMDB_OK;
}

int pimdb_exchange_estimators(pimdb_ctx* ctx, double* prim, double* prob_distinct, double* prob_longest) {
    if (!ctx) return PIMDB_E_ARG;
    if (!ctx->dv.bosonic) return ctx->fail(PIMDB_E_STATE, "exchange estimators need a bosonic system");
    const int N = ctx->N, P = ctx->P;
    const size_t tail = obs_tail(N, P);
    if (factorial(ctx)) {
        launch_factorial(ctx, ctx->s0, nullptr, nullptr, nullptr, ctx->obs + tail);
    } else {
        if (!estimator_fits(N)) return ctx->fail(PIMDB_E_ARG, "natoms too large for the exchange estimators");
        launch_exchange_forward(ctx, ctx->s0);
        launch_estimators(ctx);
    }
    CK(hipGetLastError());
    std::vector<double> est(obs_doubles(N, P) - tail);
    CK(read_obs(ctx, tail, est));
    const double* h = est.data();
    int rc = check_status(ctx);
    if (rc) return rc;
    double e[3];
    if (factorial(ctx)) std::copy(h, h + 3, e);
    else combine_estimators(N, P, ctx->dv.bt, h, e);
    if (prim) *prim = e[0];
    if (prob_distinct) *prob_distinct = e[1];
    if (prob_longest) *prob_longest = e[2];
    return PIMDB_OK;
}

}  // extern "C"

// Device time per repetition of `body`, from `reps` repetitions captured in
// one hipGraph and replayed on the context stream between two events (so
// host launch latency is not counted).
template <class F>
static int time_captured(pimdb_ctx* ctx, int reps, F body, double* ms_out) {
    hipGraph_t g = nullptr;
    hipGraphExec_t ge = nullptr;
    CK(hipStreamSynchronize(ctx->s0));
    CK(hipStreamBeginCapture(ctx->s0, hipStreamCaptureModeThreadLocal));
    int rc = PIMDB_OK;
    for (int r = 0; r < reps && !rc; ++r) rc = body();
    hipError_t e = hipStreamEndCapture(ctx->s0, &g);
    if (rc) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    if (e != hipSuccess) return ctx->fail(PIMDB_E_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
    e = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
    if (e != hipSuccess) {
        (void)hipGraphDestroy(g);
        return ctx->fail(PIMDB_E_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
    }
    float ms = 0.0f;
    (void)hipGraphLaunch(ge, ctx->s0);   // warm
    (void)hipEventRecord(ctx->t0, ctx->s0);
    (void)hipGraphLaunch(ge, ctx->s0);
    (void)hipEventRecord(ctx->t1, ctx->s0);
    e = hipEventSynchronize(ctx->t1);
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, ctx->t0, ctx->t1);
    (void)hipGraphExecDestroy(ge);
    (void)hipGraphDestroy(g);
    if (e != hipSuccess) return ctx->fail(PIMDB_E_HIP, std::string("graph timing: ") + hipGetErrorString(e));
    *ms_out = (double)ms / reps;
    return PIMDB_OK;
}

extern "C" {

int pimdb_time_kernels(pimdb_ctx* ctx, int reps, double* ms_forces, double* ms_exchange, double* ms_step) {
    if (!ctx || reps < 1) return PIMDB_E_ARG;
    int rc = PIMDB_OK;
    if (ms_forces) {
        // what a force evaluation launches, without the exchange
        rc = time_captured(ctx, reps, [&]() {
            if (ctx->merged) {
                launch_step_forces(ctx, true, false, STEP_CLOSE, false);
                launch_pair_sum(ctx);
            } else {
                launch_bead_forces(ctx, ctx->s0);
            }
            return PIMDB_OK;
        }, ms_forces);
        if (rc) return rc;
    }
    if (ms_exchange) {
        *ms_exchange = 0.0;
        if (ctx->dv.bosonic) {
            rc = time_captured(ctx, reps, [&]() {
                if (factorial(ctx)) {
                    launch_factorial(ctx, ctx->s0, nullptr, ctx->fex, nullptr, nullptr);
                } else {
                    launch_exchange_forward(ctx, ctx->s0);
                    launch_exchange_forces(ctx, ctx->s0, nullptr, ctx->fex);
                }
                return PIMDB_OK;
            }, ms_exchange);
            if (rc) return rc;
        }
    }
    if (ms_forces || ms_exchange) {
        // the force timing overwrote f with the physical and spring part
        // alone: the full forces of the current positions again
        rc = enqueue_forces(ctx);
        if (rc) return rc;
    }
    if (ms_step) {
        // whole steps (device noise), as pimdb_step launches them; this advances
        // the state by 2 * reps steps
        hipGraphExec_t held = ctx->gexec;   // (a graph is not launched into a capture)
        ctx->gexec = nullptr;
        rc = time_captured(ctx, 1, [&]() { return enqueue_steps(ctx, reps); }, ms_step);
        ctx->gexec = held;
        if (rc) return rc;
        *ms_step /= reps;
        rc = finish_steps(ctx, false);
        if (rc) return rc;
    }
    CK(hipGetLastError());
    return check_status(ctx);
}

}  // extern "C"
