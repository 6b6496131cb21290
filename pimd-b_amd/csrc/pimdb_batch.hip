// pimdb_batch.hip -- C ABI of the batched persistent form (include/pimdb_gpu.h):
// replicas of uneven N, P and T in one persistent kernel per MD step,
// replayed from a hipGraph, with the workgroup size and residency chosen by a
// small autotuner.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <numeric>
#include <queue>
#include <string>
#include <vector>

#include "pimdb_gpu.h"
#include "batch.hpp"
#include "batch_split.hpp"
#include "ctx_common.hpp"

using namespace pimdb;

struct pimdb_batch {
    std::vector<pimdb_params> prm;
    std::vector<RepDesc> desc;
    int R = 0, D = 3, kind = 0;
    int threads = 1024, resident = 0;   // resident workgroups (0: all CUs)
    int cus = 0;
    int per_cu = 1;                     // workgroups that share one CU's LDS
    size_t nx = 0, nV = 0, nC = 0, nR = 0, nH = 0;
    double* d_fx = nullptr;             // physical forces of normal-mode-propagator replicas
    double* d_rot = nullptr;            // their rotation tables
    double* d_nh = nullptr;             // Nose-Hoover chain states: eta, eta_dot, eta_dot_dot
    double* d_modes = nullptr;          // normal modes of Nose-Hoover replicas with normal-mode coupling
    double* d_xws = nullptr;            // exchange workspaces in device memory (RepDesc::xws)
    size_t xws_cap = 0;                 // doubles held by d_xws
    size_t lds = 0;
    BatchPtrs bp{};
    RepDesc* d_desc = nullptr;
    int *d_sched = nullptr, *d_sched_off = nullptr;
    int grid = 0;
    hipStream_t s = nullptr;
    hipEvent_t t0 = nullptr, t1 = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    bool fused_any = false;       // some replica takes the fused normal-mode path
    bool nmprop_any = false;      // some replica takes the normal-mode propagator
    bool nh_any = false;          // some replica takes Nose-Hoover chains
    bool xdev_any = false;        // some replica's exchange workspace is in device memory
    bool ext_any = false;         // any of the three: the EXT kernels
    bool maybe_pending = false;   // a step ran since the last finishing launch
    bool unsettled = false;       // cmp may hold what the two-kernel form does not keep (BatchPtrs)
    // the two-kernel form (batch_split.hpp)
    bool split = false;           // steps run in it
    SplitPtrs sp{};
    std::vector<StepArgs> hsteps;
    double* d_split = nullptr;    // its workspace
    unsigned long long* d_pub = nullptr;   // the recursions' published values of all replicas
    size_t npub = 0;
    StepArgs* d_steps = nullptr;
    int2* d_maps = nullptr;
    std::string err;
    int fail(int code, const std::string& m) {
        err = m;
        return code;
    }
};

#define BCK(expr)                                                                                    \
    do {                                                                                             \
        hipError_t e_ = (expr);                                                                      \
        if (e_ != hipSuccess) return b->fail(PIMDB_E_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

// Cost estimates in microseconds, fitted to 800 random batches (N = 3 .. 300, P = 2 .. 64, 2 .. 2000 replicas, every pair kind and
// dimension; rings mostly without exchange, which costs the two-kernel form up to
// a third more): 0.7 - 1.3 of the measured times in nine of ten.
//
// Steps of the pair walk (two rows per lane) over one slice; a step's cost in
// units of `us`, per axis where the pair's arithmetic is short.
static double walk_steps(const pimdb_params& p) {
    const int T = (p.natoms + PTILE - 1) / PTILE;
    return 17.0 * T + PTILE / 4 * T * (T - 1);
}
static double walk_us(const pimdb_params& p, double harmonic, double dipole, double aziz) {
    const double us = p.int_kind == PIMDB_POT_HARMONIC ? harmonic * p.ndim : p.int_kind == PIMDB_POT_DIPOLE ? dipole * p.ndim :
                      p.int_kind == PIMDB_POT_AZIZ ? aziz : 0.0;
    return us * walk_steps(p);
}
// A replica's step on a compute unit in the persistent kernel, with 16 waves a
// workgroup or less (two workgroups of 8 waves a unit).  The beads take the waves
// in whole rounds.
static double rep_cost(const pimdb_params& p, int waves) {
    const double N = p.natoms, P = p.nbeads, T = (p.natoms + PTILE - 1) / PTILE;
    const double rounds = (double)((p.nbeads + waves - 1) / waves) * waves;
    const bool ring = p.bosonic && p.nbeads > 1;
    if (waves >= 16)
        return 26.0 + 0.0057 * N * P * p.ndim + (p.nmthermostat ? 0.0013 * P * p.ndim * PTILE * T : 0.0) +
               (ring ? 11.0 + 8.0 * T + 1e-4 * N * N : 0.0) + rounds * walk_us(p, 0.0062, 0.0093, 0.052);
    return 14.0 + 0.0075 * N * P * p.ndim + (ring ? 6.0 + 5.3 * T + 2.4e-4 * N * N : 0.0) +
           rounds * walk_us(p, 0.0055, 0.0089, 0.059);
}
// The same in the two-kernel form.  N^2: the exterior forces.
static double rep_cost_split(const pimdb_params& p) {
    const double N = p.natoms, P = p.nbeads, T = (p.natoms + PTILE - 1) / PTILE;
    return 0.008 * N * P * p.ndim + (p.nmthermostat ? 0.0012 * P * p.ndim * PTILE * T : 0.0) +
           (p.bosonic && p.nbeads > 1 ? 7.5 * T + 2.8e-3 * N * N : 0.0) + 0.08 * P * T + 1.7 * p.ndim * T +
           P * walk_us(p, 0.006, 0.0098, 0.077);
}

// Longest-processing-time-first assignment of replicas to `grid` workgroups.
static void build_schedule(pimdb_batch* b, std::vector<int>& sched, std::vector<int>& off) {
    std::vector<int> order(b->R);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(),
                     [&](int a, int c) { return rep_cost(b->prm[a], b->threads / WAVE) > rep_cost(b->prm[c], b->threads / WAVE); });
    using Item = std::pair<double, int>;
    std::priority_queue<Item, std::vector<Item>, std::greater<Item>> heap;
    for (int g = 0; g < b->grid; ++g) heap.push({0.0, g});
    std::vector<std::vector<int>> lists(b->grid);
    for (int r : order) {
        Item it = heap.top();
        heap.pop();
        lists[it.second].push_back(r);
        heap.push({it.first + rep_cost(b->prm[r], b->threads / WAVE), it.second});
    }
    sched.clear();
    off.assign(1, 0);
    for (auto& l : lists) {
        sched.insert(sched.end(), l.begin(), l.end());
        off.push_back((int)sched.size());
    }
}

// LDS plan of every replica for `threads` threads per workgroup and
// `per_cu` workgroups per compute unit (each then gets 1/per_cu of its LDS):
// whether the pair forces of every wave's slice stay in LDS, how many chunk
// slots the exchange's backward pass gets, and the largest need.  A replica
// whose exchange layout does not fit even with one chunk slot gets its
// workspace in device memory instead (one slot per wave; its size in doubles
// into (*xdev)[r], 0 for the others).  Returns the dynamic LDS bytes, or 0
// (with *why) when some replica does not fit.
static size_t plan_lds(pimdb_batch* b, int threads, int per_cu, std::vector<RepDesc>& desc, std::string* why,
                       std::vector<size_t>* xdev = nullptr) {
    const size_t budget = device_lds_limit() / (size_t)per_cu / sizeof(double);   // doubles
    const size_t avail = budget > 16 ? budget - 16 : 0;                             // after the reduction slots
    const int nw = threads / WAVE;
    size_t need = 0;
    for (int r = 0; r < b->R; ++r) {
        const pimdb_params& p = b->prm[r];
        const int N = p.natoms, D = p.ndim;
        RepDesc& d = desc[r];
        d.xslots = 1;
        if (xdev) (*xdev)[r] = 0;
        if (d.bosonic) {
            // the exchange's layout with as many chunk slots (up to one per
            // wave) as fit
            if (N > XB_MAXPER * threads) {
                *why = "replica " + std::to_string(r) + ": natoms above " + std::to_string(XB_MAXPER) +
                       " per thread of a batched workgroup";
                return 0;
            }
            int slots = nw;
            size_t x = (size_t)xb_layout(N, D, nw, slots).total;
            while (slots > 1 && x > avail) x = (size_t)xb_layout(N, D, nw, --slots).total;
            if (x > avail) {   // the workspace in device memory
                slots = nw;
                if (xdev) (*xdev)[r] = (size_t)xb_layout(N, D, nw, slots).total;
                x = 0;
            }
            d.xslots = slots;
            need = std::max(need, x);
        }
        size_t nm = batch_nm_lds_doubles(p.nbeads, nw);
        if (d.nmprop) nm = std::max(nm, 4 * (size_t)p.nbeads * NMD_TC);   // wg_nm_drift's tiles
        if (p.thermostat >= PIMDB_THERMO_NOSE_HOOVER && p.nmthermostat)
            nm = std::max(nm, (size_t)p.nbeads * NMD_TC);                 // wg_nh_ostep's tiles
        if (nm > avail) {
            *why = "replica " + std::to_string(r) + ": nbeads too large for the batched workgroup";
            return 0;
        }
        need = std::max(need, nm);
        // pair forces of every wave's slice in LDS when they fit (+ the tile
        // order and its inverse, N ints each)
        const size_t pl = (size_t)nw * pair_fstride(D) * N + N;
        d.plds = pl <= avail ? 1 : 0;
        if (d.plds) need = std::max(need, pl);
    }
    return sizeof(double) * (16 + need);
}

// The largest load of a compute unit (us) in a schedule of the persistent
// kernel over the card, and the longest replica's.
static double makespan(const pimdb_batch* b, int waves, double* longest = nullptr) {
    std::vector<double> c;
    for (const pimdb_params& p : b->prm) c.push_back(rep_cost(p, waves));
    std::sort(c.rbegin(), c.rend());
    if (longest) *longest = c[0];
    std::priority_queue<double, std::vector<double>, std::greater<double>> heap;
    for (int g = 0; g < std::min(b->R, b->cus); ++g) heap.push(0.0);
    double most = 0.0;
    for (double x : c) {
        const double t = heap.top() + x;
        heap.pop();
        heap.push(t);
        most = std::max(most, t);
    }
    return most;
}

static int upload_schedule(pimdb_batch* b) {
    const int resident = b->resident > 0 ? b->resident : b->cus;
    b->grid = std::max(1, std::min(b->R, resident));
    // the LDS is planned for the residency asked for (each CU's share)
    b->per_cu = (resident + b->cus - 1) / b->cus;
    {
        std::vector<RepDesc> desc = b->desc;
        std::string why;
        std::vector<size_t> xdev(b->R, 0);
        const size_t lds = plan_lds(b, b->threads, b->per_cu, desc, &why, &xdev);
        if (!lds) return b->fail(PIMDB_E_ARG, why);
        // the device-memory exchange workspaces of this plan
        size_t total = 0;
        for (size_t n : xdev) total += n;
        if (total > b->xws_cap) {
            BCK(hipStreamSynchronize(b->s));
            if (b->d_xws) (void)hipFree(b->d_xws);
            b->d_xws = nullptr;
            b->xws_cap = 0;
            BCK(hipMalloc((void**)&b->d_xws, total * sizeof(double)));
            b->xws_cap = total;
        }
        size_t o = 0;
        for (int r = 0; r < b->R; ++r) {
            if (desc[r].bosonic) desc[r].xws = xdev[r] ? b->d_xws + o : nullptr;   // (fx is the nmprop one's)
            o += xdev[r];
        }
        b->xdev_any = total > 0;
        b->ext_any = b->nmprop_any || b->nh_any || b->xdev_any;
        b->desc = desc;
        b->lds = lds;
        if (b->d_desc)
            BCK(hipMemcpy(b->d_desc, b->desc.data(), sizeof(RepDesc) * b->R, hipMemcpyHostToDevice));
    }
    std::vector<int> sched, off;
    build_schedule(b, sched, off);
    if (b->d_sched) (void)hipFree(b->d_sched);
    if (b->d_sched_off) (void)hipFree(b->d_sched_off);
    b->d_sched = nullptr;
    b->d_sched_off = nullptr;
    BCK(hipMalloc((void**)&b->d_sched, sizeof(int) * sched.size()));
    BCK(hipMalloc((void**)&b->d_sched_off, sizeof(int) * off.size()));
    BCK(hipMemcpy(b->d_sched, sched.data(), sizeof(int) * sched.size(), hipMemcpyHostToDevice));
    BCK(hipMemcpy(b->d_sched_off, off.data(), sizeof(int) * off.size(), hipMemcpyHostToDevice));
    b->bp.sched = b->d_sched;
    b->bp.sched_off = b->d_sched_off;
    if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    b->gexec = nullptr;
    b->graph = nullptr;
    return PIMDB_OK;
}

template <int D, int KIND>
static void launch_batch_dk(pimdb_batch* b, int mode) {
    dim3 grid(b->grid), block(b->threads);
    if (b->ext_any && (mode == BM_STEP || mode == BM_FORCES || mode == BM_INTEGRATOR || mode == BM_EXCHANGE)) {
        switch (mode) {
        case BM_STEP: hipLaunchKernelGGL((k_batch_step<D, KIND, BM_STEP, true>), grid, block, b->lds, b->s, b->bp); break;
        case BM_FORCES: hipLaunchKernelGGL((k_batch_step<D, KIND, BM_FORCES, true>), grid, block, b->lds, b->s, b->bp); break;
        case BM_EXCHANGE: hipLaunchKernelGGL((k_batch_step<D, KIND, BM_EXCHANGE, true>), grid, block, b->lds, b->s, b->bp); break;
        default: hipLaunchKernelGGL((k_batch_step<D, KIND, BM_INTEGRATOR, true>), grid, block, b->lds, b->s, b->bp); break;
        }
        return;
    }
    switch (mode) {
    case BM_STEP: hipLaunchKernelGGL((k_batch_step<D, KIND, BM_STEP>), grid, block, b->lds, b->s, b->bp); break;
    case BM_FORCES: hipLaunchKernelGGL((k_batch_step<D, KIND, BM_FORCES>), grid, block, b->lds, b->s, b->bp); break;
    case BM_PAIRS: hipLaunchKernelGGL((k_batch_step<D, KIND, BM_PAIRS>), grid, block, b->lds, b->s, b->bp); break;
    case BM_EXCHANGE: hipLaunchKernelGGL((k_batch_step<D, KIND, BM_EXCHANGE>), grid, block, b->lds, b->s, b->bp); break;
    case BM_FINISH: hipLaunchKernelGGL((k_batch_step<D, KIND, BM_FINISH>), grid, block, b->lds, b->s, b->bp); break;
    default: hipLaunchKernelGGL((k_batch_step<D, KIND, BM_INTEGRATOR>), grid, block, b->lds, b->s, b->bp); break;
    }
}

template <int D>
static void launch_batch_d(pimdb_batch* b, int mode) {
    switch (b->kind) {
    case POT_HARMONIC: launch_batch_dk<D, POT_HARMONIC>(b, mode); break;
    case POT_DIPOLE: launch_batch_dk<D, POT_DIPOLE>(b, mode); break;
    case POT_AZIZ: launch_batch_dk<D, POT_AZIZ>(b, mode); break;
    default: launch_batch_dk<D, POT_FREE>(b, mode); break;
    }
}

static int launch_batch(pimdb_batch* b, int mode) {
    switch (b->D) {
    case 1: launch_batch_d<1>(b, mode); break;
    case 2: launch_batch_d<2>(b, mode); break;
    default: launch_batch_d<3>(b, mode); break;
    }
    BCK(hipGetLastError());
    return PIMDB_OK;
}

// Whether every replica can take the two-kernel form: Langevin or no
// thermostat, the Cartesian propagator, and parts that fit the LDS.
static bool split_able(const pimdb_batch* b) {
    const size_t lim = device_lds_limit();
    for (int r = 0; r < b->R; ++r) {
        const pimdb_params& p = b->prm[r];
        const bool nm = p.thermostat == PIMDB_THERMO_LANGEVIN && p.nmthermostat;
        if (p.thermostat > PIMDB_THERMO_LANGEVIN || p.propagator != PIMDB_PROP_CARTESIAN) return false;
        if (nm && p.nbeads > STEP_NM_MAXP) return false;
        if (b->desc[r].bosonic && xw_lds_bytes(p.natoms, p.ndim, SPLIT_THREADS) > lim) return false;
        if (sizeof(double) * step_noise_lds_doubles<SPLIT_THREADS>(p.nbeads, nm) > lim) return false;
    }
    return true;
}

static void free_split(pimdb_batch* b) {
    if (b->d_split) (void)hipFree(b->d_split);
    if (b->d_pub) (void)hipFree(b->d_pub);
    if (b->d_steps) (void)hipFree(b->d_steps);
    if (b->d_maps) (void)hipFree(b->d_maps);
    b->d_split = nullptr;
    b->d_pub = nullptr;
    b->d_steps = nullptr;
    b->d_maps = nullptr;
}

// About how long a slice and a noise workgroup of the two-kernel form take (a
// walk step of one of twelve waves on a compute unit, two draws per four beads).
static double slice_wg_us(const pimdb_params& p, int share) {
    const double us = p.int_kind == PIMDB_POT_FREE ? 0.0 : p.int_kind == PIMDB_POT_AZIZ ? 0.06 : 0.018;
    return 3.0 + 12.0 * us * walk_steps(p) / share;
}
static double noise_wg_us(const pimdb_params& p) { return 2.0 + 0.2 * p.nbeads; }

static int build_split_buffers(pimdb_batch* b) {
    const int D = b->D;
    std::vector<size_t> off;
    size_t nd = 0, nw = 0;
    for (int r = 0; r < b->R; ++r) {
        const pimdb_params& p = b->prm[r];
        const size_t N = p.natoms, P = p.nbeads;
        off.push_back(nd);
        nd += 4 * D * N + (N + 1) + 2 * N + P * D * N + P * SPLIT_WAVES * D + D * (size_t)step_noise_tiles(p.natoms);
        if (b->desc[r].bosonic) nw += xw_pub_words(p.natoms);
    }
    BCK(hipMalloc((void**)&b->d_split, nd * sizeof(double)));
    b->npub = nw;
    if (nw) {
        BCK(hipMalloc((void**)&b->d_pub, nw * 8));
        BCK(hipMemset(b->d_pub, 0xFF, nw * 8));
    }
    // waves per slice: enough of them for two per SIMD (8 per compute unit), where
    // the slices alone are fewer and their force arrays fit the LDS
    size_t beads = 0;
    bool fit = true;
    for (const pimdb_params& p : b->prm) {
        beads += p.nbeads;
        fit = fit && split_slice_lds(p.natoms, D) <= device_lds_limit();
    }
    int share = 1;
    while (fit && share < SPLIT_WAVES && beads * share < 8 * (size_t)b->cus) share *= 2;
    using Work = std::pair<double, int2>;
    std::vector<Work> rest;      // slices and noise, the longest first
    std::vector<int2> maps[4];   // forces, noise, full, open
    size_t lds = 0, w = 0;
    b->hsteps.clear();
    for (int r = 0; r < b->R; ++r) {
        const pimdb_params& p = b->prm[r];
        const RepDesc& d = b->desc[r];
        const Derived dv = derive(p);
        const size_t N = p.natoms, P = p.nbeads;
        StepArgs a{};
        a.fa = make_force_args(p, dv);
        a.bt = dv.bt;
        a.thermostat = p.thermostat; a.nm = p.nmthermostat; a.fixcom = p.fixcom;
        a.x = b->bp.x + d.off_x; a.p = b->bp.p + d.off_x; a.f = b->bp.f + d.off_x;
        a.V = b->bp.V + d.off_V;
        double* q = b->d_split + off[r];
        a.xc = q; q += 4 * D * N;
        a.Vb = q; q += N + 1;
        a.Shi = q; q += N;
        a.Slo = q; q += N;
        a.H = q; q += P * D * N;
        a.fpart = p.ext_kind != PIMDB_POT_FREE && p.fixcom ? q : nullptr; q += P * SPLIT_WAVES * D;
        a.hpart = q;
        a.frows = p.nbeads * share;
        a.pub = d.bosonic ? b->d_pub + w : nullptr;
        if (d.bosonic) w += xw_pub_words(p.natoms);
        a.status = b->bp.status + r;
        a.c1 = a.thermostat ? dv.c1 : 1.0;
        a.c2 = dv.c2;
        a.half_dt = 0.5 * p.dt;
        a.dt_m = p.dt / p.mass;
        a.CTt = b->bp.CTt + d.off_C;
        a.ctr = b->bp.ctl;
        a.seed = p.seed;
        b->hsteps.push_back(a);
        const int nx = d.bosonic ? xw_grid(p.natoms) : 0, ns = split_slices(p.nbeads, share), nn = step_noise_groups(a, D);
        for (int i = 0; i < nx; ++i) maps[0].push_back(int2{r, i});
        for (int i = nx; i < nx + nn; ++i) rest.push_back({noise_wg_us(p), int2{r, i}});
        for (int i = 0; i < ns; ++i) rest.push_back({slice_wg_us(p, share), int2{r, nx + nn + i}});
        for (int i = 0; i < nn; ++i) maps[1].push_back(int2{r, i});
        for (int i = 0; i < step_integrate_groups(a.fa, D, STEP_FULL); ++i) maps[2].push_back(int2{r, i});
        for (int i = 0; i < step_integrate_groups(a.fa, D, STEP_OPEN); ++i) maps[3].push_back(int2{r, i});
        if (d.bosonic) lds = std::max(lds, xw_lds_bytes(p.natoms, D, SPLIT_THREADS));
        const size_t sl = split_slice_lds(p.natoms, D);
        if (sl <= device_lds_limit()) lds = std::max(lds, sl);
        lds = std::max(lds, sizeof(double) * step_noise_lds_doubles<SPLIT_THREADS>(p.nbeads, a.thermostat && a.nm));
    }
    std::stable_sort(rest.begin(), rest.end(), [](const Work& a, const Work& c) { return a.first > c.first; });
    for (const Work& v : rest) maps[0].push_back(v.second);
    size_t nm = 0;
    for (auto& m : maps) nm += m.size();
    BCK(hipMalloc((void**)&b->d_maps, nm * sizeof(int2)));
    BCK(hipMalloc((void**)&b->d_steps, b->R * sizeof(StepArgs)));
    int2* at = b->d_maps;
    const int2* ptr[4];
    for (int k = 0; k < 4; ++k) {
        if (!maps[k].empty()) BCK(hipMemcpy(at, maps[k].data(), maps[k].size() * sizeof(int2), hipMemcpyHostToDevice));
        ptr[k] = at;
        at += maps[k].size();
    }
    BCK(hipMemcpy(b->d_steps, b->hsteps.data(), b->R * sizeof(StepArgs), hipMemcpyHostToDevice));
    BCK(hipStreamSynchronize(nullptr));
    b->sp.steps = b->d_steps;
    b->sp.forces_map = ptr[0]; b->sp.nforces = (int)maps[0].size();
    b->sp.noise_map = ptr[1]; b->sp.nnoise = (int)maps[1].size();
    b->sp.full_map = ptr[2]; b->sp.nfull = (int)maps[2].size();
    b->sp.open_map = ptr[3]; b->sp.nopen = (int)maps[3].size();
    b->sp.lds = lds;
    b->sp.share = share;
    return PIMDB_OK;
}

// The two-kernel form's workspace and maps (allocated once).
static int build_split(pimdb_batch* b) {
    if (b->d_steps) return PIMDB_OK;
    const int rc = build_split_buffers(b);
    if (rc) {
        (void)hipGetLastError();
        free_split(b);
    }
    return rc;
}

static int finish_pending(pimdb_batch* b);

// nsteps steps in the two-kernel form; the state is complete afterwards.
static int enqueue_split(pimdb_batch* b, int nsteps) {
    if (nsteps < 1) return PIMDB_OK;
    if (b->unsettled) {   // p from the persistent kernel: its owed half step, then its pending COM momentum
        const int rc = finish_pending(b);
        if (rc) return rc;
        BCK(launch_split_settle(b->bp, b->D, b->R, b->s));
        b->unsettled = false;
    }
    b->sp.bp = b->bp;
    BCK(launch_split_forces(b->sp, b->D, b->kind, false, STEP_OPEN, b->s));
    BCK(launch_split_integrate(b->sp, b->D, STEP_OPEN, b->s));
    for (int s = 1; s <= nsteps; ++s) {
        const int mode = s < nsteps ? STEP_FULL : STEP_CLOSE;
        BCK(launch_split_forces(b->sp, b->D, b->kind, true, mode, b->s));
        BCK(launch_split_integrate(b->sp, b->D, mode, b->s));
    }
    return PIMDB_OK;
}

static int capture(pimdb_batch* b);

// nsteps steps of every replica on the batch's stream, in its current form.
static int enqueue_batch_steps(pimdb_batch* b, int nsteps) {
    if (b->split) return enqueue_split(b, nsteps);
    const int rc = capture(b);
    if (rc) return rc;
    for (int s = 0; s < nsteps; ++s) BCK(hipGraphLaunch(b->gexec, b->s));
    if (nsteps > 0) b->maybe_pending = b->unsettled = true;
    return PIMDB_OK;
}

static int capture(pimdb_batch* b) {
    if (b->gexec) return PIMDB_OK;
    BCK(hipStreamSynchronize(b->s));
    BCK(hipStreamBeginCapture(b->s, hipStreamCaptureModeThreadLocal));
    int rc = launch_batch(b, BM_STEP);
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(b->s, &g);
    if (rc) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    if (e != hipSuccess) return b->fail(PIMDB_E_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
    b->graph = g;
    BCK(hipGraphInstantiate(&b->gexec, b->graph, nullptr, nullptr, 0));
    return PIMDB_OK;
}

static int check_batch_status(pimdb_batch* b) {
    std::vector<int> st(b->R);
    BCK(hipStreamSynchronize(b->s));
    BCK(hipMemcpy(st.data(), b->bp.status, sizeof(int) * b->R, hipMemcpyDeviceToHost));
    for (int r = 0; r < b->R; ++r) {
        if (st[r]) {
            bool lost = false;
            for (int s : st) lost = lost || lost_wait(s);
            BCK(hipMemset(b->bp.status, 0, sizeof(int) * b->R));
            BCK(empty_published(b->d_pub, b->npub, b->s));
            if (lost) return b->fail(PIMDB_E_HIP, LOST_WAIT_MESSAGE);
            return b->fail(PIMDB_E_NONFINITE, "non-finite bosonic exchange potential in replica " + std::to_string(r));
        }
    }
    return PIMDB_OK;
}

// Launch shape and form of a new batch, from the estimates above.
// More replicas than compute units: two workgroups of 512 threads per CU overlap
// each other's latencies (8 - 33% faster than one of 1024), where their LDS plan
// keeps every exchange workspace and force array in LDS and the longest replica,
// which 512 threads take longer for, does not bound the whole (312 uneven
// harmonic replicas of N <= 158, P <= 16: 185 us a step against 159).
// The two-kernel form where it is not estimated more than a twentieth longer
// than that.  Few replicas are many times faster in it (16 of helium, N=256,
// P=64: 122 against 1240 us a step; 256 of them 1486 against 1335), uneven ones
// faster (512 uneven dipole replicas 210 against 277), but hundreds of rings of
// more than 64 particles with few beads slower, since each block of a ring is a
// workgroup that waits (482 free ones of N=180, P=8: 233 against 100).  Of 600
// other random batches 18 were more than 8% slower than in the better form.
static int choose_form(pimdb_batch* b) {
    double longest = 0.0, persistent = makespan(b, 1024 / WAVE, &longest);
    if (b->R > b->cus && persistent > 1.3 * longest) {
        std::vector<RepDesc> one = b->desc, two = b->desc;
        std::vector<size_t> xdev(b->R, 0);
        std::string why;
        if (plan_lds(b, 1024, 1, one, &why) && plan_lds(b, 512, 2, two, &why, &xdev)) {
            bool same = true;
            for (int r = 0; r < b->R; ++r) same = same && !xdev[r] && two[r].plds == one[r].plds;
            if (same) {
                b->threads = 512;
                b->resident = 2 * b->cus;
                persistent = makespan(b, 512 / WAVE);
            }
        }
    }
    const int rc = upload_schedule(b);
    if (rc || !split_able(b)) return rc;
    double split = 0.0;
    int blocks = 0;   // of the longest ring: its chain
    for (int r = 0; r < b->R; ++r) {
        split += rep_cost_split(b->prm[r]);
        if (b->desc[r].bosonic) blocks = std::max(blocks, rec_blocks(b->prm[r].natoms));
    }
    b->split = 13.0 + 3.2 * blocks + split / b->cus < 1.05 * persistent;
    if (b->split && build_split(b) != PIMDB_OK) b->split = false;   // (no memory for its workspace)
    return PIMDB_OK;
}

extern "C" {

int pimdb_batch_create(const pimdb_params* reps, int nrep, pimdb_batch** out) {
    if (!reps || !out || nrep < 1) return PIMDB_E_ARG;
    *out = nullptr;
    std::string why;
    for (int r = 0; r < nrep; ++r) {
        if (!validate_params(reps[r], &why)) {
            set_create_error("replica " + std::to_string(r) + ": " + why);
            return PIMDB_E_ARG;
        }
        if (reps[r].bosonic && reps[r].exchange_algo != PIMDB_EXCHANGE_QUADRATIC) {
            set_create_error("batched replicas use the Feldman-Hirshberg exchange");
            return PIMDB_E_ARG;
        }
        if (reps[r].ndim != reps[0].ndim || reps[r].int_kind != reps[0].int_kind) {
            set_create_error("all replicas of a batch share ndim and the interaction kind");
            return PIMDB_E_ARG;
        }
    }
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) {
        set_create_error("no HIP device available");
        return PIMDB_E_HIP;
    }
    pimdb_batch* b = new pimdb_batch();
    b->R = nrep;
    b->D = reps[0].ndim;
    b->kind = reps[0].int_kind;
    b->prm.assign(reps, reps + nrep);
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) {
        delete b;
        set_create_error("hipGetDeviceProperties failed");
        return PIMDB_E_HIP;
    }
    b->cus = prop.multiProcessorCount;
    int Nmax = 1;
    std::vector<size_t> off_R, off_H;   // per replica: its block of the rotation tables and of the chains
    for (int r = 0; r < nrep; ++r) {
        const pimdb_params& p = reps[r];
        const Derived dv = derive(p);
        RepDesc d{};
        d.N = p.natoms; d.P = p.nbeads; d.bosonic = dv.bosonic; d.pbc = p.pbc;
        d.thermostat = p.thermostat; d.nm = p.nmthermostat; d.fixcom = p.fixcom;
        d.nmprop = p.propagator == PIMDB_PROP_NORMAL_MODES ? 1 : 0;   // (distinguishable only: validate_params)
        d.fused = (p.thermostat == PIMDB_THERMO_LANGEVIN && p.nmthermostat && p.nbeads <= NM_MFMA_MAXP &&
                   !d.nmprop) ? 1 : 0;
        if (d.fused) b->fused_any = true;
        d.L = p.size; d.invL = 1.0 / p.size; d.mass = p.mass; d.dt = p.dt;
        d.k = dv.k; d.bt = dv.bt; d.c1 = dv.c1; d.c2 = dv.c2;
        d.ext = dv.ext; d.int_k = dv.int_k; d.strength = p.int_strength; d.cutoff = dv.cutoff;
        d.cut2 = cutoff_threshold(dv.cutoff);
        d.seed = p.seed; d.rid = 0;   // noise stream keyed by the seed, as in the single-system form
        d.off_x = b->nx; b->nx += (size_t)p.nbeads * p.ndim * p.natoms;
        d.off_V = b->nV; b->nV += (size_t)p.natoms + 1;
        d.off_C = b->nC; b->nC += (size_t)p.nbeads * p.nbeads;
        off_R.push_back(b->nR); b->nR += 4 * (size_t)p.nbeads;
        off_H.push_back(b->nH);
        if (p.thermostat >= PIMDB_THERMO_NOSE_HOOVER) {
            // chains per bead and their degrees of freedom (nose_hoover.cpp:10-32, 152-163, 198-208)
            const int groups = p.thermostat == PIMDB_THERMO_NOSE_HOOVER ? 1
                               : p.thermostat == PIMDB_THERMO_NOSE_HOOVER_NP ? p.natoms : p.natoms * p.ndim;
            const int ndof = p.thermostat == PIMDB_THERMO_NOSE_HOOVER ? p.ndim * p.natoms
                             : p.thermostat == PIMDB_THERMO_NOSE_HOOVER_NP ? p.ndim : 1;
            d.nh_nc = p.nchains;
            d.nh_tbeta = dv.thermo_beta;            // beta / P
            d.nh_Qi = 1.0 * 1.0 * dv.beta / p.nbeads;   // hbar^2 beta / P
            d.nh_Q1 = ndof * d.nh_Qi;
            d.nh_required = ndof / d.nh_tbeta;
            b->nH += (size_t)p.nbeads * groups * p.nchains;
            b->nh_any = true;
        }
        b->desc.push_back(d);
        Nmax = std::max(Nmax, p.natoms);
    }
    int rc = PIMDB_OK;
    {
        // the default launch shape (1024 threads, one workgroup per CU) must fit
        std::vector<RepDesc> desc = b->desc;
        std::string why;
        b->lds = plan_lds(b, b->threads, 1, desc, &why);
        if (!b->lds) rc = b->fail(PIMDB_E_ARG, why);
        else b->desc = desc;
    }
    auto alloc = [&](double** ptr, size_t n) {
        if (rc) return;
        if (hipMalloc((void**)ptr, std::max<size_t>(1, n) * sizeof(double)) != hipSuccess ||
            hipMemset(*ptr, 0, std::max<size_t>(1, n) * sizeof(double)) != hipSuccess)
            rc = b->fail(PIMDB_E_HIP, "device allocation failed");
    };
    double *Ct = nullptr, *CTt = nullptr, *rot = nullptr;
    alloc(&b->bp.x, b->nx); alloc(&b->bp.p, b->nx); alloc(&b->bp.f, b->nx);
    alloc(&b->bp.V, b->nV);
    alloc(&b->bp.cmp, 8 * (size_t)nrep);
    alloc(&Ct, b->nC + NM_BLOCK); alloc(&CTt, b->nC + NM_BLOCK);   // padded for block reads
    alloc(&rot, b->nR);
    b->d_rot = rot;
    for (const RepDesc& d : b->desc) b->nmprop_any = b->nmprop_any || d.nmprop;
    if (b->nmprop_any) alloc(&b->d_fx, b->nx);
    if (b->nh_any) alloc(&b->d_nh, 3 * b->nH);   // the chains start at rest (alloc zeroes them)
    bool nhnm_any = false;   // Nose-Hoover with normal-mode coupling: the modes' buffer
    for (int r = 0; r < nrep; ++r) nhnm_any = nhnm_any || (reps[r].thermostat >= PIMDB_THERMO_NOSE_HOOVER && reps[r].nmthermostat);
    if (nhnm_any) alloc(&b->d_modes, b->nx);
    for (int r = 0; r < nrep && !rc; ++r) {   // the EXT paths' per-replica arrays
        RepDesc& d = b->desc[r];
        d.fx = d.nmprop ? b->d_fx + d.off_x : nullptr;   // (shares its slot with xws, bosonic replicas')
        d.rot = rot + off_R[r];
        d.nh = b->nh_any ? b->d_nh + off_H[r] : nullptr;
        d.nh_stride = b->nH;
        d.modes = nhnm_any ? b->d_modes + d.off_x : nullptr;
    }
    b->ext_any = b->nmprop_any || b->nh_any;
    b->bp.Ct = Ct;
    b->bp.CTt = CTt;
    if (!rc && (hipMalloc((void**)&b->bp.status, sizeof(int) * nrep) != hipSuccess ||
                hipMemset(b->bp.status, 0, sizeof(int) * nrep) != hipSuccess ||
                hipMalloc((void**)&b->bp.ctl, 2 * sizeof(unsigned long long)) != hipSuccess ||
                hipMemset(b->bp.ctl, 0, 2 * sizeof(unsigned long long)) != hipSuccess ||
                hipMalloc((void**)&b->d_desc, sizeof(RepDesc) * nrep) != hipSuccess ||
                hipMemcpy(b->d_desc, b->desc.data(), sizeof(RepDesc) * nrep, hipMemcpyHostToDevice) != hipSuccess))
        rc = b->fail(PIMDB_E_HIP, "device allocation failed");
    if (!rc) {
        b->bp.reps = b->d_desc;
        std::vector<double> hc(b->nC), hct(b->nC);
        for (int r = 0; r < nrep && !rc; ++r) {
            const int P = reps[r].nbeads;
            std::vector<double> C0((size_t)P * P), CT0((size_t)P * P);
            nm_matrices(P, C0.data(), CT0.data());
            transpose_square(P, C0.data(), hc.data() + b->desc[r].off_C);
            transpose_square(P, CT0.data(), hct.data() + b->desc[r].off_C);
        }
        // the free ring polymer's rotation per mode (nm_rotation, as the
        // single-system form builds it)
        std::vector<double> hr(std::max<size_t>(1, b->nR));
        for (int r = 0; r < nrep; ++r) nm_rotation(reps[r], derive(reps[r]), hr.data() + off_R[r]);
        if (hipMemcpy(Ct, hc.data(), sizeof(double) * b->nC, hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(CTt, hct.data(), sizeof(double) * b->nC, hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(rot, hr.data(), sizeof(double) * b->nR, hipMemcpyHostToDevice) != hipSuccess)
            rc = b->fail(PIMDB_E_HIP, "upload of normal-mode tables failed");
    }
    if (!rc && (hipStreamCreateWithFlags(&b->s, hipStreamNonBlocking) != hipSuccess ||
                hipEventCreate(&b->t0) != hipSuccess || hipEventCreate(&b->t1) != hipSuccess))
        rc = b->fail(PIMDB_E_HIP, "stream/event creation failed");
    if (!rc) rc = choose_form(b);
    if (rc) {
        set_create_error(b->err);
        pimdb_batch_destroy(b);
        return rc;
    }
    *out = b;
    return PIMDB_OK;
}

void pimdb_batch_destroy(pimdb_batch* b) {
    if (!b) return;
    if (b->s) (void)hipStreamSynchronize(b->s);
    if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    double* bufs[] = {b->bp.x, b->bp.p, b->bp.f, b->bp.V, b->bp.cmp,
                      const_cast<double*>(b->bp.Ct), const_cast<double*>(b->bp.CTt), b->d_rot, b->d_fx, b->d_nh,
                      b->d_modes, b->d_xws};
    for (double* p : bufs)
        if (p) (void)hipFree(p);
    if (b->bp.status) (void)hipFree(b->bp.status);
    if (b->bp.ctl) (void)hipFree(b->bp.ctl);
    if (b->d_desc) (void)hipFree(b->d_desc);
    if (b->d_sched) (void)hipFree(b->d_sched);
    if (b->d_sched_off) (void)hipFree(b->d_sched_off);
    free_split(b);
    if (b->t0) (void)hipEventDestroy(b->t0);
    if (b->t1) (void)hipEventDestroy(b->t1);
    if (b->s) (void)hipStreamDestroy(b->s);
    delete b;
}

const char* pimdb_batch_last_error(const pimdb_batch* b) { return b ? b->err.c_str() : create_error(); }

}  // extern "C"

// The second B and O-step that fused replicas leave owed after a step, done
// before the host reads or replaces a state.
static int finish_pending(pimdb_batch* b) {
    if (!b->fused_any || !b->maybe_pending) return PIMDB_OK;
    int rc = launch_batch(b, BM_FINISH);
    if (rc) return rc;
    BCK(hipStreamSynchronize(b->s));
    b->maybe_pending = false;
    return PIMDB_OK;
}

extern "C" {

int pimdb_batch_test_lost_wait(pimdb_batch* b) {
    if (!b) return PIMDB_E_ARG;
    BCK(fill_published(b->d_pub, b->npub, b->s));
    const int st = LOST_WAIT;
    BCK(hipMemcpy(b->bp.status, &st, sizeof(int), hipMemcpyHostToDevice));
    return check_batch_status(b);
}

int pimdb_batch_set_state(pimdb_batch* b, int rep, const double* x, const double* p) {
    if (!b || rep < 0 || rep >= b->R) return PIMDB_E_ARG;
    const int frc = finish_pending(b);
    if (frc) return frc;
    const pimdb_params& q = b->prm[rep];
    const size_t n = (size_t)q.nbeads * q.ndim * q.natoms;
    const RepDesc& d = b->desc[rep];
    const double* src[2] = {x, p};
    double* dst[2] = {b->bp.x + d.off_x, b->bp.p + d.off_x};
    StateArrays a{{nullptr, nullptr, nullptr}, 0, q.natoms, q.ndim, n, nullptr, 0};
    double* host[3];
    for (int k = 0; k < 2; ++k)
        if (src[k]) {
            host[a.count] = const_cast<double*>(src[k]);
            a.dev[a.count++] = dst[k];
        }
    if (a.count) BCK(copy_state<true>(a, host, b->s));
    if (p) {
        // no COM pending; the sum of p per axis for the next first O-step
        double cmp[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        for (size_t e = 0; e < n; ++e) cmp[4 + e % q.ndim] += p[e];
        BCK(hipMemcpy(b->bp.cmp + 8 * (size_t)rep, cmp, sizeof(cmp), hipMemcpyHostToDevice));
        b->unsettled = true;
    }
    return PIMDB_OK;
}

int pimdb_batch_get_state(pimdb_batch* b, int rep, double* x, double* p, double* f) {
    if (!b || rep < 0 || rep >= b->R) return PIMDB_E_ARG;
    const int frc = finish_pending(b);
    if (frc) return frc;
    const pimdb_params& q = b->prm[rep];
    const size_t n = (size_t)q.nbeads * q.ndim * q.natoms;
    const RepDesc& d = b->desc[rep];
    double* dst[3] = {x, p, f};
    double* src[3] = {b->bp.x + d.off_x, b->bp.p + d.off_x, b->bp.f + d.off_x};
    // p without the COM momentum still pending from the last O-step
    StateArrays a{{nullptr, nullptr, nullptr}, 0, q.natoms, q.ndim, n, nullptr, 0};
    double* host[3];
    for (int k = 0; k < 3; ++k)
        if (dst[k]) {
            if (k == 1) {
                a.cm = b->bp.cmp + 8 * (size_t)rep;
                a.cm_of = a.count;
            }
            host[a.count] = dst[k];
            a.dev[a.count++] = src[k];
        }
    if (a.count) BCK(copy_state<false>(a, host, b->s));
    return PIMDB_OK;
}

int pimdb_batch_forces(pimdb_batch* b) {
    if (!b) return PIMDB_E_ARG;
    if (b->split) {
        b->sp.bp = b->bp;
        BCK(launch_split_forces(b->sp, b->D, b->kind, true, STEP_FORCES, b->s));
        BCK(launch_split_integrate(b->sp, b->D, STEP_FORCES, b->s));
    } else {
        const int rc = launch_batch(b, BM_FORCES);
        if (rc) return rc;
    }
    return check_batch_status(b);
}

int pimdb_batch_step(pimdb_batch* b, int nsteps) {
    if (!b || nsteps < 0) return PIMDB_E_ARG;
    const int rc = enqueue_batch_steps(b, nsteps);
    if (rc) return rc;
    return check_batch_status(b);
}

int pimdb_batch_step_timed(pimdb_batch* b, int nsteps, double* device_ms) {
    if (!b || nsteps < 1 || !device_ms) return PIMDB_E_ARG;
    int rc = b->split ? PIMDB_OK : capture(b);
    if (rc) return rc;
    BCK(hipEventRecord(b->t0, b->s));
    rc = enqueue_batch_steps(b, nsteps);
    if (rc) return rc;
    BCK(hipEventRecord(b->t1, b->s));
    BCK(hipEventSynchronize(b->t1));
    float ms = 0.0f;
    BCK(hipEventElapsedTime(&ms, b->t0, b->t1));
    *device_ms = (double)ms;
    return check_batch_status(b);
}

int pimdb_batch_configure(pimdb_batch* b, int threads, int resident) {
    if (!b) return PIMDB_E_ARG;
    if (threads && threads != 256 && threads != 512 && threads != 1024)
        return b->fail(PIMDB_E_ARG, "threads must be 256, 512 or 1024");
    if (resident < 0) return b->fail(PIMDB_E_ARG, "resident must be >= 0");
    BCK(hipStreamSynchronize(b->s));
    const int old_threads = b->threads, old_resident = b->resident;
    if (threads) b->threads = threads;
    if (resident) b->resident = resident;
    const bool split = b->split;
    if (threads || resident) b->split = false;   // an explicit shape is the persistent kernel's
    const int rc = upload_schedule(b);
    if (rc == PIMDB_E_ARG) {   // this shape's LDS plan does not fit: keep the previous one
        const std::string why = b->err;
        b->threads = old_threads;
        b->resident = old_resident;
        b->split = split;
        const int rc2 = upload_schedule(b);
        if (rc2) return rc2;
        return b->fail(PIMDB_E_ARG, why);
    }
    return rc;
}

int pimdb_batch_form(const pimdb_batch* b, int* two_kernel, int* slice_waves) {
    if (!b) return PIMDB_E_ARG;
    if (two_kernel) *two_kernel = b->split ? 1 : 0;
    if (slice_waves) *slice_waves = b->split ? b->sp.share : 1;
    return PIMDB_OK;
}

int pimdb_batch_set_form(pimdb_batch* b, int two_kernel) {
    if (!b) return PIMDB_E_ARG;
    if (two_kernel) {
        if (!split_able(b)) return b->fail(PIMDB_E_ARG, "a replica does not take the two-kernel form");
        const int rc = build_split(b);
        if (rc) return rc;
    }
    b->split = two_kernel != 0;
    return PIMDB_OK;
}

int pimdb_batch_time_step(pimdb_batch* b, int reps, double* ms_step) {
    if (!b || reps < 1 || !ms_step) return PIMDB_E_ARG;
    int rc = enqueue_batch_steps(b, 1);
    if (rc) return rc;
    BCK(hipEventRecord(b->t0, b->s));
    rc = enqueue_batch_steps(b, reps);
    if (rc) return rc;
    BCK(hipEventRecord(b->t1, b->s));
    BCK(hipEventSynchronize(b->t1));
    float ms = 0.0f;
    BCK(hipEventElapsedTime(&ms, b->t0, b->t1));
    *ms_step = (double)ms / reps;
    return check_batch_status(b);
}

// Device ms of one launch of a phase (0 step, 1 pair forces, 2 exchange,
// 3 integrator), averaged over reps launches, from a saved state that is
// restored afterwards.
int pimdb_batch_time_phase(pimdb_batch* b, int phase, int reps, double* ms_out) {
    if (!b || reps < 1 || !ms_out || phase < 0 || phase > 3) return PIMDB_E_ARG;
    static const int modes[4] = {BM_STEP, BM_PAIRS, BM_EXCHANGE, BM_INTEGRATOR};
    double *sx = nullptr, *sp = nullptr, *sf = nullptr, *sfx = nullptr;
    unsigned long long sctl[2];
    BCK(hipStreamSynchronize(b->s));
    BCK(hipMalloc((void**)&sx, sizeof(double) * b->nx));
    BCK(hipMalloc((void**)&sp, sizeof(double) * b->nx));
    BCK(hipMalloc((void**)&sf, sizeof(double) * b->nx));
    BCK(hipMemcpy(sx, b->bp.x, sizeof(double) * b->nx, hipMemcpyDeviceToDevice));
    BCK(hipMemcpy(sp, b->bp.p, sizeof(double) * b->nx, hipMemcpyDeviceToDevice));
    BCK(hipMemcpy(sf, b->bp.f, sizeof(double) * b->nx, hipMemcpyDeviceToDevice));
    if (b->d_fx) {   // the normal-mode replicas' physical forces
        BCK(hipMalloc((void**)&sfx, sizeof(double) * b->nx));
        BCK(hipMemcpy(sfx, b->d_fx, sizeof(double) * b->nx, hipMemcpyDeviceToDevice));
    }
    std::vector<double> seta;   // the Nose-Hoover chains
    if (b->nh_any) {
        seta.resize(3 * b->nH);
        BCK(hipMemcpy(seta.data(), b->d_nh, sizeof(double) * 3 * b->nH, hipMemcpyDeviceToHost));
    }
    BCK(hipMemcpy(sctl, b->bp.ctl, sizeof(sctl), hipMemcpyDeviceToHost));
    std::vector<double> scmp(8 * (size_t)b->R);
    BCK(hipMemcpy(scmp.data(), b->bp.cmp, sizeof(double) * scmp.size(), hipMemcpyDeviceToHost));
    int rc = launch_batch(b, modes[phase]);   // warm
    if (!rc) {
        BCK(hipEventRecord(b->t0, b->s));
        for (int r = 0; r < reps && !rc; ++r) rc = launch_batch(b, modes[phase]);
        BCK(hipEventRecord(b->t1, b->s));
        BCK(hipEventSynchronize(b->t1));
        float ms = 0.0f;
        BCK(hipEventElapsedTime(&ms, b->t0, b->t1));
        *ms_out = (double)ms / reps;
    }
    BCK(hipStreamSynchronize(b->s));
    BCK(hipMemcpy(b->bp.x, sx, sizeof(double) * b->nx, hipMemcpyDeviceToDevice));
    BCK(hipMemcpy(b->bp.p, sp, sizeof(double) * b->nx, hipMemcpyDeviceToDevice));
    BCK(hipMemcpy(b->bp.f, sf, sizeof(double) * b->nx, hipMemcpyDeviceToDevice));
    if (sfx) BCK(hipMemcpy(b->d_fx, sfx, sizeof(double) * b->nx, hipMemcpyDeviceToDevice));
    if (b->nh_any) BCK(hipMemcpy(b->d_nh, seta.data(), sizeof(double) * 3 * b->nH, hipMemcpyHostToDevice));
    BCK(hipMemcpy(b->bp.ctl, sctl, sizeof(sctl), hipMemcpyHostToDevice));
    BCK(hipMemcpy(b->bp.cmp, scmp.data(), sizeof(double) * scmp.size(), hipMemcpyHostToDevice));
    (void)hipFree(sx);
    (void)hipFree(sp);
    (void)hipFree(sf);
    if (sfx) (void)hipFree(sfx);
    if (rc) return rc;
    return check_batch_status(b);
}

// Tries every workgroup size and residency (1 or 2 workgroups per CU) for
// trial_steps steps from a saved state, keeps the fastest and restores the
// state, so the batch's trajectory is unaffected.
int pimdb_batch_autotune(pimdb_batch* b, int trial_steps, int* threads_out, int* resident_out) {
    if (!b || trial_steps < 1) return PIMDB_E_ARG;
    double *sx = nullptr, *sp = nullptr, *sf = nullptr, *sfx = nullptr;
    unsigned long long sctl[2];
    BCK(hipStreamSynchronize(b->s));
    BCK(hipMalloc((void**)&sx, sizeof(double) * b->nx));
    BCK(hipMalloc((void**)&sp, sizeof(double) * b->nx));
    BCK(hipMalloc((void**)&sf, sizeof(double) * b->nx));
    BCK(hipMemcpy(sx, b->bp.x, sizeof(double) * b->nx, hipMemcpyDeviceToDevice));
    BCK(hipMemcpy(sp, b->bp.p, sizeof(double) * b->nx, hipMemcpyDeviceToDevice));
    BCK(hipMemcpy(sf, b->bp.f, sizeof(double) * b->nx, hipMemcpyDeviceToDevice));
    if (b->d_fx) {   // the normal-mode replicas' physical forces
        BCK(hipMalloc((void**)&sfx, sizeof(double) * b->nx));
        BCK(hipMemcpy(sfx, b->d_fx, sizeof(double) * b->nx, hipMemcpyDeviceToDevice));
    }
    std::vector<double> seta;   // the Nose-Hoover chains
    if (b->nh_any) {
        seta.resize(3 * b->nH);
        BCK(hipMemcpy(seta.data(), b->d_nh, sizeof(double) * 3 * b->nH, hipMemcpyDeviceToHost));
    }
    BCK(hipMemcpy(sctl, b->bp.ctl, sizeof(sctl), hipMemcpyDeviceToHost));
    std::vector<double> scmp(8 * (size_t)b->R);
    BCK(hipMemcpy(scmp.data(), b->bp.cmp, sizeof(double) * scmp.size(), hipMemcpyDeviceToHost));
    // launch shapes: threads per workgroup x workgroups per CU, at most 16
    // waves per CU (the kernel's 128 VGPRs allow 4 waves per SIMD); shapes
    // whose LDS plan does not fit, or that give the same grid as one already
    // timed, are skipped
    const int cand[6][2] = {{1024, 1}, {512, 1}, {512, 2}, {256, 1}, {256, 2}, {256, 4}};
    double best = 1e300;
    int bt = b->threads, br = b->resident;
    int rc = PIMDB_OK;
    const bool pending = b->maybe_pending;
    b->split = false;
    std::vector<std::pair<int, int>> tried;
    for (int ci = 0; ci < 6 && !rc; ++ci) {
        const int threads = cand[ci][0], per_cu = cand[ci][1], resident = b->cus * per_cu;
        const int grid = std::max(1, std::min(b->R, resident));
        // more workgroups per CU than the batch fills only tightens the plan
        if (per_cu > 1 && grid <= b->cus * (per_cu - 1)) continue;
        if (std::find(tried.begin(), tried.end(), std::make_pair(threads, grid)) != tried.end()) continue;
        tried.push_back({threads, grid});
        std::vector<RepDesc> desc = b->desc;
        std::string why;
        if (!plan_lds(b, threads, per_cu, desc, &why)) continue;
        b->threads = threads;
        b->resident = resident;
        rc = upload_schedule(b);
        double ms = 0.0;
        if (!rc) rc = pimdb_batch_time_step(b, trial_steps, &ms);
        if (!rc && ms < best) {
            best = ms;
            bt = b->threads;
            br = b->resident;
        }
    }
    b->threads = bt;
    b->resident = br;
    if (!rc) rc = upload_schedule(b);
    // the two-kernel form (last: its steps leave nothing owed)
    if (!rc && split_able(b) && build_split(b) == PIMDB_OK) {
        b->split = true;
        double ms = 0.0;
        rc = pimdb_batch_time_step(b, trial_steps, &ms);
        b->split = !rc && ms < best;
    }
    BCK(hipStreamSynchronize(b->s));
    BCK(hipMemcpy(b->bp.x, sx, sizeof(double) * b->nx, hipMemcpyDeviceToDevice));
    BCK(hipMemcpy(b->bp.p, sp, sizeof(double) * b->nx, hipMemcpyDeviceToDevice));
    BCK(hipMemcpy(b->bp.f, sf, sizeof(double) * b->nx, hipMemcpyDeviceToDevice));
    if (sfx) BCK(hipMemcpy(b->d_fx, sfx, sizeof(double) * b->nx, hipMemcpyDeviceToDevice));
    if (b->nh_any) BCK(hipMemcpy(b->d_nh, seta.data(), sizeof(double) * 3 * b->nH, hipMemcpyHostToDevice));
    BCK(hipMemcpy(b->bp.ctl, sctl, sizeof(sctl), hipMemcpyHostToDevice));
    BCK(hipMemcpy(b->bp.cmp, scmp.data(), sizeof(double) * scmp.size(), hipMemcpyHostToDevice));
    (void)hipFree(sx);
    (void)hipFree(sp);
    (void)hipFree(sf);
    if (sfx) (void)hipFree(sfx);
    b->maybe_pending = pending;   // as the restored momenta are
    b->unsettled = true;
    if (threads_out) *threads_out = b->threads;
    if (resident_out) *resident_out = b->resident;
    return rc;
}

}  // extern "C"
