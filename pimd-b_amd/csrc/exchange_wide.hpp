// exchange_wide.hpp -- the two exchange recursions of one ring with one
// workgroup per block of 64 targets and direction, for callers with a single
// ring and an idle card (the single-system context, the exchange plan).
//
// Reference: src/bosonic_exchange/quadratic_bosonic_exchange.cpp:73-128 of
// higj/pimd-b.  The recursion, w(n,q), U and the block structure are those of
// exchange.hpp (file header there).
//
// Why.  With both recursions on one workgroup each, 254 of 256 compute units
// idle and one CU's vector units carry a direction's N^2/2 terms: N=256 took
// 36.8 us and N=1000 271 us.  The terms of target block I over the sources of
// block J < I depend on earlier blocks only through the 64 values U of block
// J, so block I's workgroup evaluates everything else ahead of time and waits
// for those values.  What is left on the chain from one block to the next:
// the 64 x 64 exponentials against the previous block, one reduction, the
// in-block substitution and the publication of 64 doubles.
//
// Publication.  U (plus, backward, the source's ln(N-q) term) goes to a
// global array by relaxed device-scope atomic stores and is read by relaxed
// device-scope atomic loads until it differs from XW_EMPTY (a NaN pattern no
// result carries): the value is its own flag, so no fence is needed.  A
// workgroup waits only for lower-numbered ones, which are dispatched first,
// and a wait ends after XW_SPIN polls at the latest (the status flag is then
// set).  The last block's workgroup has read every value once all others have
// (block J publishes only after its own reads), so it puts XW_EMPTY back for
// the next launch.
//
// Scaling.  The in-block part needs no min-plus pass.  With the one-particle
// cycles' energies e_r = beta~ ecyc(r) and their running sum
// g_t = sum_{r <= t} e_r over the block's targets,
//     z_t = exp(-(U_t - g_t - sigma)),  sigma = U of the last earlier target,
// obeys  z_t = s_t + sum_{j<t} B(j,t) z_j,  B(j,t) = exp(g_t - g_j - w(t,j)),
//     s_t = sum_{q earlier} exp(sigma + g_t - w(t,q) - U_q):
// B is known before any U arrives and s needs no running minimum for the
// sources of the previous block (farther ones keep their online log-sum-exp,
// off the chain).  z_t is at least the one-particle path's product of 1/n,
// e^-621 for N = 2^14, and it overflows only where longer cycles are favoured
// by e^700 within one block; such a block (z not in [1e-290, 1e290]) is taken
// again by the exact min-plus form (xw_block_safe).
#pragma once

#include "exchange.hpp"

namespace pimdb {

// Threads of a workgroup (template parameter NT): 1024 where a ring has the
// card to itself; 256 beside other rings' work, where the idle waves of a
// waiting workgroup would hold registers that others could use.
constexpr int XW_THREADS = 1024;
constexpr unsigned long long XW_EMPTY = ~0ull;
constexpr long long XW_SPIN = 1ll << 22;             // polls of one wait (seconds)

// Global workspace of one ring: the published values of both directions.
__host__ __device__ inline size_t xw_pub_words(int N) { return 2 * ((size_t)N + 1); }
__host__ __device__ inline int xw_grid(int N) { return 2 * rec_blocks(N); }

// LDS doubles: the ring, the block's gauge and source logarithms, the
// in-block matrix, per-wave partials, the substitution's results, the wave
// totals of the prefix sums and a flag.
__host__ __device__ inline size_t xw_shared_doubles(int N, int D, int nw) {
    return (size_t)(2 * D + 2) * N + 2 * REC_B + (size_t)REC_TRI + 2 * (size_t)nw * REC_B + 2 * REC_B + 2 * (size_t)nw + 2;
}
inline size_t xw_lds_bytes(int N, int D, int threads = XW_THREADS) {
    return sizeof(double) * xw_shared_doubles(N, D, threads / WAVE);
}

struct XwShared {
    double *x1, *xP, *Shi, *Slo;   // the ring [D][N], [D][N], [N], [N]
    double *g, *lgs;               // [REC_B] gauge; ln(N-q) of the block as sources (backward)
    double *a;                     // [REC_TRI] in-block matrix at rec_idx(j, t)
    double *part, *psum;           // [waves][REC_B]
    double *R, *z;                 // [REC_B]
    double *tot;                   // [2 waves] wave totals of the prefix sums
    int* flag;
};

template <int NT>
__device__ __forceinline__ XwShared xw_carve(double* p, int N, int D) {
    constexpr int NW = NT / WAVE;
    XwShared s;
    s.x1 = p; p += (size_t)D * N;
    s.xP = p; p += (size_t)D * N;
    s.Shi = p; p += N;
    s.Slo = p; p += N;
    s.g = p; p += REC_B;
    s.lgs = p; p += REC_B;
    s.a = p; p += REC_TRI;
    s.part = p; p += NW * REC_B;
    s.psum = p; p += NW * REC_B;
    s.R = p; p += REC_B;
    s.z = p; p += REC_B;
    s.tot = p; p += 2 * NW;
    s.flag = (int*)p;
    return s;
}

template <int CTRL, int ROWS>
__device__ __forceinline__ DD dd_scan_step(DD v) {
    return dd_add(DD{dpp_or_zero<CTRL, ROWS>(v.hi), dpp_or_zero<CTRL, ROWS>(v.lo)}, v);
}
// Inclusive sums over the lanes of a wave (wave_scan's steps).
__device__ __forceinline__ DD dd_wave_scan(DD v) {
    v = dd_scan_step<0x111, 0xF>(v);
    v = dd_scan_step<0x112, 0xF>(v);
    v = dd_scan_step<0x114, 0xF>(v);
    v = dd_scan_step<0x118, 0xF>(v);
    v = dd_scan_step<0x142, 0xA>(v);
    v = dd_scan_step<0x143, 0xC>(v);
    return v;
}

// One bead's positions: axis a of particle i at p[a sa + i si].
struct BeadView {
    const double* p;
    long long sa, si;
    __device__ __forceinline__ double at(int a, int i) const { return p[a * sa + i * si]; }
};

// Beads 1 and P into LDS and the split prefix sums of the ring's links
// (exchange.hpp, Ring), by the whole workgroup: every thread sums a run of
// links, the waves scan their totals.  Every workgroup of a ring computes the
// same values.  Shi_out / Slo_out / xc_out (may be null) receive the sums and
// a copy [2][D][N] of the two beads.
template <int D, int NT>
__device__ __forceinline__ Ring xw_stage(const XwShared& sh, int N, BeadView x1, BeadView xP, double k, bool pbc, double L,
                                         double* Shi_out, double* Slo_out, double* xc_out) {
    constexpr int NW = NT / WAVE;
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const Ring r = make_ring(sh.x1, sh.xP, sh.Shi, sh.Slo, k, pbc, L);
    for (int e = tid; e < D * N; e += NT) {
        const int a = D == 1 ? 0 : e / N, i = e - a * N;
        const double u = x1.at(a, i), v = xP.at(a, i);
        sh.x1[e] = u;
        sh.xP[e] = v;
        if (xc_out) {
            xc_out[e] = u;
            xc_out[(size_t)D * N + e] = v;
        }
    }
    const int c = (N + NT - 1) / NT, v0 = tid * c;
    auto link = [&](int v) {
        double d[D];
#pragma unroll
        for (int ax = 0; ax < D; ++ax) d[ax] = ring_image(x1.at(ax, v + 1) - xP.at(ax, v), r);
        return norm2_fma<D>(d);
    };
    DD sum{0.0, 0.0};
    double first = 0.0;   // the thread's first link, kept for the running sums of runs of one
    for (int v = v0; v < min(v0 + c, N - 1); ++v) {
        const double l = link(v);
        if (v == v0) first = l;
        sum = dd_add(sum, DD{l, 0.0});
    }
    const DD inc = dd_wave_scan(sum);
    if (lane == WAVE - 1) {
        sh.tot[2 * wave] = inc.hi;
        sh.tot[2 * wave + 1] = inc.lo;
    }
    __syncthreads();
    DD tw{0.0, 0.0};
    if (lane < NW) tw = DD{sh.tot[2 * lane], sh.tot[2 * lane + 1]};
    tw = dd_wave_scan(tw);
    const double total = wave_bcast_uniform(tw.hi, NW - 1);
    DD ex{dpp_or_zero<0x138, 0xF>(inc.hi), dpp_or_zero<0x138, 0xF>(inc.lo)};   // wave_shr:1
    if (wave > 0) ex = dd_add(DD{wave_bcast_uniform(tw.hi, wave - 1), wave_bcast_uniform(tw.lo, wave - 1)}, ex);
    const double q = total > 0.0 ? ldexp(1.0, ilogb(total) - 40) : 1.0;
    const double invq = 1.0 / q;
    for (int v = v0; v < min(v0 + c, N); ++v) {
        const double h = rint(ex.hi * invq) * q, l = (ex.hi - h) + ex.lo;
        sh.Shi[v] = h;
        sh.Slo[v] = l;
        if (Shi_out) {
            Shi_out[v] = h;
            Slo_out[v] = l;
        }
        if (v + 1 < v0 + c && v < N - 1) ex = dd_add(ex, DD{v == v0 ? first : link(v), 0.0});
    }
    __syncthreads();
    return r;
}

// The target side of w(n,q) of one lane, and w(n,q) without the source's
// logarithm (backward: ln(N-q) travels with the published U).
template <int DIR, int D>
__device__ __forceinline__ RecTarget<D> xw_target(const XwShared& sh, int N, int n) {
    RecTarget<D> t;
    const int idx = DIR == 0 ? n - 1 : N - n;
    const double* xs = DIR == 0 ? sh.xP : sh.x1;
#pragma unroll
    for (int a = 0; a < D; ++a) t.x[a] = xs[a * N + idx];
    t.shi = sh.Shi[idx];
    t.slo = sh.Slo[idx];
    t.lg = DIR == 0 ? log((double)n) : 0.0;
    return t;
}
template <int DIR, int D>
__device__ __forceinline__ double xw_w(const XwShared& sh, const Ring& r, double bk, int N, const RecTarget<D>& t,
                                       int q) {
    const int idx = DIR == 0 ? q : N - 1 - q;
    const double* xs = DIR == 0 ? sh.x1 : sh.xP;
    double d[D];
#pragma unroll
    for (int a = 0; a < D; ++a) d[a] = ring_image(xs[a * N + idx] - t.x[a], r);
    const double sd = DIR == 0 ? ring_sdiff(t.shi, t.slo, sh.Shi[idx], sh.Slo[idx])
                               : ring_sdiff(sh.Shi[idx], sh.Slo[idx], t.shi, t.slo);
    return fma(bk, sd + norm2_fma<D>(d), t.lg);
}

__device__ __forceinline__ unsigned long long xw_bits(double v) { return (unsigned long long)__double_as_longlong(v); }
// Stores a value for the other workgroups (a NaN with the empty pattern as
// another NaN).
__device__ __forceinline__ void xw_publish(unsigned long long* p, double v) {
    unsigned long long b = xw_bits(v);
    if (b == XW_EMPTY) b = 0x7FF8000000000000ull;
    __hip_atomic_store(p, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The 64 values of a finished block, one per lane (whole wave).
__device__ __forceinline__ double xw_wait(unsigned long long* p, int lane, int* status) {
    unsigned long long b = XW_EMPTY;
    long long spin = 0;
    for (;;) {
        b = __hip_atomic_load(p + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__all(b != XW_EMPTY)) break;
        if (++spin >= XW_SPIN) {
            if (lane == 0) raise_status(status);
            break;
        }
        __builtin_amdgcn_s_sleep(1);
    }
    return __longlong_as_double((long long)b);
}

// One block with the exact min-plus shifts (exchange.hpp, steps (1)-(4)),
// every earlier U being published: for blocks whose z left the range.  All
// threads; U of the lane's target in every lane of wave 0.
template <int DIR, int D, int NT>
__device__ __noinline__ double xw_block_safe(int I, int N, int nb, double bk, double u0, const Ring r, const XwShared sh,
                                             unsigned long long* pub) {
    constexpr int NW = NT / WAVE, XW_SRC = REC_B / NW;   // sources of a block per wave
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int n0 = 1 + I * REC_B;
    const RecTarget<D> tg = xw_target<DIR, D>(sh, N, n0 + min(lane, nb - 1));
    double m = INFINITY, s = 0.0;
    auto add = [&](int q, double uq) {
        const double y = xw_w<DIR, D>(sh, r, bk, N, tg, q) + uq;
        const double mn = fmin(m, y);
        s = fma(s, exp_pair(mn - m), exp_pair(mn - y));   // m = inf (first source): s = 0 stays 0
        m = mn;
    };
    if (wave == 0) add(0, u0);
    for (int J = 0; J < I; ++J)
        for (int u = 0; u < XW_SRC; ++u) {
            const int q = J * REC_B + 1 + wave * XW_SRC + u;
            add(q, __longlong_as_double((long long)__hip_atomic_load(pub + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)));
        }
    sh.part[wave * REC_B + lane] = lane < nb ? m : INFINITY;
    sh.psum[wave * REC_B + lane] = lane < nb ? s : 0.0;
    for (int vr = wave; vr < REC_B / 2; vr += NW) {
        int t, j;
        rec_tri(vr, lane, t, j);
        if (t < 0) continue;
        double w = INFINITY;
        if (t < nb) w = xw_w<DIR, D>(sh, r, bk, N, xw_target<DIR, D>(sh, N, n0 + t), n0 + j) + sh.lgs[j];
        sh.a[rec_idx(j, t)] = w;
    }
    __syncthreads();
    if (wave == 0) {
        double rr = INFINITY;
        for (int w = 0; w < NW; ++w) rr = fmin(rr, sh.part[w * REC_B + lane]);
        rec_inblock_seq<0>(sh.a, lane, rr, sh.R);
    }
    __syncthreads();
    {
        const double sw = sh.psum[wave * REC_B + lane];
        double c = 0.0;
        if (lane < nb && sw > 0.0) c = sw * exp_pair(sh.R[lane] - sh.part[wave * REC_B + lane]);
        sh.psum[wave * REC_B + lane] = c;
    }
    for (int vr = wave; vr < REC_B / 2; vr += NW) {
        int t, j;
        rec_tri(vr, lane, t, j);
        if (t >= 0) sh.a[rec_idx(j, t)] = t < nb ? exp_pair(-(sh.a[rec_idx(j, t)] + sh.R[j] - sh.R[t])) : 0.0;
    }
    __syncthreads();
    double u = 0.0;
    if (wave == 0) {
        double z0 = 0.0;
        for (int w = 0; w < NW; ++w) z0 += sh.psum[w * REC_B + lane];
        rec_inblock_seq<1>(sh.a, lane, z0, sh.z);
        u = sh.R[lane] - log(sh.z[lane]);
    }
    __syncthreads();
    return u;
}

// Target block I of one recursion on one workgroup of NT threads
// (the ring staged).  pub: this direction's published values [N+1].
template <int DIR, int D, int NT>
__device__ __forceinline__ void xw_block(int I, int N, double bt, const Ring& r, const XwShared& sh,
                                         unsigned long long* __restrict__ pub, double* __restrict__ V,
                                         double* __restrict__ Vb, double* __restrict__ VB, int* __restrict__ status) {
    constexpr int NW = NT / WAVE, XW_SRC = REC_B / NW;   // sources of a block per wave
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int ntarget = DIR == 0 ? N : N - 1;
    const int n0 = 1 + I * REC_B, nb = min(REC_B, ntarget - n0 + 1);
    if (I == 0 && tid == 0) {
        if (DIR == 0) V[0] = 0.0;
        else Vb[N] = 0.0;
    }
    if (nb <= 0) return;   // (the backward recursion's empty last block)
    const bool last = n0 + nb > ntarget;
    const double bk = bt * r.halfk;
    const int tn = n0 + min(lane, nb - 1);
    const RecTarget<D> tg = xw_target<DIR, D>(sh, N, tn);
    const double u0 = DIR == 0 ? 0.0 : log((double)N);   // source 0
    // the gauge: running sum of the one-particle cycles' energies
    double e1;
    {
        const int idx = DIR == 0 ? tn - 1 : N - tn;
        double d[D];
#pragma unroll
        for (int a = 0; a < D; ++a) d[a] = ring_image(sh.x1[a * N + idx] - sh.xP[a * N + idx], r);
        e1 = bk * norm2_fma<D>(d);
    }
    const double g = wave_scan(e1);
    const double lgs = DIR == 0 ? 0.0 : log((double)max(1, N - (n0 + lane)));   // the lane's target as a source
    if (wave == 0) {
        sh.g[lane] = g;
        sh.lgs[lane] = lgs;
    }
    __syncthreads();
    for (int vr = wave; vr < REC_B / 2; vr += NW) {
        int t, j;
        rec_tri(vr, lane, t, j);
        if (t < 0) continue;
        double c = 0.0;
        if (t < nb) {
            const double w = xw_w<DIR, D>(sh, r, bk, N, xw_target<DIR, D>(sh, N, n0 + t), n0 + j) + sh.lgs[j];
            c = exp_pair((sh.g[t] - sh.g[j]) - w);
        }
        sh.a[rec_idx(j, t)] = c;
    }
    // earlier sources: source 0 on wave 0, then XW_SRC of every block per wave
    double m = INFINITY, s = 0.0, near = 0.0, sigma = u0;
    if (wave == 0) {
        m = xw_w<DIR, D>(sh, r, bk, N, tg, 0) + u0;
        s = 1.0;
    }
    // (four sources in registers at a time; the first four of a block are
    // evaluated while their U are awaited)
    constexpr int XQ = 4;
    for (int J = 0; J < I; ++J) {
        const int qb = J * REC_B + 1, q0 = wave * XW_SRC;
        double w[XQ], uq[XQ];
#pragma unroll
        for (int u = 0; u < XQ; ++u) w[u] = xw_w<DIR, D>(sh, r, bk, N, tg, qb + q0 + u);
        const double v = xw_wait(pub + qb, lane, status);
        if (J == I - 1) sigma = wave_bcast_uniform(v, REC_B - 1);
#pragma unroll 1
        for (int c = 0; c < XW_SRC; c += XQ) {
#pragma unroll
            for (int u = 0; u < XQ; ++u) {
                uq[u] = wave_bcast_uniform(v, q0 + c + u);
                if (c > 0) w[u] = xw_w<DIR, D>(sh, r, bk, N, tg, qb + q0 + c + u);
            }
            if (J < I - 1) {
                double mn = m;
#pragma unroll
                for (int u = 0; u < XQ; ++u) {
                    w[u] += uq[u];
                    mn = fmin(mn, w[u]);
                }
                s *= exp_pair(mn - m);   // m = inf: s = 0 stays 0
                m = mn;
#pragma unroll
                for (int u = 0; u < XQ; ++u) s += exp_pair(mn - w[u]);
            } else {
#pragma unroll
                for (int u = 0; u < XQ; ++u) near += exp_pair((sigma - uq[u]) + (g - w[u]));
            }
        }
    }
    if (s > 0.0) near = fma(s, exp_pair((sigma - m) + g), near);
    sh.psum[wave * REC_B + lane] = lane < nb ? near : 0.0;
    __syncthreads();
    double u = 0.0;
    if (wave == 0) {
        double z0 = 0.0;
#pragma unroll
        for (int w = 0; w < NW; ++w) z0 += sh.psum[w * REC_B + lane];
        rec_inblock_seq<1>(sh.a, lane, z0, sh.z);
        const double z = sh.z[lane];
        u = (sigma + g) - log(z);
        const bool ok = lane >= nb || (z >= 1e-290 && z <= 1e290);
        const bool all = __all(ok);
        if (all && !last) xw_publish(pub + n0 + lane, u + lgs);
        if (lane == 0) *sh.flag = all ? 0 : 1;
    }
    __syncthreads();
    if (*sh.flag) {
        u = xw_block_safe<DIR, D, NT>(I, N, nb, bk, u0, r, sh, pub);
        if (wave == 0) {
            if (lane < nb && !isfinite(u)) raise_status(status);
            if (!last) xw_publish(pub + n0 + lane, u + lgs);
        }
    }
    if (wave == 0 && lane < nb) {
        const int n = n0 + lane;
        if (DIR == 0) {
            V[n] = u / bt;
            if (n == N) {
                Vb[0] = u / bt;   // V_backwards[0] = V[N], :127
                if (VB) *VB = u / bt;
            }
        } else {
            Vb[N - n] = u / bt;
        }
    }
    if (last) {   // every value has been read by every workgroup: empty for the next launch
        for (int q = tid; q < n0; q += NT)
            __hip_atomic_store(pub + q, XW_EMPTY, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Workgroup b of xw_grid(N): block b / 2, forward (even) or backward (odd);
// lower blocks first.  pub: xw_pub_words(N) words, all XW_EMPTY on entry and
// on return.  Block 0's forward workgroup writes the prefix sums and, where
// asked (xc, VB not null), the beads' copy and V[N].
template <int D, int NT>
__device__ __forceinline__ void xw_recursions(double* smem, int b, int N, double bt, double k, int pbc, double L,
                                              BeadView x1, BeadView xP, double* __restrict__ V,
                                              double* __restrict__ Vb, double* __restrict__ VB,
                                              double* __restrict__ Shi, double* __restrict__ Slo, double* __restrict__ xc,
                                              unsigned long long* __restrict__ pub, int* __restrict__ status) {
    const XwShared sh = xw_carve<NT>(smem, N, D);
    const bool first = b == 0;
    const Ring r = xw_stage<D, NT>(sh, N, x1, xP, k, pbc != 0, L, first ? Shi : nullptr, first ? Slo : nullptr,
                               first ? xc : nullptr);
    if ((b & 1) == 0) xw_block<0, D, NT>(b >> 1, N, bt, r, sh, pub, V, Vb, VB, status);
    else xw_block<1, D, NT>(b >> 1, N, bt, r, sh, pub + N + 1, V, Vb, nullptr, status);
}

template <int D>
static __global__ void __launch_bounds__(XW_THREADS)
k_exchange_wide(int N, double bt, double k, int pbc, double L, BeadView x1, BeadView xP, double* __restrict__ V,
                double* __restrict__ Vb, double* __restrict__ VB, double* __restrict__ Shi, double* __restrict__ Slo,
                double* __restrict__ xc, unsigned long long* __restrict__ pub, int* __restrict__ status) {
    extern __shared__ double smem[];
    xw_recursions<D, XW_THREADS>(smem, blockIdx.x, N, bt, k, pbc, L, x1, xP, V, Vb, VB, Shi, Slo, xc, pub, status);
}

}  // namespace pimdb
