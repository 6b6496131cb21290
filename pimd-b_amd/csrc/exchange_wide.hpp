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
// J, so block I's workgroup prepares everything else and waits for those.
//
// Scaling.  No running minimum is needed between neighbours.  Let
//     G_t = sum_{r <= t} (e_r + l_r / 2)
// over a block's targets, e_r = beta~ ecyc(r) the one-particle cycle's energy
// and l_r the logarithm its term carries (ln n forward, ln(N-q) backward; a
// scale only, so the hardware's single-precision logarithm serves), and
//     z_t = exp(-(U_t - G_t - sigma)),   sigma = U of the last earlier target
// (plus, backward, its logarithm as a source; 0 in block 0).  Then
//     z_t = s_t + sum_{j<t} B(j,t) z_j,      B(j,t) = c(j,t) exp(G_t - G_j - w'(t,j)),
//     s_t = [ sum_{j in J} E(j,t) z_j + f_t ] / z_last,
//     E(j,t) = c(j,t) exp(G_t + G^J_last - G^J_j - w'(t,j)),   J the block before,
// w' being w without its logarithm and c the factor that stands for it (1/n
// forward; backward 1/(N-j), and in E (N-last)/(N-j)), f_t the farther sources
// in J's scale (an online log-sum-exp, finished a block earlier).  B, E and f
// are known before block J's z arrive, so the chain from block to block is
// 64 x 64 multiply-adds on four waves, a reduction, the in-block substitution
// (row by row of 16 lanes, xw_substitute) and the publication of 64 values: no
// exponential or logarithm, and no minimum.
//
// What bounds it: instructions on the chain.  One wave issues a dependent
// instruction every 8 cycles (measured, single and double precision alike), so
// the substitution's 60 dependent steps and their operands' addressing, the
// prefix sums' scans and every logarithm (470 cycles) show.  Hence the dense
// in-block matrix (xw_b), sums split before they are scanned (xw_stage), and
// work off the chain on other waves.  Both recursions with the exterior force
// took 10.9, 12.7, 25.2, 42.4 and 76.8 us at N = 4, 64, 256, 500 and 1000 with
// the block's exponentials, its logarithm and a substitution through scalar
// registers on the chain, and take 8.0, 9.5, 19.3, 31.1 and 54.1 us so.
//
// Range.  z stays near exp(-+ sum l_r / 2), 1e-116 .. 1e116 for the largest
// rings here, between one-particle and freely exchanging cycles.  A block with
// z outside 1e-140 .. 1e140, or after one whose z falls below 1e-140 of its
// largest (an entry of B or E that underflowed could count then; one that
// overflowed makes z infinite or NaN), is taken again by the exact min-plus
// form (xw_block_safe) and publishes XW_BAD, on which the next block takes its
// U like a farther block's and the exact form at once.  Rings that exchange
// strongly take it throughout, at about 7 us a block: a step of helium whose
// bead P of each particle lies at its neighbour's bead 1 takes 29.6 us at N=64,
// P=64, 64.6 at N=256 and 201 at N=1000, P=32 (18.9, 26.8 and 82 without
// exchange; 60, 100 and 359 with one workgroup per direction; 26.8, 99.5 and 628
// when the exact form took every earlier source again).
//
// Publication.  z, and off the chain U (plus, backward, the source's ln(N-q)),
// go to global arrays by relaxed device-scope atomic stores and are read by
// relaxed device-scope atomic loads until they differ from XW_EMPTY (NaN
// patterns that no result carries): the value is its own flag, so no fence is
// needed.  A wait ends after XW_SPIN polls at the latest (the flag of a lost
// wait is then set, and the host puts XW_EMPTY back, empty_published).  The last
// block's workgroup reads U of every block
// before it, each published after that block's own reads, so it puts XW_EMPTY
// back for the next launch.
//
// Progress.  A workgroup's block is its place in the order in which the
// workgroups started (xw_place), not its index in the grid, and it waits only for
// lower places.  So whatever it waits for is running already and waits only for
// still lower ones: launches of other streams or processes that hold compute
// units can delay a ring, but no set of waiting workgroups can keep each other's
// predecessors out, as they could where the dies start a grid's workgroups
// independently of each other.  The place costs an atomic per workgroup, 0.6 us
// where the chain is the longest part (V_B of N=65 20.4 -> 21.0 us a call, of
// N=500 36.7 -> 37.3, the observables of N=256 50.1 -> 50.9) and nothing where
// other work covers it (a helium step of N=256 or N=1000).
#pragma once

#include "exchange.hpp"

namespace pimdb {

// Threads of a workgroup (template parameter NT): 1024 where a ring has the
// card to itself; 256 beside other rings' work, where the idle waves of a
// waiting workgroup would hold registers that others could use.
constexpr int XW_THREADS = 1024;
constexpr unsigned long long XW_EMPTY = ~0ull, XW_BAD = ~1ull;
constexpr double XW_RANGE = 1e140;
constexpr long long XW_SPIN = 1ll << 22;             // polls of one wait (seconds)

// Global workspace of one ring: z and U of both directions, then the counter of
// xw_place.
__host__ __device__ inline size_t xw_places_word(int N) { return 4 * ((size_t)N + 1); }
__host__ __device__ inline size_t xw_pub_words(int N) { return xw_places_word(N) + 1; }
__host__ __device__ inline int xw_grid(int N) { return 2 * rec_blocks(N); }

// The place of this workgroup, one of n, among those of the launch in the order
// of their start.  counter: all bits set (XW_EMPTY) or as n such workgroups leave
// it (each launch of n counts from n - 1 round to n - 1).  lds: any word, free
// again on return.
__device__ __forceinline__ int xw_place(unsigned long long* counter, int n, double* lds) {
    if (threadIdx.x == 0) {
        const unsigned c = atomicInc((unsigned*)counter, (unsigned)(n - 1));
        *(volatile int*)lds = c >= (unsigned)(n - 1) ? 0 : (int)c + 1;
    }
    __syncthreads();
    const int place = uni(*(volatile int*)lds);
    __syncthreads();
    return place;
}

// The in-block matrix by rows of 16 sources and, in a row, by target: entry
// (j, t), 16 R <= j < 16 R + 16, t >= 16 R, at xw_b(j, t), so that a target's
// 16 coefficients are contiguous and, 18 apart, meet every bank alike; entries
// j >= t of the diagonal parts are 0.
constexpr int XW_BS = 18;
__host__ __device__ __forceinline__ constexpr int xw_brow(int R) { return XW_BS * (REC_B * R - 8 * R * (R - 1)); }
__device__ __forceinline__ int xw_b(int j, int t) {
    const int R = j / 16;
    return xw_brow(R) + (t - 16 * R) * XW_BS + (j - 16 * R);
}
constexpr int XW_MAT = xw_brow(4);
static_assert(XW_MAT >= REC_TRI + 2 * REC_B, "the safe form's arrays lie in the matrix's place");

// LDS doubles: the ring, the in-block matrix, the per-wave partials, the
// block's gauge, the previous block's gauge and factors as sources, the
// targets' logarithms as sources, the prefix sums' wave totals, the flags.
__host__ __device__ inline size_t xw_shared_doubles(int N, int D, int nw) {
    return (size_t)(2 * D + 2) * N + (size_t)XW_MAT + (size_t)nw * REC_B + 4 * REC_B + 3 * (size_t)nw + 1 + 2;
}
inline size_t xw_lds_bytes(int N, int D, int threads = XW_THREADS) {
    return sizeof(double) * xw_shared_doubles(N, D, threads / WAVE);
}

struct XwShared {
    double *a;                     // [XW_MAT] in-block matrix B
    double *psum;                  // [waves][REC_B]
    double *g;                     // [REC_B] gauge
    double *off, *rat;             // [REC_B] the previous block's: G_last - G_j, and backward (N-last)/(N-j)
    double *lq;                    // [REC_B] ln n of the targets; backward, ln(N-q) of them as sources
    double *tot;                   // [3 waves] wave totals: links, their split sums; then G_last of the previous block
    int* flag;                     // [0] the block left the range, [1] the previous one did, [2] its z fall too far
    double *x1, *xP, *Shi, *Slo;   // the ring [D][N], [D][N], [N], [N]
};

template <int NT>
__device__ __forceinline__ XwShared xw_carve(double* p, int N, int D) {
    constexpr int NW = NT / WAVE;
    XwShared s;
    s.a = p; p += XW_MAT;
    s.psum = p; p += NW * REC_B;
    s.g = p; p += REC_B;
    s.off = p; p += REC_B;
    s.rat = p; p += REC_B;
    s.lq = p; p += REC_B;
    s.tot = p; p += 3 * NW + 1;
    s.flag = (int*)p; p += 2;
    s.x1 = p; p += (size_t)D * N;
    s.xP = p; p += (size_t)D * N;
    s.Shi = p; p += N;
    s.Slo = p;
    return s;
}

// One bead's positions: axis a of particle i at p[a sa + i si].
struct BeadView {
    const double* p;
    long long sa, si;
    __device__ __forceinline__ double at(int a, int i) const { return p[a * sa + i * si]; }
};

// 1 / x within an ulp (x normal).
__device__ __forceinline__ double rcp_newton(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    return fma(r, fma(-x, r, 1.0), r);
}

// The gauge of target block I over the ring's particles, one target per lane
// (whole wave): positions loaded ahead (get), then the scan.
template <int DIR, int D>
struct XwGauge {
    double u[D], v[D];
    __device__ __forceinline__ void get(int I, int N, int lane, BeadView x1, BeadView xP) {
        const int n = 1 + I * REC_B + lane, idx = DIR == 0 ? min(n, N) - 1 : max(N - n, 0);
#pragma unroll
        for (int ax = 0; ax < D; ++ax) {
            u[ax] = x1.at(ax, idx);
            v[ax] = xP.at(ax, idx);
        }
    }
    __device__ __forceinline__ double scan(int I, int N, int lane, double bk, const Ring& r) const {
        const int n = 1 + I * REC_B + lane;
        double d[D];
#pragma unroll
        for (int ax = 0; ax < D; ++ax) d[ax] = ring_image(u[ax] - v[ax], r);
        // l / 2 = ln 2 / 2 log2(n) or log2(N - n + 1)
        const float c = (float)max(1, DIR == 0 ? n : N - n + 1);
        return wave_scan(fma(bk, norm2_fma<D>(d), (double)(0.34657359f * __builtin_amdgcn_logf(c))));
    }
};

// Beads 1 and P into LDS, the split prefix sums of the ring's links
// (exchange.hpp, Ring), the gauges of target block I (wave 1) and of the block
// before it (wave 2), the latter's factors and the targets' logarithms (wave
// 3), by the whole workgroup.  The links are split into multiples of
// q = 2^(e-40) and remainders before they are summed, 2^e <= their total <
// 2^(e+1): the multiples add exactly (at most 42 bits) in any order and the
// remainders' sums stay below N q / 2, so plain sums keep what a sum in double
// double kept, in a tenth of the instructions.  Every workgroup of a ring
// computes the same values.  Shi_out / Slo_out / xc_out (may be null) receive
// the sums and a copy [2][D][N] of the two beads.
template <int DIR, int D, int NT>
__device__ __forceinline__ Ring xw_stage(const XwShared& sh, int I, int N, double bt, BeadView x1, BeadView xP, double k,
                                         bool pbc, double L, double* Shi_out, double* Slo_out, double* xc_out) {
    constexpr int NW = NT / WAVE;
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const Ring r = make_ring(sh.x1, sh.xP, sh.Shi, sh.Slo, k, pbc, L);
    const double bk = bt * r.halfk;
    const int c = (N + NT - 1) / NT, v0 = tid * c;
    auto keep = [&](int a, int i, double u, double v) {
        const int e = a * N + i;
        sh.x1[e] = u;
        sh.xP[e] = v;
        if (xc_out) {
            xc_out[e] = u;
            xc_out[(size_t)D * N + e] = v;
        }
    };
    auto split_link = [&](int v) {   // (more than one link per thread: from LDS)
        double d[D];
#pragma unroll
        for (int ax = 0; ax < D; ++ax) d[ax] = ring_image(sh.x1[ax * N + v + 1] - sh.xP[ax * N + v], r);
        return norm2_fma<D>(d);
    };
    auto put = [&](int v, double h, double l) {
        sh.Shi[v] = h;
        sh.Slo[v] = l;
        if (Shi_out) {
            Shi_out[v] = h;
            Slo_out[v] = l;
        }
    };
    XwGauge<DIR, D> ga;
    const bool gauges = wave == 1 || (wave == 2 && I > 0);
    if (gauges) ga.get(I - (wave - 1), N, lane, x1, xP);
    double sum = 0.0;   // the thread's links
    if (c == 1) {       // a particle and its link per thread, all loads together
        if (tid < N) {
            double u[D], v[D], w[D], d[D];
#pragma unroll
            for (int ax = 0; ax < D; ++ax) {
                u[ax] = x1.at(ax, tid);
                v[ax] = xP.at(ax, tid);
                w[ax] = x1.at(ax, min(tid + 1, N - 1));
            }
#pragma unroll
            for (int ax = 0; ax < D; ++ax) {
                keep(ax, tid, u[ax], v[ax]);
                d[ax] = ring_image(w[ax] - v[ax], r);
            }
            if (tid < N - 1) sum = norm2_fma<D>(d);
        }
    } else {
        for (int e = tid; e < D * N; e += NT) {
            const int a = D == 1 ? 0 : e / N, i = e - a * N;
            keep(a, i, x1.at(a, i), xP.at(a, i));
        }
        __syncthreads();
        for (int v = v0; v < min(v0 + c, N - 1); ++v) sum += split_link(v);
    }
    if (tid < 4) sh.flag[tid] = 0;
    if (gauges) {
        const double g = ga.scan(I - (wave - 1), N, lane, bk, r);
        if (wave == 1) sh.g[lane] = g;
        if (wave == 2) {
            const double gl = wave_bcast_uniform(g, WAVE - 1);
            sh.off[lane] = gl - g;
            sh.tot[3 * NW] = gl;
        }
    }
    if (wave == 3) {
        const int n0 = 1 + I * REC_B;
        if (DIR == 1 && I > 0) sh.rat[lane] = (double)(N - n0 + 1) * rcp_newton((double)(N - n0 + REC_B - lane));   // j = n0 - 64 + lane
        sh.lq[lane] = log((double)(DIR == 0 ? n0 + lane : max(1, N - n0 - lane)));
    }
    // the quantum from the links' total, the same bits in every wave
    auto quantum = [](double total) { return total > 0.0 ? __builtin_amdgcn_frexp_exp(total) - 41 : 0; };
    if (N <= WAVE && c == 1) {   // one wave has every link
        if (wave == 0) {
            const int qe = quantum(wave_total(sum));
            const double h = ldexp(rint(ldexp(sum, -qe)), qe), l = sum - h;
            const double hs = wave_scan(h) - h, ls = wave_scan(l) - l;
            if (lane < N) put(lane, hs, ls);
        }
        __syncthreads();
        return r;
    }
    const double wt = wave_scan(sum);
    if (lane == WAVE - 1) sh.tot[wave] = wt;
    __syncthreads();
    auto row_scan = [](double v) {   // (at most 16 waves)
        v += dpp_or_zero<0x111, 0xF>(v);
        v += dpp_or_zero<0x112, 0xF>(v);
        v += dpp_or_zero<0x114, 0xF>(v);
        v += dpp_or_zero<0x118, 0xF>(v);
        return v;
    };
    const int qe = quantum(wave_bcast_uniform(row_scan(lane < NW ? sh.tot[lane] : 0.0), NW - 1));
    double h = 0.0, l = 0.0;
    auto add = [&](double x) {
        const double m = ldexp(rint(ldexp(x, -qe)), qe);
        h += m;
        l += x - m;
    };
    if (c == 1) add(sum);
    else
        for (int v = v0; v < min(v0 + c, N - 1); ++v) add(split_link(v));
    const double hi = wave_scan(h), li = wave_scan(l);
    if (lane == WAVE - 1) {
        sh.tot[NW + wave] = hi;
        sh.tot[2 * NW + wave] = li;
    }
    __syncthreads();
    double hs = hi - h, ls = li - l;
    if (wave > 0) {
        hs += wave_bcast_uniform(row_scan(lane < NW ? sh.tot[NW + lane] : 0.0), wave - 1);
        ls += wave_bcast_uniform(row_scan(lane < NW ? sh.tot[2 * NW + lane] : 0.0), wave - 1);
    }
    if (c == 1) {
        if (tid < N) put(tid, hs, ls);
    } else {
        for (int v = v0; v < min(v0 + c, N); ++v) {
            put(v, hs, ls);
            if (v < N - 1) {
                h = hs;
                l = ls;
                add(split_link(v));
                hs = h;
                ls = l;
            }
        }
    }
    __syncthreads();
    return r;
}

// The target side of w(n,q) of one lane, and w(n,q) without its logarithm
// (forward ln n, backward ln(N-q)).
template <int DIR, int D>
__device__ __forceinline__ RecTarget<D> xw_target(const XwShared& sh, int N, int n) {
    RecTarget<D> t;
    const int idx = DIR == 0 ? n - 1 : N - n;
    const double* xs = DIR == 0 ? sh.xP : sh.x1;
#pragma unroll
    for (int a = 0; a < D; ++a) t.x[a] = xs[a * N + idx];
    t.shi = sh.Shi[idx];
    t.slo = sh.Slo[idx];
    t.lg = 0.0;
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
    return bk * (sd + norm2_fma<D>(d));
}

__device__ __forceinline__ unsigned long long xw_bits(double v) { return (unsigned long long)__double_as_longlong(v); }
// Stores a value for the other workgroups (a NaN with the empty pattern as
// another NaN).
__device__ __forceinline__ void xw_publish(unsigned long long* p, double v) {
    unsigned long long b = xw_bits(v);
    if (b == XW_EMPTY) b = 0x7FF8000000000000ull;
    __hip_atomic_store(p, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Whether a wait ends after this many polls without its values: its own bound,
// or the flag of another one that did (looked at every 1024 polls).
__device__ __forceinline__ bool xw_give_up(long long polls, int* status) {
    if (polls >= XW_SPIN) {
        raise_lost_wait(status);
        return true;
    }
    return polls % 1024 == 0 && (__hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) & 0xFF00) != 0;
}
// The 64 values of a finished block from p, one per lane (whole wave; p[at]
// for the lane).
__device__ __forceinline__ double xw_wait(unsigned long long* p, int at, int* status) {
    // (asleep between polls: what is awaited here is off the chain, and the polls
    // of the whole card share the caches with those that are on it)
    unsigned long long b = XW_EMPTY;
    long long spin = 0;
    for (;;) {
        b = __hip_atomic_load(p + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__all(b != XW_EMPTY)) break;
        if (xw_give_up(++spin, status)) break;
        __builtin_amdgcn_s_sleep(4);
    }
    return __longlong_as_double((long long)b);
}

// One block with the exact min-plus shifts (exchange.hpp, steps (1)-(4)), for
// blocks whose z left the range: rings that exchange strongly (a two-particle
// cycle that is favoured by e^10 moves z by that).  Every earlier source is in
// the waves' online sums m, s already, all but the previous block's since
// before the wait; the in-block weights (xw_safe_weights) need no U at all.  All
// threads; U of the lane's target in every lane of wave 0.
template <int DIR, int D, int NT>
__device__ __noinline__ void xw_safe_weights(int N, int n0, int nb, double bk, const Ring r, const XwShared sh) {
    constexpr int NW = NT / WAVE;
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
    __syncthreads();   // (the matrix is no longer read)
    for (int vr = wave; vr < REC_B / 2; vr += NW) {
        int t, j;
        rec_tri(vr, lane, t, j);
        if (t < 0) continue;
        double w = INFINITY;
        if (t < nb) w = xw_w<DIR, D>(sh, r, bk, N, xw_target<DIR, D>(sh, N, n0 + t), n0 + j) + sh.lq[DIR == 0 ? t : j];
        sh.a[rec_idx(j, t)] = w;
    }
}
// forward: sh.lq holds the targets' logarithms.
template <int NT>
__device__ __noinline__ double xw_block_safe(bool forward, int nb, const XwShared sh, double m, double s) {
    constexpr int NW = NT / WAVE;
    double *R = sh.a + REC_TRI, *z = R + REC_B;   // (the triangle and these in the matrix's place)
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
    const int tl = min(lane, nb - 1);
    __syncthreads();   // (the partials are no longer read)
    m += forward ? sh.lq[tl] : 0.0;
    sh.psum[wave * REC_B + lane] = lane < nb ? m : INFINITY;
    __syncthreads();
    if (wave == 0) {
        double rr = INFINITY;
        for (int w = 0; w < NW; ++w) rr = fmin(rr, sh.psum[w * REC_B + lane]);
        rec_inblock_seq<0>(sh.a, lane, rr, R);
    }
    __syncthreads();
    sh.psum[wave * REC_B + lane] = lane < nb && s > 0.0 ? s * exp_pair(R[lane] - m) : 0.0;
    for (int vr = wave; vr < REC_B / 2; vr += NW) {
        int t, j;
        rec_tri(vr, lane, t, j);
        if (t >= 0) sh.a[rec_idx(j, t)] = t < nb ? exp_pair(-(sh.a[rec_idx(j, t)] + R[j] - R[t])) : 0.0;
    }
    __syncthreads();
    double u = 0.0;
    if (wave == 0) {
        double z0 = 0.0;
        for (int w = 0; w < NW; ++w) z0 += sh.psum[w * REC_B + lane];
        rec_inblock_seq<1>(sh.a, lane, z0, z);
        u = R[lane] - log(z[lane]);
    }
    __syncthreads();
    return u;
}

// Row R (lanes 16R .. 16R+15) of v in every row.
template <int R>
__device__ __forceinline__ unsigned row_everywhere(unsigned v) {
    const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    const unsigned x = h[R / 2];
    const auto q = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    return q[R % 2];
}
template <int R>
__device__ __forceinline__ double row_everywhere(double v) {
    return __hiloint2double((int)row_everywhere<R>((unsigned)__double2hiint(v)),
                            (int)row_everywhere<R>((unsigned)__double2loint(v)));
}
// w += c * (lane J of the row's w), and acc += c * (lane J of the row's w):
// one instruction, the broadcast being its DPP operand (two wait states after
// the write of w).
template <int J>
__device__ __forceinline__ void row_step(double& w, double c) {
    asm("s_nop 1\n\tv_fmac_f64_dpp %0, %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "+v"(w) : "v"(c), "n"(J));
}
template <int J>
__device__ __forceinline__ void row_add(double& acc, double w, double c) {
    asm("s_nop 1\n\tv_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
        : "+v"(acc)
        : "v"(w), "v"(c), "n"(J));
}
// 16 contiguous coefficients (16-byte aligned).
__device__ __forceinline__ void xw_coefs(const double* a, double (&d)[16]) {
#pragma unroll
    for (int j = 0; j < 16; j += 2) {
        const double2 v = *(const double2*)(a + j);
        d[j] = v.x;
        d[j + 1] = v.y;
    }
}
template <int J>
__device__ __forceinline__ void row_steps(double& w, const double (&d)[16]) {
    if constexpr (J < 15) {
        row_step<J>(w, d[J]);
        row_steps<J + 1>(w, d);
    }
}
template <int J>
__device__ __forceinline__ void row_adds(double& v0, double& v1, double w, const double (&u)[16]) {
    if constexpr (J < 16) {
        row_add<J>(v0, w, u[J]);
        row_add<J + 1>(v1, w, u[J + 1]);
        row_adds<J + 2>(v0, v1, w, u);
    }
}
// One row of 16 targets: its own substitution in every row at once, then its
// share of the later rows' sums.  d: the row's own coefficients, replaced by
// the next row's.
template <int R>
__device__ __forceinline__ void xw_row(const double* a, int lane, int nb, double& v, double& z, double (&d)[16]) {
    if (16 * R >= nb) return;   // (uniform)
    double u[16];
    if constexpr (R < 3) xw_coefs(a + xw_brow(R) + max(lane - 16 * R, 0) * XW_BS, u);
    double w = row_everywhere<R>(v);
    row_steps<0>(w, d);
    z = lane / 16 == R ? w : z;
    if constexpr (R < 3) {
        xw_coefs(a + xw_brow(R + 1) + lane % 16 * XW_BS, d);
        double v1 = 0.0;
        row_adds<0>(v, v1, w, u);
        v += v1;
        xw_row<R + 1>(a, lane, nb, v, z, d);
    }
}
// The substitution z_t = s_t + sum_{j<t} B(j,t) z_j of one wave, lane t
// holding s_t, for a block of nb targets.  Values of rows already done are not
// used again, so the later sums run over all rows without a mask.  A step is
// one multiply-add with the broadcast in it (16 cycles) instead of two
// cross-lane reads through scalar registers and a multiply-add (52).
__device__ __forceinline__ double xw_substitute(const double* a, int lane, int nb, double v) {
    double d[16], z = 0.0;
    xw_coefs(a + lane % 16 * XW_BS, d);
    xw_row<0>(a, lane, nb, v, z, d);
    return z;
}

// The 16 z of a row of the previous block in every row of lanes and its last
// one, zl (XW_BAD in place of both if that block left the range).
__device__ __forceinline__ void xw_wait_z(unsigned long long* p, int row, int lane, int* status, double& z, double& zl) {
    unsigned long long b = XW_EMPTY, e = XW_EMPTY;
    for (long long spin = 0;; ++spin) {
        b = __hip_atomic_load(p + 16 * row + lane % 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        e = __hip_atomic_load(p + REC_B - 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__all(b != XW_EMPTY && e != XW_EMPTY)) break;
        if (xw_give_up(spin + 1, status)) {
            b = e = XW_BAD;
            break;
        }
    }
    z = __longlong_as_double((long long)b);
    zl = __longlong_as_double((long long)e);
}

// Target block I of one recursion on one workgroup of NT threads (the ring
// staged).  zpub, upub: this direction's published values [N+1].
template <int DIR, int D, int NT>
__device__ __forceinline__ void xw_block(int I, int N, double bt, const Ring& r, const XwShared& sh,
                                         unsigned long long* __restrict__ zpub, unsigned long long* __restrict__ upub,
                                         double* __restrict__ V, double* __restrict__ Vb, double* __restrict__ VB,
                                         int* __restrict__ status) {
    constexpr int NW = NT / WAVE, XW_SRC = REC_B / NW;   // farther sources of a block per wave
    constexpr int ZW = 4;                                // waves that take the previous block's z, a row each
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
    const int tl = min(lane, nb - 1), tn = n0 + tl;   // the lane's target (clamped)
    const int qn = n0 - REC_B;                        // the previous block's first target (I > 0)
    const double g = sh.g[lane];
    const double cn = DIR == 0 ? rcp_newton((double)tn) : 1.0;       // the target's factor
    const double c0 = DIR == 0 ? cn : rcp_newton((double)N);         // source 0's
    const RecTarget<D> tg = xw_target<DIR, D>(sh, N, tn);
    // the z waves' coefficients of the previous block
    double E[16];
    if (I > 0 && wave < ZW) {
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int j = 16 * wave + u;
            E[u] = exp_pair((g + sh.off[j]) - xw_w<DIR, D>(sh, r, bk, N, tg, qn + j)) * (DIR == 0 ? cn : sh.rat[j]);
        }
    }
    // the in-block matrix, by the other waves if there are any and E was to do
    const int w0 = NW > ZW && I > 0 ? ZW : 0;
    if (wave >= w0) {
        for (int e = tid - w0 * WAVE; e < 4 * 256; e += NT - w0 * WAVE) {   // zeros of the diagonal parts
            const int t = e / 16, j = t / 16 * 16 + e % 16;
            if (j >= t) sh.a[xw_b(j, t)] = 0.0;
        }
        for (int vr = wave - w0; vr < REC_B / 2; vr += NW - w0) {
            int t, j;
            rec_tri(vr, lane, t, j);
            if (t < 0) continue;
            double c = 0.0;
            if (t < nb) {
                const double w = xw_w<DIR, D>(sh, r, bk, N, xw_target<DIR, D>(sh, N, n0 + t), n0 + j);
                c = exp_pair((sh.g[t] - sh.g[j]) - w) * rcp_newton((double)(DIR == 0 ? n0 + t : N - n0 - j));
            }
            sh.a[xw_b(j, t)] = c;
        }
    }
    // farther sources: source 0 on wave 0, then XW_SRC of every block per
    // wave, four in registers at a time
    const int q0 = wave * XW_SRC;
    double m = INFINITY, s = 0.0, before = 0.0;   // before: the scale of the previous block's z
    auto far = [&](int J) {
        constexpr int XQ = 4;
        const int qb = J * REC_B + 1;
        double w[XQ];
#pragma unroll
        for (int u = 0; u < XQ; ++u) w[u] = xw_w<DIR, D>(sh, r, bk, N, tg, qb + q0 + u);
        const double v = xw_wait(upub + qb, lane, status);
#pragma unroll 1
        for (int c = 0; c < XW_SRC; c += XQ) {
            double mn = m;
#pragma unroll
            for (int u = 0; u < XQ; ++u) {
                if (c > 0) w[u] = xw_w<DIR, D>(sh, r, bk, N, tg, qb + q0 + c + u);
                w[u] += wave_bcast_uniform(v, q0 + c + u);
                mn = fmin(mn, w[u]);
            }
            s *= exp_pair(mn - m);   // m = inf: s = 0 stays 0
            m = mn;
#pragma unroll
            for (int u = 0; u < XQ; ++u) s += exp_pair(mn - w[u]);
        }
        return wave_bcast_uniform(v, REC_B - 1);
    };
    if (wave == 0) {
        m = xw_w<DIR, D>(sh, r, bk, N, tg, 0);
        s = DIR == 0 ? 1.0 : c0;   // (forward the target's factor comes last)
    }
    double z = 0.0, sigma = 0.0;   // wave 0: the lane's s_t, then z_t
    bool safe = false;             // (uniform) the exact form
    if (I == 0) {
        z = s * cn * exp_pair(g - m);
        __syncthreads();
    } else {
        for (int J = 0; J < I - 1; ++J) before = far(J);
        const double cf = DIR == 0 ? cn : (double)(N - n0 + 1);
        double acc = s > 0.0 ? s * cf * exp_pair((before + (sh.tot[3 * NW] + g)) - m) : 0.0;
        if (NW > ZW) {
            sh.psum[wave * REC_B + lane] = acc;
        }
        __syncthreads();   // (the matrix is complete, too)
        if (wave < ZW) {
            if (NW > ZW) {   // the slots of waves wave, wave + 4, ...; the first is then written
                acc = 0.0;
#pragma unroll
                for (int w = 0; w < NW / ZW; ++w) acc += sh.psum[(wave + w * ZW) * REC_B + lane];
            }
            // (in registers before the wait: the compiler would move them into the branch)
#pragma unroll
            for (int u = 0; u < 16; ++u) asm volatile("" : "+v"(E[u]));
            asm volatile("" : "+v"(acc));
            double zv, zl;
            xw_wait_z(zpub + qn, wave, lane, status, zv, zl);
            if (xw_bits(zl) != XW_BAD) {
                double v1 = 0.0;
                row_adds<0>(acc, v1, zv, E);
                acc = (acc + v1) * rcp_newton(zl);
                if (!__all(zl * XW_RANGE >= zv) && lane == 0) sh.flag[2] = 1;
            } else if (lane == 0) {
                sh.flag[1] = 1;
            }
            sh.psum[wave * REC_B + lane] = acc;
        }
        __syncthreads();
        if (sh.flag[1]) {   // (uniform) the block before left the range: this one will, too
            if (wave == 0 && !last) __hip_atomic_store(zpub + n0 + lane, XW_BAD, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            xw_safe_weights<DIR, D, NT>(N, n0, nb, bk, r, sh);
            far(I - 1);
            safe = true;
        } else {
            const double* ps = sh.psum + lane;
            z = (ps[0] + ps[REC_B]) + (ps[2 * REC_B] + ps[3 * REC_B]);
        }
    }
    double u = 0.0;
    if (!safe) {
        if (wave == 0) {
            z = xw_substitute(sh.a, lane, nb, lane < nb ? z : 0.0);
            const bool all = __all(lane >= nb || (z >= 1.0 / XW_RANGE && z <= XW_RANGE)) && !sh.flag[2];
            if (!last) {
                const unsigned long long b = all ? xw_bits(z) : XW_BAD;
                __hip_atomic_store(zpub + n0 + lane, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            if (I > 0) sigma = wave_bcast_uniform(xw_wait(upub + qn, lane, status), REC_B - 1);   // (all 64: see the reset below)
            if (all) {
                u = (sigma + g) - log(z);
                if (!last) xw_publish(upub + n0 + lane, DIR == 0 ? u : u + sh.lq[lane]);
            }
            if (lane == 0) sh.flag[0] = all ? 0 : 1;
        }
        __syncthreads();
        safe = sh.flag[0] != 0;
        if (safe) {
            xw_safe_weights<DIR, D, NT>(N, n0, nb, bk, r, sh);
            if (I > 0) far(I - 1);
        }
    }
    if (safe) {
        u = xw_block_safe<NT>(DIR == 0, nb, sh, m, s);
        if (wave == 0) {
            if (lane < nb && !isfinite(u)) raise_status(status);
            if (!last) xw_publish(upub + n0 + lane, DIR == 0 ? u : u + sh.lq[lane]);
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
        for (int q = tid; q < n0; q += NT) {
            __hip_atomic_store(zpub + q, XW_EMPTY, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(upub + q, XW_EMPTY, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// The workgroup in place b of xw_grid(N): block b / 2, forward (even) or backward
// (odd); lower blocks first.  pub: xw_pub_words(N) words, all but the counter
// XW_EMPTY on entry and on return.  Block 0's forward workgroup writes the prefix sums and, where
// asked (xc, VB not null), the beads' copy and V[N].
template <int D, int NT>
__device__ __forceinline__ void xw_recursions(double* smem, int b, int N, double bt, double k, int pbc, double L,
                                              BeadView x1, BeadView xP, double* __restrict__ V,
                                              double* __restrict__ Vb, double* __restrict__ VB,
                                              double* __restrict__ Shi, double* __restrict__ Slo, double* __restrict__ xc,
                                              unsigned long long* __restrict__ pub, int* __restrict__ status) {
    const XwShared sh = xw_carve<NT>(smem, N, D);
    const bool first = b == 0, fwd = (b & 1) == 0;
    const int I = b >> 1;
    double *sh_out = first ? Shi : nullptr, *sl_out = first ? Slo : nullptr, *x_out = first ? xc : nullptr;
    if (fwd) {
        const Ring r = xw_stage<0, D, NT>(sh, I, N, bt, x1, xP, k, pbc != 0, L, sh_out, sl_out, x_out);
        xw_block<0, D, NT>(I, N, bt, r, sh, pub, pub + N + 1, V, Vb, VB, status);
    } else {
        const Ring r = xw_stage<1, D, NT>(sh, I, N, bt, x1, xP, k, pbc != 0, L, nullptr, nullptr, nullptr);
        xw_block<1, D, NT>(I, N, bt, r, sh, pub + 2 * (N + 1), pub + 3 * (N + 1), V, Vb, nullptr, status);
    }
}

// The place of workgroup wg of a launch that xw_grid(N) workgroups of one ring
// take part in (a single block waits for nothing).
__device__ __forceinline__ int xw_ring_place(unsigned long long* pub, int N, int wg, double* lds) {
    const int n = xw_grid(N);
    return n > 2 ? xw_place(pub + xw_places_word(N), n, lds) : wg;
}

template <int D>
static __global__ void __launch_bounds__(XW_THREADS)
k_exchange_wide(int N, double bt, double k, int pbc, double L, BeadView x1, BeadView xP, double* __restrict__ V,
                double* __restrict__ Vb, double* __restrict__ VB, double* __restrict__ Shi, double* __restrict__ Slo,
                double* __restrict__ xc, unsigned long long* __restrict__ pub, int* __restrict__ status) {
    extern __shared__ __align__(16) double smem[];
    const int b = xw_ring_place(pub, N, blockIdx.x, smem);
    xw_recursions<D, XW_THREADS>(smem, b, N, bt, k, pbc, L, x1, xP, V, Vb, VB, Shi, Slo, xc, pub, status);
}

}  // namespace pimdb
