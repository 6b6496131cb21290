// small_steps.hpp -- many MD steps of a handful of particles in one launch of
// one workgroup, the whole state in LDS.
//
// Reference: Simulation::run (src/simulation.cpp:246-259) as in steps.hpp, the
// recursions of src/bosonic_exchange/quadratic_bosonic_exchange.cpp:73-128 and
// the exterior forces :159-215 of higj/pimd-b.
//
// Why.  A step of N=4, P=32 is two kernels of 11.1 us together, of which the
// start of a kernel and the loads behind it are more than half; here 5.8, and
// 4.2 against 9.8 without exchange.  What bounds it: the recursion's chain (0.45
// us a target, beside noise and forces on the other waves), then the barriers.
// Larger rings and states are faster over the card (us a step, two kernels and
// here: N=8, P=64 15.8, 9.9; N=16, P=8 11.0, 12.9; without exchange N=16, P=32
// 9.4, 7.9, and with normal-mode coupling N=16, P=42 12.6, 14.8).
//
// A step here (the same keys of the noise and the same updates as steps.hpp):
//   A  waves 0 and 1 the two recursions, one target after another, lane q
//      holding source q (its links summed as the targets go by, so no difference
//      of sums is taken); the other waves the forces and the noise
//   B  exterior forces, 16 lanes per particle and bead; normal-mode coupling of
//      the noise
//   C  the momenta with their mean taken out, the positions
#pragma once

#include "steps.hpp"

namespace pimdb {

constexpr int SMALL_N = 16;            // particles
constexpr int SMALL_RING = 8;          // particles with exchange (half a DPP row of sources)
constexpr int SMALL_E = 1536;          // elements P D N
constexpr int SMALL_THREADS = 1024;
constexpr int SMALL_WAVES = SMALL_THREADS / WAVE;
constexpr int SMALL_STEPS = 512;       // of one launch (a few ms)
constexpr int SMALL_EACH = (SMALL_E + SMALL_THREADS - 1) / SMALL_THREADS;

__host__ __device__ inline size_t small_lds_doubles(int N, int P, int D, bool nm) {
    return (size_t)P * D * N * (nm ? 5 : 4) + (nm ? (size_t)P * P : 0);
}

// v of the row's lanes combined in every lane of the row (row_ror 1, 2, 4, 8).
template <int N>
__device__ __forceinline__ double row_turn(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x120 | N, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x120 | N, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double row_min(double v) {
    v = fmin(v, row_turn<1>(v));
    v = fmin(v, row_turn<2>(v));
    v = fmin(v, row_turn<4>(v));
    return fmin(v, row_turn<8>(v));
}
__device__ __forceinline__ double row_sum(double v) {
    v += row_turn<1>(v);
    v += row_turn<2>(v);
    v += row_turn<4>(v);
    return v + row_turn<8>(v);
}

// One recursion on one wave (each of its four rows alike): V[0..N] forward
// (DIR 0), Vb[1..N] backward, in units of 1 / beta~.  x1, xP: [D][N].  What a
// target takes without its sources' U is made first, for all targets; the chain
// from target to target is then a minimum and a sum over the row, an
// exponential and a logarithm (N=16: 0.8 us a target in one pass, 0.45 so).
// links (forward): |x1[l+1] - xP[l]|^2.
template <int DIR, int D>
__device__ __forceinline__ void small_recursion(const double* x1, const double* xP, int N, double bt, const Ring& r,
                                                double* V, double* links, int* status) {
    const int lane = threadIdx.x % WAVE, l = lane % 16, li = min(l, N - 1);   // the source's particle
    const double bk = bt * r.halfk;
    const int steps = DIR == 0 ? N : N - 1;   // targets: particle v = n-1 forward, u backward
    double xs[D], ys[D], d[D];                // of the lane's particle: the source bead's and the target bead's
#pragma unroll
    for (int a = 0; a < D; ++a) {
        xs[a] = (DIR == 0 ? x1 : xP)[a * N + li];
        ys[a] = (DIR == 0 ? xP : x1)[a * N + li];
        d[a] = ring_image(x1[a * N + min(li + 1, N - 1)] - xP[a * N + li], r);
    }
    const double link = norm2_fma<D>(d);
    if (DIR == 0 && lane < N) links[lane] = link;
    // the backward source's factor 1 / (v+1), the forward target's 1 / n
    const double lv = DIR == 0 ? 0.0 : log_unit<true>((double)(li + 1)), inv = rcp_newton((double)(li + 1));
    double T = 0.0, w[SMALL_RING];               // links between source and target; the terms without U
#pragma unroll
    for (int k = 0; k < SMALL_RING; ++k) {
        if (k >= steps) break;
        const int t = DIR == 0 ? k : N - 1 - k;
        if (k > 0) {   // the link t-1 -> t (forward), t -> t+1 (backward)
            const double c = wave_bcast_uniform(link, DIR == 0 ? t - 1 : t);
            if (DIR == 0 ? l < t : l > t) T += c;
        }
#pragma unroll
        for (int a = 0; a < D; ++a) d[a] = ring_image(xs[a] - wave_bcast_uniform(ys[a], t), r);
        const bool live = DIR == 0 ? l <= t : (l >= t && l < N);
        w[k] = live ? fma(bk, T + norm2_fma<D>(d), lv) : INFINITY;
    }
    double u = 0.0;   // U of the source: 0 for source 0 forward and for v = N-1 backward
#pragma unroll
    for (int k = 0; k < SMALL_RING; ++k) {
        if (k >= steps) break;
        const int t = DIR == 0 ? k : N - 1 - k;
        const double y = w[k] + u, m = row_min(y);
        double sum = row_sum(exp_pair(m - y));   // (0 for a lane without a source)
        if (DIR == 0) sum *= wave_bcast_uniform(inv, t);
        const double ut = m - log_unit<true>(sum);
        if (DIR == 0 ? l == t + 1 : l == t - 1) u = ut;
        if (lane == 0) {
            if (!isfinite(ut)) raise_status(status);
            V[DIR == 0 ? t + 1 : t] = ut;
        }
    }
    if (lane == 0) V[DIR == 0 ? 0 : N] = 0.0;
}

// nsteps steps.  x, p, f and the step counter as k_step_integrate leaves them.
template <int D, int KIND>
static __global__ void __launch_bounds__(SMALL_THREADS) k_small_steps(StepArgs s, int nsteps) {
    extern __shared__ __align__(16) double smem[];
    __shared__ double V[SMALL_RING + 1], Vb[SMALL_RING + 1], links[SMALL_RING], red[D][SMALL_WAVES];
    const int N = s.fa.N, P = s.fa.P, nc = D * N, E = P * nc;
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const bool nm = s.thermostat && s.nm, pbc = s.fa.pbc != 0, boson = s.fa.bosonic != 0;
    double *x = smem, *p = x + E, *f = p + E, *H = f + E, *G = H + E, *CT = G + E;   // G, CT: nm only
    for (int e = tid; e < E; e += SMALL_THREADS) {
        x[e] = s.x[e];
        p[e] = s.p[e];
        f[e] = s.f[e];
        H[e] = 0.0;
    }
    if (nm)
        for (int e = tid; e < P * P; e += SMALL_THREADS) CT[e] = s.CTt[e];
    const uint32_t step0 = (uint32_t)*s.ctr;
    const Ring ring = make_ring(x, x + (size_t)(P - 1) * nc, nullptr, nullptr, s.fa.k_spring, pbc, s.fa.L);
    const PairParams pp = make_pair_params(s.fa.L, s.fa.pbc, s.fa.cutoff, s.fa.cut2, s.fa.int_k, s.fa.strength);
    __syncthreads();

    auto noise = [&](const StepCoef& co, int mode, uint32_t step, int t0) {   // by threads t0 and up
        if (!s.thermostat) return;
        double* out = nm ? G : H;
        for (int e = tid - t0; e < (P + 1) / 2 * nc; e += SMALL_THREADS - t0) {
            const int m = e / nc, col = e - m * nc;
            double g0 = 0.0, g1 = 0.0, h0, h1;
            if (mode != STEP_OPEN) {
                gauss2<false>((uint32_t)e, step, 1u, 0u, s.seed, g0, g1);
                g0 *= co.k2;
                g1 *= co.k2;
            }
            if (mode != STEP_CLOSE) {
                gauss2<false>((uint32_t)e, step, 0u, 0u, s.seed, h0, h1);
                g0 += h0;
                g1 += h1;
            }
            out[2 * m * nc + col] = s.c2 * g0;
            if (2 * m + 1 < P) out[(2 * m + 1) * nc + col] = s.c2 * g1;
        }
    };
    auto couple = [&]() {   // H = C^T G
        if (!nm) return;
        for (int e = tid; e < E; e += SMALL_THREADS) {
            const int b = e / nc, col = e - b * nc;
            double t = 0.0;
#pragma unroll 4
            for (int k = 0; k < P; ++k) t = fma(CT[k * P + b], G[k * nc + col], t);
            H[e] = t;
        }
    };
    auto forces = [&](int t0) {
        for (int t = tid - t0; t < P * N; t += SMALL_THREADS - t0) {
            const int b = t / N, i = t - b * N;
            const double* xb = x + (size_t)b * nc;
            double xi[D], acc[D], fe[D];
#pragma unroll
            for (int a = 0; a < D; ++a) {
                xi[a] = xb[a * N + i];
                acc[a] = 0.0;
                fe[a] = 0.0;
            }
            if constexpr (KIND != POT_FREE) {
                if (s.fa.cutoff != 0.0) {
                    auto run = [&](auto img) {
                        constexpr int IMG = decltype(img)::value;
                        for (int j = 0; j < N; ++j) {
                            double xj[D], d[D], g;
#pragma unroll
                            for (int a = 0; a < D; ++a) xj[a] = xb[a * N + j];
                            if (j != i && pair_grad<D, KIND, IMG>(xi, xj, pp, d, g)) {
#pragma unroll
                                for (int a = 0; a < D; ++a) acc[a] = fma(-g, d[a], acc[a]);
                            }
                        }
                    };
                    switch (pair_image(pp)) {
                    case 0: run(std::integral_constant<int, 0>()); break;
                    case 1: run(std::integral_constant<int, 1>()); break;
                    default: run(std::integral_constant<int, 2>()); break;
                    }
                }
            }
            ext_force<D>(s.fa.ext, xi, fe);
            const double* xp = x + (size_t)(b == 0 ? P - 1 : b - 1) * nc;
            const double* xn = x + (size_t)(b == P - 1 ? 0 : b + 1) * nc;
            const bool exchange = boson && (b == 0 || b == P - 1);
#pragma unroll
            for (int a = 0; a < D; ++a) {
                const double phys = fe[a] + acc[a];
                const int o = a * N + i;
                f[b * nc + o] = exchange ? phys
                                         : s.fa.k_spring * (disp(xi[a], xp[o], pbc, s.fa.L) + disp(xi[a], xn[o], pbc, s.fa.L)) + phys;
            }
        }
    };
    // exterior forces of beads 1 and P (exchange.hpp, exterior_force): row of 16
    // lanes per particle and bead, lane j the partner
    auto exterior = [&]() {
        const int task = tid / 16, j = tid % 16;
        const int which = task < N ? 0 : 1, l = task - which * N;
        if (task >= 2 * N) return;   // (whole rows)
        const double *x1 = x, *xP = x + (size_t)(P - 1) * nc;
        const double *self = which == 0 ? x1 : xP, *other = which == 0 ? xP : x1;
        const int jc = min(j, N - 1), row = which == 0 ? jc : l, col = which == 0 ? l : jc;
        double d[D], S[D];
#pragma unroll
        for (int a = 0; a < D; ++a) d[a] = ring_image(other[a * N + jc] - self[a * N + l], ring);
        const bool link = col == row + 1, live = j < N && col <= row + 1;
        double T = 0.0;   // links of the cycle col .. row
        for (int k = col; k < row; ++k) T += links[k];
        const double e = s.bt * ring.halfk * (T + norm2_fma<D>(d));
        const double VN = V[N];
        const double w = link ? V[row + 1] + Vb[row + 1] : V[col] + e + Vb[row + 1];
        const double ex = exp_minimax(VN - w);
        const double pr = !live ? 0.0 : link ? 1.0 - ex : ex / (double)(row + 1);
        const double* near = x + (size_t)(which == 0 ? 1 % P : P - 2) * nc;
#pragma unroll
        for (int a = 0; a < D; ++a) {
            S[a] = row_sum(pr * d[a]) + ring_image(near[a * N + l] - self[a * N + l], ring);
            if (j == 0) f[(which == 0 ? 0 : (P - 1) * nc) + a * N + l] += s.fa.k_spring * S[a];
        }
    };
    auto integrate = [&](const StepCoef& co, int mode) {
        double v[SMALL_EACH], c[D];
#pragma unroll
        for (int a = 0; a < D; ++a) c[a] = 0.0;
#pragma unroll
        for (int k = 0; k < SMALL_EACH; ++k) {
            const int e = tid + k * SMALL_THREADS;
            if (e >= E) continue;
            v[k] = step_kept(co, fma(co.beta, f[e], p[e]), H[e]);
            const int ax = e % nc / N;
#pragma unroll
            for (int a = 0; a < D; ++a) c[a] += a == ax ? v[k] : 0.0;
        }
        if (s.fixcom) {
#pragma unroll
            for (int a = 0; a < D; ++a) {
                c[a] = wave_total(c[a]);
                if (lane == 0) red[a][wave] = c[a];
            }
            __syncthreads();
#pragma unroll
            for (int a = 0; a < D; ++a) {
                c[a] = 0.0;
                for (int w = 0; w < SMALL_WAVES; ++w) c[a] += red[a][w];
                c[a] /= (double)(N * P);
            }
        }
#pragma unroll
        for (int k = 0; k < SMALL_EACH; ++k) {
            const int e = tid + k * SMALL_THREADS;
            if (e >= E) continue;
            double w = v[k];
            if (s.fixcom) {
                const int ax = e % nc / N;
#pragma unroll
                for (int a = 0; a < D; ++a)
                    if (a == ax) w -= c[a];
            }
            if (mode != STEP_CLOSE) {
                w = fma(co.gamma, f[e], w);
                x[e] = fma(s.dt_m, w, x[e]);
            }
            p[e] = w;
        }
        __syncthreads();
    };

    noise(step_coef(s, STEP_OPEN), STEP_OPEN, step0, 0);
    __syncthreads();
    couple();
    if (nm) __syncthreads();
    integrate(step_coef(s, STEP_OPEN), STEP_OPEN);
    for (int k = 1; k <= nsteps; ++k) {
        const int mode = k < nsteps ? STEP_FULL : STEP_CLOSE;
        const StepCoef co = step_coef(s, mode);
        if (boson && wave < 2) {
            if (wave == 0) small_recursion<0, D>(x, x + (size_t)(P - 1) * nc, N, s.bt, ring, V, links, s.status);
            else small_recursion<1, D>(x, x + (size_t)(P - 1) * nc, N, s.bt, ring, Vb, links, s.status);
        } else {
            const int t0 = boson ? 2 * WAVE : 0;
            noise(co, mode, step0 + (uint32_t)k, t0);
            forces(t0);
        }
        __syncthreads();
        if (boson) exterior();
        couple();
        if (boson || nm) __syncthreads();
        integrate(co, mode);
    }
    for (int e = tid; e < E; e += SMALL_THREADS) {
        s.x[e] = x[e];
        s.p[e] = p[e];
        s.f[e] = f[e];
    }
    if (tid == 0) *s.ctr += nsteps;
}

}  // namespace pimdb
