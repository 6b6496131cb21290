// observables.hpp -- per-bead sums, energies and the bosonic estimators behind
// the energy, classical and bosonic observables.
//
// Reference: EnergyObservable (src/observables/energy.cpp:21-111),
// ClassicalObservable (src/observables/classical.cpp:131-188),
// BosonicObservable (src/observables/bosonic.cpp:17-22),
// Simulation::classicalSpringEnergy (src/simulation.cpp:464-486),
// BosonicExchange::primEstimator / getDistinctProbability /
// getLongestProbability (quadratic_bosonic_exchange.cpp:222-279).
//
// The primitive estimator's recursion (:250-279),
//     prim[m] = sum_{j<m} W(m,j) (prim[j] - ecyc(j, m-1)),
//     W(m,j)  = exp(-bt (ecyc(j,m-1) + V[j] - V[m])) / m,
// is linear, and its adjoint from prim[N] is known: the weight of term m is
// G_m = exp(-bt (V[m] + Vb[m] - V[N])), and G_m W(m,j) is the connection
// probability P[m-1][j] (:142-157).  So
//     prim[N] = - sum_{u<=l} P[l][u] ecyc(u,l),
// the mean energy of the cycles, summed in parallel (k_ring_estimator) where
// the recursion took N dependent block reductions (N=256: 260 us).
#pragma once

#include "device_common.hpp"
#include "exchange_wide.hpp"
#include "forces.hpp"

namespace pimdb {

// out[b] = {classical spring energy of link (b-1, b), sum of p^2}.
// One workgroup of NT threads per bead; red: 2 NT/64 doubles of LDS.
template <int D, int NT>
__device__ __forceinline__ void bead_sums(int b, int N, int P, double k, int pbc, double L, const double* __restrict__ x,
                                          const double* __restrict__ p, double* __restrict__ out, double* red) {
    constexpr int NW = NT / WAVE;
    const size_t bs = (size_t)D * N;
    const double* xb = x + bs * b;
    const double* xprev = x + bs * ((b - 1 + P) % P);
    const double* pb = p + bs * b;
    double sp = 0.0, kp = 0.0;
    for (int e = threadIdx.x; e < D * N; e += NT) {
        const double d = disp(xb[e], xprev[e], pbc != 0, L);
        sp += d * d;
        kp += pb[e] * pb[e];
    }
    sp = wave_total(sp);
    kp = wave_total(kp);
    if (threadIdx.x % WAVE == 0) {
        red[threadIdx.x / WAVE] = sp;
        red[NW + threadIdx.x / WAVE] = kp;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double s0 = 0.0, s1 = 0.0;
        for (int w = 0; w < NW; ++w) { s0 += red[w]; s1 += red[NW + w]; }
        out[2 * b] = s0 * (0.5 * k);
        out[2 * b + 1] = s1;
    }
}

template <int D>
static __global__ void __launch_bounds__(256) k_bead_sums(int N, int P, double k, int pbc, double L,
                                                   const double* __restrict__ x, const double* __restrict__ p,
                                                   double* __restrict__ out) {
    __shared__ double red[2 * 256 / WAVE];
    bead_sums<D, 256>(blockIdx.x, N, P, k, pbc, L, x, p, out, red);
}

// Everything of a single system's observables but the estimators in one
// launch: the recursions (whose latency covers the rest), the energy tiles and
// the bead sums.
struct ObserveArgs {
    ForceArgs fa;
    double bt;
    int nx, nf;                    // workgroups of the recursions and of the energy tiles
    const double *x, *p;
    double *V, *Vb, *Shi, *Slo;
    unsigned long long* pub;
    int* status;
    double *sums, *epart;          // [P][2], [P][tiles][3]
};

template <int D, int KIND>
static __global__ void __launch_bounds__(XW_THREADS) k_observe(ObserveArgs o) {
    extern __shared__ __align__(16) double smem[];
    const int wg = blockIdx.x, N = o.fa.N, P = o.fa.P;
    if (wg < o.nx) {
        const int b = xw_ring_place(o.pub, N, wg, smem);
        xw_recursions<D, XW_THREADS>(smem, b, N, o.bt, o.fa.k_spring, o.fa.pbc, o.fa.L, BeadView{o.x, N, 1},
                                     BeadView{o.x + (size_t)(P - 1) * D * N, N, 1}, o.V, o.Vb, nullptr, o.Shi, o.Slo,
                                     nullptr, o.pub, o.status);
    } else if (wg < o.nx + o.nf) {
        const int nt = (N + FORCE_TILE - 1) / FORCE_TILE, id = wg - o.nx;
        bead_energies_tile<D, KIND>(o.fa, id / nt, id % nt, o.x, o.epart, smem);
    } else {
        bead_sums<D, XW_THREADS>(wg - o.nx - o.nf, N, P, o.fa.k_spring, o.fa.pbc, o.fa.L, o.x, o.p, o.sums, smem);
    }
}

// out[l] = sum_{u<=l} P[l][u] ecyc(u,l), out[N+l] = ecyc(l,l), one wave per l;
// out[2N] = ecyc(0, N-1), out[2N+1] = V[N].
template <int D>
static __global__ void __launch_bounds__(256) k_ring_estimator(int N, double bt, double k, int pbc, double L,
                                                        const double* __restrict__ x1, const double* __restrict__ xP,
                                                        const double* __restrict__ Shi, const double* __restrict__ Slo,
                                                        const double* __restrict__ V, const double* __restrict__ Vb,
                                                        double* __restrict__ out) {
    const int l = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    if (l >= N) return;
    const Ring r = make_ring(x1, xP, Shi, Slo, k, pbc != 0, L);
    double xl[D];
#pragma unroll
    for (int a = 0; a < D; ++a) xl[a] = xP[a * N + l];
    const double sh = Shi[l], sl = Slo[l], vl = Vb[l + 1], VN = V[N];
    double s = 0.0;
#pragma unroll 4
    for (int u = lane; u <= l; u += WAVE) {
        double d[D];
#pragma unroll
        for (int a = 0; a < D; ++a) d[a] = ring_image(x1[a * N + u] - xl[a], r);
        const double e = ring_ecyc<D>(r, d, Shi[u], Slo[u], sh, sl);
        s = fma(e, exp_minimax(-bt * (V[u] + e + vl - VN)), s);
        if (u == l) out[N + l] = e;
        if (u == 0 && l == N - 1) {
            out[2 * N] = e;
            out[2 * N + 1] = VN;
        }
    }
    s = wave_total(s);
    if (lane == 0) out[l] = s / (l + 1);
}

}  // namespace pimdb
