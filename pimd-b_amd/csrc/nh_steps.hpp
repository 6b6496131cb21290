// nh_steps.hpp -- the Nose-Hoover half steps of a single system around its
// force evaluation as one kernel (Cartesian coupling and propagator).
//
// Reference: Simulation::run (src/simulation.cpp:246-259), thermostats as in
// nose_hoover.hpp.
//
// Why.  A step was k_nh_ostep twice, k_kick_drift, the forces and
// k_exchange_forces: 27 us for N=8, P=16, of which the chains' arithmetic is
// about 2.  The closing half of a step (B, O, zeroMomentum) and the opening half
// of the next (O, zeroMomentum, B, A) touch no other bead unless zeroMomentum
// couples them.  So a workgroup does both, for one bead or, with zeroMomentum,
// for the whole system where that is small enough for one workgroup (a sum over
// all beads between the two O-steps); it also evaluates the exchange forces of
// its beads 1 and P while those are few per wave.  What bounds it: the latency of
// two chain updates (six exponentials in turn each).  A step, us, chains per
// particle: N=8, P=16 without zeroMomentum 23.2 -> 14.5 and with it 25.4 -> 18.0;
// N=128, P=64 without 29.4 -> 22.5.  Larger systems with zeroMomentum keep their
// kernels (N=16, P=64: 26.0, 32.3 in one workgroup), the closing half with the
// exchange forces up to 32 particles (N=16 22.2, N=32 26.3 -> 25.0, N=64 26.7
// -> 30.5).
#pragma once

#include "nose_hoover.hpp"
#include "steps.hpp"

namespace pimdb {

constexpr int NH_THREADS = 1024;
constexpr int NH_WAVES = NH_THREADS / WAVE;
constexpr int NH_EXT = 64;   // particles up to which the exchange forces are evaluated here (four a wave)

// LDS doubles of a workgroup of nb beads.
__host__ __device__ inline size_t nh_step_lds_doubles(int N, int D, int nb, bool exterior) {
    return (size_t)D * N * (nb + (exterior ? 2 : 0));
}

// One of P / nb workgroups, nb beads each.  zeroMomentum: all beads in one
// workgroup, or (a closing half alone) h.com_out, the partial sums for it.  f
// complete but for the exchange forces if `exterior`.  mode: OPEN, FULL, CLOSE.
template <int D>
static __global__ void __launch_bounds__(NH_THREADS) k_nh_steps(StepArgs s, NhArgs h, int nb, int exterior, int mode) {
    extern __shared__ __align__(16) double smem[];
    __shared__ double red[D][NH_WAVES];
    const int N = s.fa.N, P = s.fa.P, bs = D * N, ne = nb * bs, b0 = blockIdx.x * nb;
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const size_t base = (size_t)b0 * bs;
    const bool close = mode != STEP_OPEN, open = mode != STEP_CLOSE;
    double* pl = smem;         // [bead][axis][particle]
    double* fx = smem + ne;    // [2][axis][particle]
    if (blockIdx.x == 0 && tid == 0 && open) *s.ctr += 1;
    if (close && exterior) {
        const bool first = b0 == 0, last = b0 + nb == P;
        const int ntask = (first ? N : 0) + (last ? N : 0);
        const size_t cs = bs;
        const Ring r = make_ring(s.xc, s.xc + cs, s.Shi, s.Slo, s.fa.k_spring, s.fa.pbc != 0, s.fa.L);
        for (int t = wave; t < ntask; t += NH_WAVES) {
            const int which = first ? t / N : 1, l = t % N;
            double F[D];
            exterior_force<D>(which, l, N, lane, s.bt, s.fa.k_spring, r, s.V, s.Vb, s.xc + 2 * cs, s.xc + 3 * cs, false, F);
#pragma unroll
            for (int a = 0; a < D; ++a)
                if (lane == a) fx[which * bs + a * N + l] = F[a];
        }
        __syncthreads();
    }
    for (int e = tid; e < ne; e += NH_THREADS) {
        double v = s.p[base + e];
        if (close) {
            double f = s.f[base + e];
            const int b = b0 + e / bs;
            if (exterior && (b == 0 || b == P - 1)) {
                f = fx[(b == 0 ? 0 : bs) + e % bs] + f;
                s.f[base + e] = f;
            }
            v += h.half_dt * f;
        }
        pl[e] = v;
    }
    __syncthreads();
    auto ostep = [&]() {
        const int nc = h.nc;
        auto chain = [&](int b, int g, double ce) {
            const size_t o = ((size_t)(b0 + b) * h.groups + g) * nc;
            return nh_chain_step(h, h.eta + o, h.eta_dot + o, h.eta_dot_dot + o, ce);
        };
        if (h.kind == PIMDB_THERMO_NOSE_HOOVER) {   // a wave per bead
            for (int b = wave; b < nb; b += NH_WAVES) {
                double* pb = pl + (size_t)b * bs;
                double t = 0.0;
                for (int e = lane; e < bs; e += WAVE) t = fma(pb[e], pb[e], t);
                t = wave_total(t);
                double sc = 0.0;
                if (lane == 0) sc = chain(b, 0, t / h.mass);
                sc = wave_bcast_uniform(sc, 0);
                for (int e = lane; e < bs; e += WAVE) pb[e] *= sc;
            }
        } else if (h.kind == PIMDB_THERMO_NOSE_HOOVER_NP) {
            for (int t = tid; t < nb * N; t += NH_THREADS) {
                const int b = t / N, i = t % N;
                double* pb = pl + (size_t)b * bs + i;
                double ce = 0.0;
#pragma unroll
                for (int a = 0; a < D; ++a) ce += pb[a * N] * pb[a * N];
                const double sc = chain(b, i, ce / h.mass);
#pragma unroll
                for (int a = 0; a < D; ++a) pb[a * N] *= sc;
            }
        } else {
            for (int e = tid; e < ne; e += NH_THREADS) {
                const int b = e / bs, a = e % bs / N, i = e % N;
                pl[e] *= chain(b, i * D + a, pl[e] * pl[e] / h.mass);
            }
        }
        __syncthreads();
        if (!s.fixcom) return;
        double c[D];
#pragma unroll
        for (int a = 0; a < D; ++a) c[a] = 0.0;
        for (int e = tid; e < ne; e += NH_THREADS) {
            const int ax = e % bs / N;
#pragma unroll
            for (int a = 0; a < D; ++a) c[a] += a == ax ? pl[e] : 0.0;
        }
#pragma unroll
        for (int a = 0; a < D; ++a) {
            c[a] = wave_total(c[a]);
            if (lane == 0) red[a][wave] = c[a];
        }
        __syncthreads();
#pragma unroll
        for (int a = 0; a < D; ++a) {
            c[a] = 0.0;
            for (int w = 0; w < NH_WAVES; ++w) c[a] += red[a][w];
            if (h.com_out && tid == 0) h.com_out[(size_t)blockIdx.x * D + a] = c[a];
            c[a] /= (double)(N * P);
        }
        if (h.com_out) return;
        for (int e = tid; e < ne; e += NH_THREADS) {
            const int ax = e % bs / N;
#pragma unroll
            for (int a = 0; a < D; ++a)
                if (a == ax) pl[e] -= c[a];
        }
        __syncthreads();
    };
    if (close) ostep();
    if (open) ostep();
    for (int e = tid; e < ne; e += NH_THREADS) {
        double v = pl[e];
        if (open) {
            v += h.half_dt * s.f[base + e];
            s.x[base + e] = fma(s.dt_m, v, s.x[base + e]);
        }
        s.p[base + e] = v;
    }
}

}  // namespace pimdb
