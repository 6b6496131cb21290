// forces.hpp -- per-slice physical forces (external trap + pair interaction
// with cutoff and minimum image) and the interior ring-polymer springs.
//
// Reference: Simulation::updateForces / updateSpringForces /
// updatePhysicalForces, src/simulation.cpp:353-455; potentials in
// src/potentials/{harmonic,dipole,aziz}.cpp.
//
// One workgroup handles 64 particles i of one bead (time slice) b: the bead's
// N x D positions are staged in LDS, each of the 16 waves runs a sixteenth of
// the partners j (four waves per SIMD hide the FP64 latency chains), and the
// partial forces are reduced in LDS.  Every ordered pair
// (i,j) evaluates gradV(r_i - r_j); for central potentials this is bitwise
// the negation of gradV(r_j - r_i), so the result equals the reference's
// Newton's-third-law loop up to summation order.  Up to 128 particles; larger
// single systems take slice_groups.hpp.
#pragma once

#include "device_common.hpp"
#include "pairs.hpp"

namespace pimdb {

struct ForceArgs {
    int N, P, bosonic, pbc;
    double L, k_spring;
    ExtPot ext;              // external potential
    double int_k, strength;  // pair harmonic constant, dipole strength
    double cutoff;           // effective cutoff (0: no pair loop; < 0: all pairs)
    double cut2;             // cutoff_threshold(cutoff)
};

constexpr int FORCE_TILE = 64;
constexpr int FORCE_WAVES = 16;

// The external and spring forces of particle i of bead b and its pair forces
// `pair` into f (and fext: external and pair alone); fe receives the external
// force.  Exchange beads get no spring part (added later).
template <int D>
__device__ __forceinline__ void row_forces(const ForceArgs& fa, int b, int i, const double* __restrict__ x,
                                           const double (&pair)[D], double* __restrict__ f, double* __restrict__ fext,
                                           double (&fe)[D]) {
    const int N = fa.N, P = fa.P;
    const size_t bs = (size_t)D * N;
    const bool exchange_bead = fa.bosonic && (b == 0 || b == P - 1), pbc = fa.pbc != 0;
    const double* xprev = x + bs * ((b - 1 + P) % P);
    const double* xnext = x + bs * ((b + 1) % P);
    double xv[D];
#pragma unroll
    for (int a = 0; a < D; ++a) xv[a] = x[bs * b + (size_t)a * N + i];
    ext_force<D>(fa.ext, xv, fe);
#pragma unroll
    for (int a = 0; a < D; ++a) {
        const size_t idx = bs * b + (size_t)a * N + i;
        const double xi = xv[a];
        const double phys = fe[a] + pair[a];
        if (fext) fext[idx] = phys;
        double spring = 0.0;
        if (!exchange_bead) {
            const double dp = disp(xi, xprev[(size_t)a * N + i], pbc, fa.L);
            const double dn = disp(xi, xnext[(size_t)a * N + i], pbc, fa.L);
            spring = fa.k_spring * (dp + dn);
        }
        f[idx] = exchange_bead ? phys : spring + phys;
    }
}

// The forces of particles tile*64 .. +63 of bead b by a workgroup of 1024
// threads.  smem: the staged slice (GX: none) and the reduction.  Exchange
// beads get the physical forces alone.  fpart (may be null): the tile's sums of
// the external forces per axis at fpart[(b nt + tile) D + a], nt tiles per bead.
// GX: the slice is read in place from device memory instead of being staged
// in LDS (slices larger than a workgroup's LDS); the LDS then holds only the
// reduction.
template <int D, int KIND, bool GX = false>
__device__ __forceinline__ void bead_forces_tile(const ForceArgs& fa, int b, int tile, const double* __restrict__ x,
                                                 double* __restrict__ f, double* __restrict__ fext,
                                                 double* __restrict__ fpart, double* smem) {
    double* red = smem + (GX ? 0 : (size_t)D * fa.N);   // [FORCE_WAVES-1][D][FORCE_TILE]
    const int N = fa.N, P = fa.P;
    const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
    const size_t bs = (size_t)D * N;
    const double* xb = x + bs * b;
    const double* sx;                                   // [D][N]
    if constexpr (GX) {
        sx = xb;
    } else {
        for (int e = tid; e < D * N; e += FORCE_TILE * FORCE_WAVES) smem[e] = xb[e];
        __syncthreads();
        sx = smem;
    }

    const int i = tile * FORCE_TILE + lane;
    const bool pbc = fa.pbc != 0;
    double acc[D];
#pragma unroll
    for (int a = 0; a < D; ++a) acc[a] = 0.0;
    if constexpr (KIND != POT_FREE) {
        if (i < N && fa.cutoff != 0.0) {
            double xi[D];
#pragma unroll
            for (int a = 0; a < D; ++a) xi[a] = sx[a * N + i];
            const int chunk = (N + FORCE_WAVES - 1) / FORCE_WAVES;
            const int jlo = wave * chunk, jhi = min(N, jlo + chunk);
            const PairParams pp = make_pair_params(fa.L, fa.pbc, fa.cutoff, fa.cut2, fa.int_k, fa.strength);
            auto run = [&](auto img) {
                constexpr int IMG = decltype(img)::value;
                const ImageGrad<D, KIND, IMG> grad{pp, image_params<KIND, IMG>(pp)};
                for (int j = jlo; j < jhi; ++j) {
                    if (j == i) continue;
                    double xj[D], d[D], g;
#pragma unroll
                    for (int a = 0; a < D; ++a) xj[a] = sx[a * N + j];
                    if (grad(xi, xj, d, g)) {
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
        if (wave > 0) {
#pragma unroll
            for (int a = 0; a < D; ++a) red[((wave - 1) * D + a) * FORCE_TILE + lane] = acc[a];
        }
        __syncthreads();
    }
    if (wave != 0) return;
    double fe[D];
#pragma unroll
    for (int a = 0; a < D; ++a) fe[a] = 0.0;
    if (i < N) {
        if constexpr (KIND != POT_FREE) {
            for (int w = 1; w < FORCE_WAVES; ++w) {
#pragma unroll
                for (int a = 0; a < D; ++a) acc[a] += red[((w - 1) * D + a) * FORCE_TILE + lane];
            }
        }
        row_forces<D>(fa, b, i, x, acc, f, fext, fe);
    }
    if (fpart) {
        const int nt = (N + FORCE_TILE - 1) / FORCE_TILE;
#pragma unroll
        for (int a = 0; a < D; ++a) {
            const double s = wave_total(fe[a]);
            if (lane == 0) fpart[((size_t)b * nt + tile) * D + a] = s;
        }
    }
}

template <int D, int KIND, bool GX = false>
static __global__ void __launch_bounds__(FORCE_TILE * FORCE_WAVES)
k_bead_forces(ForceArgs fa, const double* __restrict__ x, double* __restrict__ f, double* __restrict__ fext) {
    extern __shared__ double smem[];
    bead_forces_tile<D, KIND, GX>(fa, blockIdx.y, blockIdx.x, x, f, fext, nullptr, smem);
}

// Pair energy V and g with gradV = g d (harmonic.cpp:9-23, dipole.cpp:5-45,
// aziz.cpp:18-106) from r^2, sharing the root, the exponentials and the
// reciprocal powers; each elementary function within an ulp or so.  A distance
// of 0, or one whose square overflows, gives what 1/r = inf or 0 does.
template <int KIND>
__device__ __forceinline__ void pair_energy_grad(double r2, double kpair, double strength, double& e, double& g) {
    // (the refinement of an estimate of inf or 0 is NaN)
    double inv = rsqrt_refined(r2), norm = r2 * inv;
    if (!__builtin_amdgcn_class(r2, 0x180)) {   // (positive, normal or not)
        inv = __builtin_amdgcn_rsq(r2);
        norm = r2;
    }
    if constexpr (KIND == POT_HARMONIC) {
        e = 0.5 * kpair * r2;
        g = kpair;
    } else if constexpr (KIND == POT_DIPOLE) {
        const double i2 = inv * inv;
        e = strength * (i2 * inv);
        g = -3.0 * strength * (i2 * i2 * inv);
    } else if constexpr (KIND == POT_AZIZ) {
        const double ix = Aziz::rm * inv, ix2 = ix * ix, ix6 = ix2 * ix2 * ix2;
        const double rep = Aziz::A * exp_minimax((-Aziz::alpha / Aziz::rm) * norm);
        const double pe = fma(fma(Aziz::C10, ix2, Aziz::C8), ix2, Aziz::C6);
        double F = 1.0, att = ix6 * pe;
        double datt = ix6 * ix * fma(fma(10.0 * Aziz::C10, ix2, 8.0 * Aziz::C8), ix2, 6.0 * Aziz::C6);
        if (norm < Aziz::D * Aziz::rm) {
            if (norm > HARD_CORE_EPS * Aziz::rm && norm < 0.01 * Aziz::rm) {   // the repulsion alone
                att = 0.0;
                datt = 0.0;
            } else {
                const double t = fma(Aziz::D, ix, -1.0);
                F = exp_minimax(-t * t);
                datt = F * fma(-2.0 * Aziz::D * ix2 * t, att, datt);
                att *= F;
            }
        }
        e = Aziz::epsilon * (rep - att);
        g = (Aziz::epsilon / Aziz::rm) * (datt - Aziz::alpha * rep) * inv;
    } else {
        e = 0.0;
        g = 0.0;
    }
}

// Pair and external potential energies and virial of particles tile*64 .. +63
// of bead b, by a workgroup of 1024 threads, for the energy observable
// (src/observables/energy.cpp:56-111): part[(b nt + tile)] = {ext_pot, int_pot,
// virial_sum} (un-normalised sums of the reference; pairs (i, j > i), the
// virial with r_i alone).  The waves take the partners j > i in turn.  GX and
// smem as for bead_forces_tile.
template <int D, int KIND, bool GX = false>
__device__ __forceinline__ void bead_energies_tile(const ForceArgs& fa, int b, int tile, const double* __restrict__ x,
                                                   double* __restrict__ part, double* smem) {
    const int N = fa.N;
    const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
    const size_t bs = (size_t)D * N;
    const double* xb = x + bs * b;
    const double* sx;
    if constexpr (GX) {
        sx = xb;
    } else {
        for (int e = tid; e < D * N; e += FORCE_TILE * FORCE_WAVES) smem[e] = xb[e];
        __syncthreads();
        sx = smem;
    }
    const int i = tile * FORCE_TILE + lane;
    const bool pbc = fa.pbc != 0;
    const double invL = pbc ? 1.0 / fa.L : 0.0;
    double ext = 0.0, ipot = 0.0, vir = 0.0;
    if (i < N) {
        double xi[D];
#pragma unroll
        for (int a = 0; a < D; ++a) xi[a] = sx[a * N + i];
        if (wave == 0 && fa.ext.kind != POT_FREE) {
            double fe[D];
            ext = ext_energy<D>(fa.ext, xi);
            ext_force<D>(fa.ext, xi, fe);
#pragma unroll
            for (int a = 0; a < D; ++a) vir -= xi[a] * fe[a];
        }
        if constexpr (KIND != POT_FREE) {
            if (fa.cutoff != 0.0) {
                const bool all = fa.cutoff < 0.0;
                for (int j = tile * FORCE_TILE + 1 + wave; j < N; j += FORCE_WAVES) {
                    double d[D];
#pragma unroll
                    for (int a = 0; a < D; ++a) d[a] = disp_fast(sx[a * N + j], xi[a], pbc, fa.L, invL);
                    const double r2 = norm2<D>(d);
                    if (j > i && (all || r2 < fa.cut2)) {
                        double e, g;
                        pair_energy_grad<KIND>(r2, fa.int_k, fa.strength, e, g);
                        ipot += e;
#pragma unroll
                        for (int a = 0; a < D; ++a) vir = fma(xi[a], g * d[a], vir);
                    }
                }
            }
        }
    }
    ext = wave_total(ext);
    ipot = wave_total(ipot);
    vir = wave_total(vir);
    double* red = smem + (GX ? 0 : (size_t)D * N);
    if (lane == 0) {
        red[wave * 3 + 0] = ext;
        red[wave * 3 + 1] = ipot;
        red[wave * 3 + 2] = vir;
    }
    __syncthreads();
    if (tid == 0) {
        double e = 0, ip = 0, v = 0;
        for (int w = 0; w < FORCE_WAVES; ++w) { e += red[w * 3]; ip += red[w * 3 + 1]; v += red[w * 3 + 2]; }
        const int nt = (N + FORCE_TILE - 1) / FORCE_TILE;
        double* o = part + ((size_t)b * nt + tile) * 3;
        o[0] = e; o[1] = ip; o[2] = v;
    }
}

template <int D, int KIND, bool GX = false>
static __global__ void __launch_bounds__(FORCE_TILE * FORCE_WAVES)
k_bead_energies(ForceArgs fa, const double* __restrict__ x, double* __restrict__ part) {
    extern __shared__ double smem[];
    bead_energies_tile<D, KIND, GX>(fa, blockIdx.y, blockIdx.x, x, part, smem);
}

}  // namespace pimdb
