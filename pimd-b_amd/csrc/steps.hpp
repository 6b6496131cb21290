// steps.hpp -- one MD step of a single system as two kernels: everything that
// needs the positions (k_step_forces) and everything that moves them
// (k_step_integrate).
//
// Reference: Simulation::run (src/simulation.cpp:246-259): O, zeroMomentum,
// B, A, forces, B, O, zeroMomentum per step; updateForces (:353-455).
//
// Why.  A step as a graph of seven kernels on two streams spent more time at
// its kernel boundaries than in its kernels: N=4, P=32 took 44 us of which 26
// were kernels, and N=256, P=64 85 us of which 65 were kernels (the fork and
// join alone cost about 8 us, an ordinary boundary 1 us plus the 2 - 3 us that
// any kernel takes to start).  Two facts let the chain close:
//
// * The closing half of step s (B, O, zeroMomentum) and the opening half of
//   step s+1 (O, zeroMomentum, B, A) act on the same force, and the Langevin
//   O-steps are affine: with h = dt/2 and G the (mode-coupled) noise c2 xi,
//       p' = c1 [c1 (p + h f) + G2 - cm2] + G1 - cm1 + h f
//          = c1^2 (p + h f) + H - shift + h f,       H = c1 G2 + G1,
//       shift = c1 cm2 + cm1 = mean(c1^2 (p + h f) + H)
//   (the momenta after a zeroMomentum sum to zero, so cm1 = mean(G1)).  H
//   depends on no force, and neither does its sum: both are made beside the
//   forces.  sum(f) is the sum of the external forces (pair, spring and
//   exchange forces sum to zero up to rounding).
// * The exchange forces on beads 1 and P need the finished recursions, but
//   only the integration needs them: it evaluates them itself.
//
// k_step_forces: workgroups of 1024 threads take one of three parts, in this
// order: the recursions (exchange_wide.hpp), tiles of the bead forces
// (forces.hpp), and tiles of H with the partial sums for the shift.  The
// recursions' latency covers the rest up to about N = 500.
// k_step_integrate: the exterior forces and update of beads 1 and P, one wave
// per particle and bead, and the update of the others, elementwise.
#pragma once

#include "device_common.hpp"
#include "exchange_wide.hpp"
#include "forces.hpp"

namespace pimdb {

constexpr int STEP_TILE = 64;         // columns (one axis) per noise workgroup
constexpr int STEP_NM_MAXP = 64;      // beads of the matrix-core noise transform

struct StepArgs {
    ForceArgs fa;
    double bt;
    int nx, nf, nn;                   // workgroups of the three parts
    double *x, *p, *f, *fext;
    // recursions
    double *V, *Vb, *Shi, *Slo, *xc;  // xc: copies [4][D][N] of beads 1, P, 2, P-1
    unsigned long long* pub;
    int* status;
    // noise and the shift
    int thermostat, nm, fixcom;
    double c1, c2, half_dt, dt_m;     // dt_m = dt / mass
    const double* CTt;                // nm -> cart transposed: CTt[k P + b]
    double* H;                        // [P][D][N]
    double* fpart;                    // [P nt][D] external force sums of the force tiles (null: none)
    double* hpart;                    // [noise tiles][D] sums of c1^2 p + H
    unsigned long long* ctr;          // steps done
    uint32_t seed;
};

__host__ __device__ inline int step_noise_tiles(int N) { return (N + STEP_TILE - 1) / STEP_TILE; }
__host__ __device__ inline int step_pad16(int P) { return (P + 15) & ~15; }
__host__ __device__ inline size_t step_noise_lds_doubles(int P, bool nm) {
    const size_t Pp = (size_t)step_pad16(P);
    return XW_WAVES + (nm ? Pp * Pp + Pp * STEP_TILE : 0);
}

typedef double step_v4d __attribute__((ext_vector_type(4)));

// H of particles i0 .. i0+63 of axis a for all beads, and the tile's sum of
// c1^2 p + H.  The noise has the keys of the single O-steps: modes (beads)
// 2m and 2m+1 of column (a, i) from one Box-Muller pair, the closing O-step
// of the step just made (O-step 1) and the opening one of the next (O-step
// 0), both at the current step count.  Normal-mode coupling: H = C^T (c1 xi2 +
// xi1) c2 on the matrix cores (v_mfma_f64_16x16x4f64; lane l, item v:
// A[l%16][l/16], B[l/16][l%16], D[l/16 + 4v][l%16]).
template <int D>
__device__ __forceinline__ void step_noise(const StepArgs& s, int idx, double* smem) {
    const int N = s.fa.N, P = s.fa.P, ncols = D * N;
    const int tiles = step_noise_tiles(N);
    const int a = idx / tiles, i0 = (idx % tiles) * STEP_TILE;
    const int nc = min(STEP_TILE, N - i0);
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const uint32_t step = (uint32_t)*s.ctr;
    const double c1sq = s.c1 * s.c1;
    const int half = (P + 1) / 2;
    double* red = smem;
    double sum = 0.0;
    auto draw = [&](int m, int col, double& g0, double& g1) {
        double h0, h1;
        const uint32_t key = (uint32_t)((size_t)m * ncols + col);
        gauss2<true>(key, step, 1u, 0u, s.seed, h0, h1);
        gauss2<true>(key, step, 0u, 0u, s.seed, g0, g1);
        g0 = s.c2 * fma(s.c1, h0, g0);
        g1 = s.c2 * fma(s.c1, h1, g1);
    };
    if (s.thermostat == 0) {
        for (int e = tid; e < P * STEP_TILE; e += XW_THREADS) {
            const int b = e / STEP_TILE, c = e % STEP_TILE;
            if (c < nc) sum += s.p[(size_t)b * ncols + a * N + i0 + c];
        }
    } else if (!s.nm) {
        for (int e = tid; e < half * STEP_TILE; e += XW_THREADS) {
            const int m = e / STEP_TILE, c = e % STEP_TILE;
            if (c >= nc) continue;
            const int col = a * N + i0 + c;
            double g[2];
            draw(m, col, g[0], g[1]);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (2 * m + h < P) {
                    const size_t q = (size_t)(2 * m + h) * ncols + col;
                    s.H[q] = g[h];
                    sum += fma(c1sq, s.p[q], g[h]);
                }
            }
        }
    } else {
        const int Pp = step_pad16(P), MB = Pp / 16, KK = Pp / 4;
        double* CTl = smem + XW_WAVES;          // [k][b], zero padded
        double* pn = CTl + (size_t)Pp * Pp;     // [column / 16][k][16]
        for (int e = tid; e < Pp * Pp; e += XW_THREADS) {
            const int k = e / Pp, b = e % Pp;
            CTl[e] = (k < P && b < P) ? s.CTt[(size_t)k * P + b] : 0.0;
        }
        for (int e = tid; e < (Pp / 2) * STEP_TILE; e += XW_THREADS) {
            const int m = e / STEP_TILE, c = e % STEP_TILE;
            double g0 = 0.0, g1 = 0.0;
            if (m < half && c < nc) draw(m, a * N + i0 + c, g0, g1);
            double* out = pn + (size_t)(c / 16) * Pp * 16 + c % 16;
            out[(2 * m) * 16] = 2 * m < P ? g0 : 0.0;
            out[(2 * m + 1) * 16] = 2 * m + 1 < P ? g1 : 0.0;
        }
        __syncthreads();
        const int q4 = lane / 16, c16 = lane % 16;
        for (int task = wave; task < MB * (STEP_TILE / 16); task += XW_WAVES) {
            const int bb = task % MB, g = task / MB, c = g * 16 + c16;
            step_v4d acc = {0.0, 0.0, 0.0, 0.0};
            const double* B = pn + (size_t)g * Pp * 16;
            for (int kk = 0; kk < KK; ++kk) {
                const int k = 4 * kk + q4;
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(CTl[(size_t)k * Pp + bb * 16 + c16], B[k * 16 + c16], acc, 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int b = bb * 16 + q4 + 4 * v;
                if (b < P && c < nc) {
                    const size_t q = (size_t)b * ncols + a * N + i0 + c;
                    s.H[q] = acc[v];
                    sum += fma(c1sq, s.p[q], acc[v]);
                }
            }
        }
    }
    if (s.fixcom) {
        sum = wave_total(sum);
        if (lane == 0) red[wave] = sum;
        __syncthreads();
        if (tid == 0) {
            double t = 0.0;
            for (int w = 0; w < XW_WAVES; ++w) t += red[w];
            s.hpart[(size_t)(idx % tiles) * D + a] = t;
        }
    }
}

// x, p, f: bead-major SoA [b][a][i].  Dynamic LDS: the largest part's need.
template <int D, int KIND>
static __global__ void __launch_bounds__(XW_THREADS) k_step_forces(StepArgs s) {
    extern __shared__ double smem[];
    const int wg = blockIdx.x;
    if (wg < s.nx) {
        const int N = s.fa.N, P = s.fa.P;
        const size_t bs = (size_t)D * N;
        if (wg == 0) {   // beads 2 and P-1 for the exterior forces (the recursions copy beads 1 and P)
            const double* x2 = s.x + bs * (1 % P);
            const double* xPm1 = s.x + bs * ((P - 2 + P) % P);
            for (int e = threadIdx.x; e < D * N; e += XW_THREADS) {
                s.xc[2 * bs + e] = x2[e];
                s.xc[3 * bs + e] = xPm1[e];
            }
        }
        xw_recursions<D>(smem, wg, N, s.bt, s.fa.k_spring, s.fa.pbc, s.fa.L, s.x, s.x + bs * (P - 1), s.V, s.Vb, s.Shi,
                         s.Slo, s.xc, s.pub, s.status);
    } else if (wg < s.nx + s.nf) {
        const int nt = (s.fa.N + FORCE_TILE - 1) / FORCE_TILE, id = wg - s.nx;
        bead_forces_tile<D, KIND>(s.fa, id / nt, id % nt, s.x, s.f, s.fext, s.fpart, smem);
    } else {
        step_noise<D>(s, wg - s.nx - s.nf, smem);
    }
}

// Workgroups of k_step_integrate: 4 (particle, bead) tasks of the exchange
// beads each, then 256 elements of the other beads each.
__host__ __device__ inline int step_exterior_groups(const ForceArgs& fa) { return fa.bosonic ? (2 * fa.N + 3) / 4 : 0; }
__host__ __device__ inline size_t step_inner_elements(const ForceArgs& fa, int D) {
    return (size_t)(fa.bosonic ? fa.P - 2 : fa.P) * D * fa.N;
}

// The closing half of a step and the opening half of the next (file header).
// Leaves f complete.  The positions that other particles' exterior forces
// need are read from the copies xc, so x is free to be written.
template <int D>
static __global__ void __launch_bounds__(256) k_step_integrate(StepArgs s) {
    const int N = s.fa.N, P = s.fa.P;
    const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
    __shared__ double shift[4];
    const int ng = step_exterior_groups(s.fa);
    const bool exterior = (int)blockIdx.x < ng;
    const size_t bs = (size_t)D * N;
    const double c1sq = s.c1 * s.c1, h = s.half_dt;
    // the element's (or, exterior, lane's) data first: the loads overlap the
    // reduction below
    const int task = blockIdx.x * 4 + wave;
    size_t e = 0;
    bool mine = false;
    int ax = 0;
    if (exterior) {
        const int which = task / N, l = task % N;
        if (task < 2 * N && lane < D) {
            mine = true;
            ax = lane;
            e = ((size_t)(which == 0 ? 0 : P - 1) * D + lane) * N + l;
        }
    } else {
        const size_t o = (size_t)(blockIdx.x - ng) * 256 + tid;
        mine = o < step_inner_elements(s.fa, D);
        e = o + (s.fa.bosonic ? bs : 0);
        ax = (int)((e / N) % D);
    }
    double pv = 0.0, fv = 0.0, xv = 0.0, hv = 0.0;
    if (mine) {
        pv = s.p[e];
        fv = s.f[e];
        xv = s.x[e];
        if (s.thermostat) hv = s.H[e];
    }
    if (s.fixcom) {
        if (wave < D) {
            const int rows = step_noise_tiles(N);
            double t = 0.0;
            for (int r = lane; r < rows; r += WAVE) t += s.hpart[(size_t)r * D + wave];
            if (s.fpart) {
                const int nt = P * ((N + FORCE_TILE - 1) / FORCE_TILE);
                double u = 0.0;
                for (int r = lane; r < nt; r += WAVE) u += s.fpart[(size_t)r * D + wave];
                t = fma(c1sq * h, u, t);
            }
            t = wave_total(t);
            if (lane == 0) shift[wave] = t / (double)(N * P);
        }
        __syncthreads();
    }
    if (blockIdx.x == 0 && tid == 0) *s.ctr += 1;
    if (exterior) {
        if (task >= 2 * N) return;
        const int which = task / N, l = task % N;
        const Ring r = make_ring(s.xc, s.xc + bs, s.Shi, s.Slo, s.fa.k_spring, s.fa.pbc != 0, s.fa.L);
        double F[D];
        exterior_force<D>(which, l, N, lane, s.bt, s.fa.k_spring, r, s.V, s.Vb, s.xc + 2 * bs, s.xc + 3 * bs, false, F);
#pragma unroll
        for (int a = 0; a < D; ++a)
            if (lane == a) fv = F[a] + fv;
        if (mine) s.f[e] = fv;
    }
    if (!mine) return;
    const double hf = h * fv;
    double v = fma(c1sq, pv + hf, hv) + hf;
    if (s.fixcom) v -= shift[ax];
    s.p[e] = v;
    s.x[e] = fma(s.dt_m, v, xv);
}

}  // namespace pimdb
