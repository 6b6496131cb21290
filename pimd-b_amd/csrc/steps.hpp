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
//   exchange forces sum to zero up to rounding).  The first opening and the
//   last closing half of a run are the same update with other coefficients
//   (StepMode), so a run needs no other kernels.
// * The exchange forces on beads 1 and P need the finished recursions, but
//   only the integration needs them: it evaluates them itself.
//
// Forces kernel: workgroups take one of three parts, in this order: the
// recursions (exchange_wide.hpp), tiles of H with the partial sums for the
// shift, and the bead forces (forces.hpp, slice_groups.hpp or, batched,
// pimdb_split.hip, where slices and tiles come longest first).  The
// recursions' latency covers the rest of a single system up to about N = 500.
// Integration kernel: the exterior forces and update of beads 1 and P, one
// wave per particle and bead, and the update of the others, elementwise.
#pragma once

#include "device_common.hpp"
#include "exchange_wide.hpp"
#include "forces.hpp"
#include "slice_groups.hpp"

namespace pimdb {

constexpr int STEP_TILE = 64;         // columns (one axis) per noise workgroup
constexpr int STEP_NM_MAXP = 64;      // beads of the matrix-core noise transform

// What an integration does: p' = a1 a2 (p + beta f) + H - mean(...) + gamma f,
// then (but for CLOSE) x += dt/m p'.
enum StepMode : int {
    STEP_OPEN = 0,    // O, zeroMomentum, B, A with complete forces
    STEP_FULL = 1,    // the closing half of a step and the opening half of the next
    STEP_CLOSE = 2,   // B, O, zeroMomentum
    STEP_FORCES = 3   // nothing but the exterior forces into f
};

struct StepArgs {
    ForceArgs fa;
    double bt;
    double *x, *p, *f, *fext;
    // recursions
    double *V, *Vb, *Shi, *Slo, *xc;  // xc: copies [4][D][N] of beads 1, P, 2, P-1
    unsigned long long* pub;
    int* status;
    // noise and the shift
    int thermostat, nm, fixcom;
    double c1, c2, half_dt, dt_m;     // c1 = 1 without a thermostat; dt_m = dt / mass
    const double *Ct, *CTt, *rot;     // cart -> nm and nm -> cart transposed (CTt[k P + b]); free-ring rotation
    double* H;                        // [P][D][N]
    double* fpart;                    // [frows][D] partial sums of the external forces (null: none)
    double* hpart;                    // [noise tiles][D] sums of a1 a2 p + H
    int frows;
    PairGroups pg;                    // G > 0: the pair forces by groups, f to be completed from pg.cpart
    unsigned long long* ctr;          // steps done
    uint32_t seed;
};

// a1, a2: the two O-steps' factors (1 for one that is not there), applied one
// after the other: c1 c1 rounded once would be the same error in every step, and
// add up over the momenta's memory of 2 / (gamma dt) steps.
struct StepCoef {
    double a1, a2, beta, gamma, k2, k1;   // H = c2 (k2 xi2 + k1 xi1)
};
__device__ __forceinline__ StepCoef step_coef(const StepArgs& s, int mode) {
    if (mode == STEP_OPEN) return StepCoef{s.c1, 1.0, 0.0, s.half_dt, 0.0, 1.0};
    if (mode == STEP_FULL) return StepCoef{s.c1, s.c1, s.half_dt, s.half_dt, s.c1, 1.0};
    return StepCoef{s.c1, 1.0, s.half_dt, 0.0, 1.0, 0.0};
}
__device__ __forceinline__ double step_kept(const StepCoef& co, double p, double h) { return fma(co.a1, co.a2 * p, h); }

__host__ __device__ inline int step_noise_tiles(int N) { return (N + STEP_TILE - 1) / STEP_TILE; }
// Noise workgroups of a replica: none where nothing is drawn or summed.
__host__ __device__ inline int step_noise_groups(const StepArgs& s, int D) {
    return s.thermostat || s.fixcom ? D * step_noise_tiles(s.fa.N) : 0;
}
__host__ __device__ inline int step_pad16(int P) { return (P + 15) & ~15; }
template <int NT>
__host__ __device__ inline size_t step_noise_lds_doubles(int P, bool nm) {
    const size_t Pp = (size_t)step_pad16(P);
    return XW_THREADS / WAVE + (nm ? (NT == XW_THREADS ? Pp * Pp : 0) + Pp * STEP_TILE : 0);
}

typedef double step_v4d __attribute__((ext_vector_type(4)));

// H of particles i0 .. i0+63 of axis a for all beads, and the tile's sum of
// a1 a2 p + H, by a workgroup of NT threads.  The noise has the keys of the
// single O-steps: modes (beads) 2m and 2m+1 of column (a, i) from one
// Box-Muller pair, at the current step count with O-step 1 for a closing half
// (xi2) and 0 for an opening one (xi1).  Normal-mode coupling: C^T on the
// matrix cores (v_mfma_f64_16x16x4f64; lane l, item v: A[l%16][l/16],
// B[l/16][l%16], D[l/16 + 4v][l%16]).
template <int D, int NT>
__device__ __forceinline__ void step_noise(const StepArgs& s, int mode, int idx, double* smem) {
    constexpr int NW = NT / WAVE;
    // a single system's deviates are k_momenta's, with the correctly rounded
    // quotient and root (N=64, P=64: 14.6 -> 14.9 us a step, N=256 the same), a
    // batch's the persistent kernel's
    constexpr bool FAST = NT != XW_THREADS;
    const StepCoef co = step_coef(s, mode);
    const int N = s.fa.N, P = s.fa.P, ncols = D * N;
    const int tiles = step_noise_tiles(N);
    const int a = idx / tiles, i0 = (idx % tiles) * STEP_TILE;
    const int nc = min(STEP_TILE, N - i0);
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const uint32_t step = (uint32_t)*s.ctr;
    const int half = (P + 1) / 2;
    double* red = smem;
    double sum = 0.0;
    auto draw = [&](int m, int col, double& g0, double& g1) {
        const uint32_t key = (uint32_t)((size_t)m * ncols + col);
        g0 = 0.0;
        g1 = 0.0;
        if (mode != STEP_OPEN) {
            gauss2<FAST>(key, step, 1u, 0u, s.seed, g0, g1);
            g0 *= co.k2;
            g1 *= co.k2;
        }
        if (mode != STEP_CLOSE) {
            double h0, h1;
            gauss2<FAST>(key, step, 0u, 0u, s.seed, h0, h1);
            g0 += h0;
            g1 += h1;
        }
        g0 *= s.c2;
        g1 *= s.c2;
    };
    if (s.thermostat == 0) {
        for (int e = tid; e < P * STEP_TILE; e += NT) {
            const int b = e / STEP_TILE, c = e % STEP_TILE;
            if (c < nc) sum += s.p[(size_t)b * ncols + a * N + i0 + c];
        }
    } else if (!s.nm) {
        for (int e = tid; e < half * STEP_TILE; e += NT) {
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
                    sum += step_kept(co, s.p[q], g[h]);
                }
            }
        }
    } else {
        // C^T is staged in LDS where the workgroup has the compute unit to
        // itself (N=128, P=64: 18.5 us a step, 21.5 without); beside other
        // workgroups, which the 32 KB would keep out, a wave holds its rows of it.
        constexpr int KMAX = STEP_NM_MAXP / 4;
        constexpr bool STAGED = NT == XW_THREADS;
        const int Pp = step_pad16(P), MB = Pp / 16, KK = Pp / 4;
        double* CTl = smem + XW_THREADS / WAVE;                     // [k][b], zero padded
        double* pn = CTl + (STAGED ? (size_t)Pp * Pp : 0);          // [column / 16][k][16]
        if constexpr (STAGED) {
            for (int e = tid; e < Pp * Pp; e += NT) {
                const int k = e / Pp, b = e % Pp;
                CTl[e] = (k < P && b < P) ? s.CTt[(size_t)k * P + b] : 0.0;
            }
        }
        const int q4 = lane / 16, c16 = lane % 16;
        const int ntask = MB * (STEP_TILE / 16);
        double A[KMAX];
        int held = -1;
        auto rows = [&](int bb) {
            held = bb;
            const int b = bb * 16 + c16;
#pragma unroll
            for (int kk = 0; kk < KMAX; ++kk) {
                const int k = 4 * kk + q4;
                const double v = s.CTt[(size_t)min(k, P - 1) * P + min(b, P - 1)];
                A[kk] = k < P && b < P ? v : 0.0;
            }
        };
        if (!STAGED && wave < ntask) rows(wave % MB);
        for (int e = tid; e < (Pp / 2) * STEP_TILE; e += NT) {
            const int m = e / STEP_TILE, c = e % STEP_TILE;
            double g0 = 0.0, g1 = 0.0;
            if (m < half && c < nc) draw(m, a * N + i0 + c, g0, g1);
            double* out = pn + (size_t)(c / 16) * Pp * 16 + c % 16;
            out[(2 * m) * 16] = 2 * m < P ? g0 : 0.0;
            out[(2 * m + 1) * 16] = 2 * m + 1 < P ? g1 : 0.0;
        }
        __syncthreads();
        for (int task = wave; task < ntask; task += NW) {
            const int bb = task % MB, g = task / MB, c = g * 16 + c16;
            if (!STAGED && bb != held) rows(bb);
            step_v4d acc = {0.0, 0.0, 0.0, 0.0};
            const double* B = pn + (size_t)g * Pp * 16;
            if constexpr (STAGED) {
                for (int kk = 0; kk < KK; ++kk) {
                    const int k = 4 * kk + q4;
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(CTl[(size_t)k * Pp + bb * 16 + c16], B[k * 16 + c16], acc, 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int kk = 0; kk < KMAX; ++kk)
                    if (kk < KK) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(A[kk], B[(4 * kk + q4) * 16 + c16], acc, 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int b = bb * 16 + q4 + 4 * v;
                if (b < P && c < nc) {
                    const size_t q = (size_t)b * ncols + a * N + i0 + c;
                    s.H[q] = acc[v];
                    sum += step_kept(co, s.p[q], acc[v]);
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
            for (int w = 0; w < NW; ++w) t += red[w];
            s.hpart[(size_t)(idx % tiles) * D + a] = t;
        }
    }
}

// The workgroup in place wg of xw_grid(N): the recursions (exchange_wide.hpp), with copies
// of the beads that the exterior forces read after the positions moved on.
template <int D, int NT>
__device__ __forceinline__ void step_recursions(const StepArgs& s, int wg, double* smem) {
    const int N = s.fa.N, P = s.fa.P;
    const size_t bs = (size_t)D * N;
    if (wg == 0) {   // beads 2 and P-1 (the recursions copy beads 1 and P)
        const double* x2 = s.x + bs * (1 % P);
        const double* xPm1 = s.x + bs * ((P - 2 + P) % P);
        for (int e = threadIdx.x; e < D * N; e += NT) {
            s.xc[2 * bs + e] = x2[e];
            s.xc[3 * bs + e] = xPm1[e];
        }
    }
    xw_recursions<D, NT>(smem, wg, N, s.bt, s.fa.k_spring, s.fa.pbc, s.fa.L, BeadView{s.x, N, 1},
                         BeadView{s.x + bs * (P - 1), N, 1}, s.V, s.Vb, nullptr, s.Shi, s.Slo, s.xc, s.pub, s.status);
}

// Workgroups of an integration: 4 particles of an exchange bead each (their
// forces are complete before an opening half), then 256 elements of the other
// beads each.
__host__ __device__ inline int step_exterior_groups(const ForceArgs& fa, int mode) {
    return fa.bosonic && mode != STEP_OPEN ? (2 * fa.N + 3) / 4 : 0;   // (also STEP_FORCES)
}
__host__ __device__ inline size_t step_inner_elements(const ForceArgs& fa, int D, int mode) {
    return (size_t)(fa.bosonic && mode != STEP_OPEN ? fa.P - 2 : fa.P) * D * fa.N;
}
__host__ __device__ inline int step_integrate_groups(const ForceArgs& fa, int D, int mode) {
    return step_exterior_groups(fa, mode) + (int)((step_inner_elements(fa, D, mode) + 255) / 256);
}

// The momentum per particle and axis that an integration takes out, into
// shift[0 .. D-1] (wave a for axis a; a barrier is the caller's).
template <int D>
__device__ __forceinline__ void step_shift(const StepArgs& s, int mode, int wave, int lane, double* shift) {
    if (wave >= D) return;
    const StepCoef co = step_coef(s, mode);
    const int rows = step_noise_tiles(s.fa.N);
    double t = 0.0;
    for (int r = lane; r < rows; r += WAVE) t += s.hpart[(size_t)r * D + wave];
    if (s.fpart && mode != STEP_OPEN) {
        double u = 0.0;
        for (int r = lane; r < s.frows; r += WAVE) u += s.fpart[(size_t)r * D + wave];
        t = step_kept(co, co.beta * u, t);
    }
    t = wave_total(t);
    if (lane == 0) shift[wave] = t / (double)(s.fa.N * s.fa.P);
}

// Workgroup blk of an integration, 256 threads (file header).  Leaves f
// complete.  The positions that other particles' exterior forces need are
// read from the copies xc, so x is free to be written.
template <int D>
__device__ __forceinline__ void step_integrate(const StepArgs& s, int mode, int blk) {
    const StepCoef co = step_coef(s, mode);
    const int N = s.fa.N, P = s.fa.P;
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    __shared__ double shift[4];
    const int ng = step_exterior_groups(s.fa, mode);
    const bool exterior = blk < ng;
    const size_t bs = (size_t)D * N;
    // the element's (or, exterior, lane's) data first: the loads overlap the
    // reduction below
    const int task = blk * 4 + wave;
    size_t e = 0;
    bool mine = false;
    int ax = 0;
    if (exterior) {
        if (task < 2 * N && lane < D) {   // a wave per particle, its first lanes an axis each
            mine = true;
            ax = lane;
            e = ((size_t)(task < N ? 0 : P - 1) * D + ax) * N + task % N;
        }
    } else {
        const size_t o = (size_t)(blk - ng) * 256 + tid;
        mine = o < step_inner_elements(s.fa, D, mode);
        e = o + (ng ? bs : 0);
        ax = (int)((e / N) % D);
    }
    double pv = 0.0, fv = 0.0, xv = 0.0, hv = 0.0;
    if (mode == STEP_FORCES && !exterior) return;
    if (mine) {
        fv = s.f[e];
        if (mode != STEP_FORCES) {
            pv = s.p[e];
            if (mode != STEP_CLOSE) xv = s.x[e];
            if (s.thermostat) hv = s.H[e];
        }
        if (mode != STEP_OPEN && s.pg.G) {
            const size_t n = (size_t)P * bs;
            double c = 0.0;
            for (int k = 0, m = s.pg.slots((int)(e / bs)); k < m; ++k) c += s.pg.cpart[k * n + e];
            fv += c;
        }
    }
    if (s.fixcom && mode != STEP_FORCES) {
        step_shift<D>(s, mode, wave, lane, shift);
        __syncthreads();
    }
    if (exterior) {
        if (task >= 2 * N) return;
        const Ring r = make_ring(s.xc, s.xc + bs, s.Shi, s.Slo, s.fa.k_spring, s.fa.pbc != 0, s.fa.L);
        double F[D];
        exterior_force<D>(task / N, task % N, N, lane, s.bt, s.fa.k_spring, r, s.V, s.Vb, s.xc + 2 * bs, s.xc + 3 * bs,
                          false, F);
#pragma unroll
        for (int a = 0; a < D; ++a)
            if (lane == a) fv = F[a] + fv;
        if (mine) s.f[e] = fv;
    } else if (mine && s.pg.G && mode != STEP_OPEN) {
        s.f[e] = fv;
    }
    if (!mine || mode == STEP_FORCES) return;
    double v = step_kept(co, fma(co.beta, fv, pv), hv);
    if (s.fixcom) v -= shift[ax];
    if (mode == STEP_CLOSE) {
        s.p[e] = v;
    } else {
        v = fma(co.gamma, fv, v);
        s.p[e] = v;
        s.x[e] = fma(s.dt_m, v, xv);
    }
}

// ---- one system ----
// nx, nn: workgroups of the recursions and of the noise; the rest are the pair
// groups or force tiles.  x, p, f: bead-major SoA [b][a][i].  Dynamic LDS: the largest part's.
template <int D, int KIND>
static __global__ void __launch_bounds__(XW_THREADS) k_step_forces(StepArgs s, int nx, int nn, int mode) {
    extern __shared__ __align__(16) double smem[];
    const int wg = blockIdx.x;
    if (wg < nx) {
        step_recursions<D, XW_THREADS>(s, xw_ring_place(s.pub, s.fa.N, wg, smem), smem);
    } else if (wg < nx + nn) {
        step_noise<D, XW_THREADS>(s, mode, wg - nx, smem);
    } else {
        const int nt = (s.fa.N + FORCE_TILE - 1) / FORCE_TILE, id = wg - nx - nn;
        if constexpr (KIND != POT_FREE) {
            if (s.pg.G) {
                group_forces<D, KIND>(s.fa, s.pg, id, s.x, s.f, s.fext, s.fpart, smem);
                return;
            }
        }
        bead_forces_tile<D, KIND>(s.fa, id / nt, id % nt, s.x, s.f, s.fext, s.fpart, smem);
    }
}

template <int D>
static __global__ void __launch_bounds__(256) k_step_integrate(StepArgs s, int mode) {
    if (blockIdx.x == 0 && threadIdx.x == 0 && mode != STEP_CLOSE) *s.ctr += 1;
    step_integrate<D>(s, mode, blockIdx.x);
}

// ---- the normal-mode propagator (distinguishable particles) ----
// What k_step_integrate does, with the kicks on the physical forces fext and
// the free ring polymer's rotation of the modes for the drift
// (normal_modes_propagator.cpp:19-53): 16 columns (one axis) of all beads per
// workgroup, the four P x P products on the matrix cores (step_noise's lane
// layout).  OPEN and FULL; a closing half is step_integrate's.  What bounds it
// is latency (21 workgroups for N=101): a step of N=101, P=24 took 25.8 us as
// k_momenta, k_nm_propagate, forces and k_momenta and takes 16.3 so, half of it
// this kernel.
constexpr int MODE_COLS = 16;
__host__ __device__ inline int step_modes_groups(int N, int D) { return D * ((N + MODE_COLS - 1) / MODE_COLS); }
__host__ __device__ inline size_t step_modes_lds_doubles(int P) { return (size_t)step_pad16(P) * (4 * MODE_COLS + 4); }

template <int D>
static __global__ void __launch_bounds__(256) k_step_modes(StepArgs s, int mode) {
    extern __shared__ __align__(16) double smem[];
    __shared__ double shift[4];
    constexpr int NW = 256 / WAVE, KMAX = STEP_NM_MAXP / 4, EMAX = STEP_NM_MAXP * MODE_COLS / 256;
    const StepCoef co = step_coef(s, mode);
    const int N = s.fa.N, P = s.fa.P, tiles = (N + MODE_COLS - 1) / MODE_COLS;
    const int a = blockIdx.x / tiles, i0 = (blockIdx.x % tiles) * MODE_COLS, nc = min(MODE_COLS, N - i0);
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int q4 = lane / 16, c16 = lane % 16;
    const int Pp = step_pad16(P), MB = Pp / 16, KK = Pp / 4, ntask = 2 * MB;   // task: 16 rows of x or of p
    if (blockIdx.x == 0 && tid == 0) *s.ctr += 1;
    double* in = smem;                                // [x, p'][bead][16]
    double* md = in + 2 * (size_t)Pp * MODE_COLS;     // [x, p'][mode][16]
    double* rc = md + 2 * (size_t)Pp * MODE_COLS;     // [mode][4]: x = xx q + xp p, p = px q + pp p
    // all loads first: the elements, then a wave's rows of both matrices
    double xv[EMAX], pv[EMAX], fv[EMAX], hv[EMAX];
#pragma unroll
    for (int u = 0; u < EMAX; ++u) {
        const int e = tid + u * 256, b = e / MODE_COLS, c = e % MODE_COLS;
        xv[u] = pv[u] = fv[u] = hv[u] = 0.0;
        if (b < P && c < nc) {
            const size_t g = ((size_t)b * D + a) * N + i0 + c;
            xv[u] = s.x[g];
            pv[u] = s.p[g];
            fv[u] = s.fext[g];
            if (s.thermostat) hv[u] = s.H[g];
        }
    }
    double A[KMAX], B[KMAX];
    auto rows = [&](const double* M, int bb, double (&R)[KMAX]) {
        const int m = bb * 16 + c16;
#pragma unroll
        for (int kk = 0; kk < KMAX; ++kk) {
            if (kk >= KK) break;
            const int k = 4 * kk + q4;
            const double v = M[(size_t)min(k, P - 1) * P + min(m, P - 1)];
            R[kk] = k < P && m < P ? v : 0.0;
        }
    };
    if (wave < ntask) {
        rows(s.Ct, wave % MB, A);
        rows(s.CTt, wave % MB, B);
    }
    if (tid < Pp) {
        double xx = 0.0, xp = 0.0, px = 0.0, pp = 0.0;
        if (tid < P) {
            const double cs = s.rot[4 * tid], sn = s.rot[4 * tid + 1], mw = s.rot[4 * tid + 2], w = s.rot[4 * tid + 3];
            xx = w == 0 ? 1.0 : cs;
            xp = w == 0 ? s.dt_m : sn / mw;
            px = w == 0 ? 0.0 : (-1) * mw * sn;
            pp = w == 0 ? 1.0 : cs;
        }
        rc[4 * tid] = xx;
        rc[4 * tid + 1] = xp;
        rc[4 * tid + 2] = px;
        rc[4 * tid + 3] = pp;
    }
    if (s.fixcom) {
        step_shift<D>(s, mode, wave, lane, shift);
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < EMAX; ++u) {
        const int e = tid + u * 256;
        if (e < Pp * MODE_COLS) {
            double v = step_kept(co, fma(co.beta, fv[u], pv[u]), hv[u]);
            if (s.fixcom) v -= shift[a];
            in[e] = xv[u];
            in[Pp * MODE_COLS + e] = e / MODE_COLS < P ? fma(co.gamma, fv[u], v) : 0.0;
        }
    }
    __syncthreads();
    auto product = [&](int t, const double* M, double (&R)[KMAX], auto&& operand, auto&& store) {
        const int bb = t % MB;
        if (t != wave && bb != wave % MB) rows(M, bb, R);
        step_v4d acc[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};   // (two chains; KK is a multiple of 4)
#pragma unroll
        for (int kk = 0; kk < KMAX; ++kk)
            if (kk < KK) acc[kk % 2] = __builtin_amdgcn_mfma_f64_16x16x4f64(R[kk], operand(4 * kk + q4), acc[kk % 2], 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 4; ++v) store(bb * 16 + q4 + 4 * v, acc[0][v] + acc[1][v]);
    };
    for (int t = wave; t < ntask; t += NW) {
        const size_t o = (size_t)(t / MB) * Pp * MODE_COLS + c16;
        product(t, s.Ct, A, [&](int k) { return in[o + k * MODE_COLS]; },
                [&](int k, double v) { md[o + k * MODE_COLS] = v; });
    }
    __syncthreads();
    for (int t = wave; t < ntask; t += NW) {
        const int w = t / MB;
        double* out = w == 0 ? s.x : s.p;
        product(t, s.CTt, B,
                [&](int k) {
                    const double q = md[k * MODE_COLS + c16], pm = md[(Pp + k) * MODE_COLS + c16];
                    return fma(rc[4 * k + 2 * w], q, rc[4 * k + 2 * w + 1] * pm);
                },
                [&](int b, double v) {
                    if (b < P && c16 < nc) out[((size_t)b * D + a) * N + i0 + c16] = v;
                });
    }
}

}  // namespace pimdb
