// pimdb_split.hip -- the two-kernel form of a batched MD step (batch_split.hpp).
//
// What bounds it.  The persistent kernel gives a replica one workgroup: 16
// helium replicas (N=256, P=64) kept 16 of 256 compute units busy and took
// 1236 us a step, as long as 256 of them.  Here a replica's step is spread
// over workgroups of 256 threads: its recursions (one per block of 64 targets
// and direction), slices (a bead on one, two or four waves), noise tiles, and the integration's
// rows.  The pair walk is then bound by vector issue at every replica count;
// what it costs against the persistent kernel is the second exponential per
// exchange term (the recursions and the exterior forces do not share them,
// about 80 us of one CU per replica against 1090 for its pairs).
//
// The recursions of all replicas come first, a ring's blocks in the order of
// their start (xw_place), then slices and noise tiles, the
// longest first, so that the last round over the card is a short one.  Three
// workgroups share a compute unit (44 KB of LDS, the ring of N=256), since the
// noise no longer stages C^T (66 KB).  With these two and one particle a wave in
// the exterior forces, helium N=256, P=64: 4 replicas 64.4 -> 58.2 us a step, 16
// 148.5 -> 121.6, 40 335 -> 268, 128 875 -> 718.
#include "batch_split.hpp"

namespace pimdb {

// Slice workgroup id of a replica: the pair, trap and spring forces of
// SPLIT_WAVES / share beads (wg_bead_forces of batch.hpp, with a slice's pairs
// cut over `share` waves and their force arrays added in wave order).
// Exchange beads get the physical forces; fpart (may be null): the external
// forces' sums per (bead, wave) and axis.
template <int D, int KIND>
__device__ __noinline__ void split_slice(const RepDesc& r_, const BatchPtrs& bp, double* lds_, int id_, int share_,
                                         int plds_, double* fpart_) {
    const RepDesc r = rep_uniform(r_);
    const int id = uni(id_), share = uni(share_);
    double* fpart = uni(fpart_);
    lds_double* F = (lds_double*)uni(lds_);
    const int N = r.N, P = r.P;
    const double* x = uni(bp.x) + r.off_x;
    double* f = uni(bp.f) + r.off_x;
    const bool pbc = r.pbc != 0;
    const double invL = 1.0 / r.L, invL_s = pbc ? invL : 0.0;
    const size_t bs = (size_t)D * N;
    const int lane = threadIdx.x % WAVE;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
    const int sub = wave % share;                                  // the wave's part of its slice
    const int b = id * (SPLIT_WAVES / share) + wave / share;       // its bead
    const PairParams pp = make_pair_params(r.L, r.pbc, r.cutoff, r.cut2, r.int_k, r.strength);
    FracParams fp = make_frac_params(pp);
    fp.cut2 = uni(fp.cut2); fp.kh = uni(fp.kh); fp.kd = uni(fp.kd); fp.ex = uni(fp.ex);
    fp.b0 = uni(fp.b0); fp.b1 = uni(fp.b1); fp.b2 = uni(fp.b2); fp.dl = uni(fp.dl);
    fp.b1v = vgpr_copy(fp.b1);
    fp.b2v = vgpr_copy(fp.b2);
    const size_t fs = (size_t)pair_fstride(D) * N;
    lds_double* Fw = F + (size_t)wave * fs;
    lds_int* perm = (lds_int*)(F + (size_t)SPLIT_WAVES * fs);   // [N] particle at each tile position
    lds_int* iperm = perm + N;                                   // [N] tile position of each particle
    const bool pairs = KIND != POT_FREE && r.cutoff != 0.0;
    const bool in_lds = pairs && uni(plds_) != 0;
    if (in_lds) {
        lds_uint* key = (lds_uint*)F;
        const bool order = KIND == POT_AZIZ && pbc;
        for (int i = threadIdx.x; i < N; i += SPLIT_THREADS) {
            double xi[D];
#pragma unroll
            for (int a = 0; a < D; ++a) xi[a] = x[a * N + i];
            key[i] = order ? pair_order_key<D>(xi, invL, N, i) : (unsigned)i;
        }
        __syncthreads();
        for (int i = threadIdx.x; i < N; i += SPLIT_THREADS) {
            const unsigned ki = key[i];
            int rank = i;
            if (order) {
                rank = 0;
                for (int j = 0; j < N; ++j) rank += key[j] < ki ? 1 : 0;
            }
            perm[rank] = i;
            iperm[i] = rank;
        }
        __syncthreads();
    }
    const bool live = b < P;
    const double* xs = x + bs * (live ? b : 0);
    double* fo = f + bs * (live ? b : 0);
    if (in_lds) {
        if (live && share == 1) {
            switch (pair_image(pp)) {
            case 0: slice_pair_forces_lds<D, KIND, 0>(xs, N, WalkGrad<D, KIND, 0>{pp, fp}, lane, Fw, perm); break;
            case 1: slice_pair_forces_lds<D, KIND, 1>(xs, N, WalkGrad<D, KIND, 1>{pp, fp}, lane, Fw, perm); break;
            default: slice_pair_forces_lds<D, KIND, 2>(xs, N, WalkGrad<D, KIND, 2>{pp, fp}, lane, Fw, perm); break;
            }
        } else if (live) {
            switch (pair_image(pp)) {
            case 0: slice_pair_forces_part<D, KIND, 0>(xs, N, WalkGrad<D, KIND, 0>{pp, fp}, lane, Fw, perm, sub, share); break;
            case 1: slice_pair_forces_part<D, KIND, 1>(xs, N, WalkGrad<D, KIND, 1>{pp, fp}, lane, Fw, perm, sub, share); break;
            default: slice_pair_forces_part<D, KIND, 2>(xs, N, WalkGrad<D, KIND, 2>{pp, fp}, lane, Fw, perm, sub, share); break;
            }
        }
        __syncthreads();
    } else if (live && pairs) {   // (share 1)
        switch (pair_image(pp)) {
        case 0: slice_pair_forces<D, KIND, 0>(xs, fo, N, pp, lane); break;
        case 1: slice_pair_forces<D, KIND, 1>(xs, fo, N, pp, lane); break;
        default: slice_pair_forces<D, KIND, 2>(xs, fo, N, pp, lane); break;
        }
    }
    if (!live) return;
    const bool exchange_bead = r.bosonic && (b == 0 || b == P - 1);
    const double* xprev = x + bs * ((b - 1 + P) % P);
    const double* xnext = x + bs * ((b + 1) % P);
    const lds_double* Fb = F + (size_t)(wave - sub) * fs;
    double fsum[D];
#pragma unroll
    for (int a = 0; a < D; ++a) fsum[a] = 0.0;
    for (int i = sub * WAVE + lane; i < N; i += share * WAVE) {
        double xv[D], fe[D];
        const int ip = in_lds ? iperm[i] * pair_fstride(D) : 0;
#pragma unroll
        for (int a = 0; a < D; ++a) xv[a] = xs[a * N + i];
        ext_force<D>(r.ext, xv, fe);
#pragma unroll
        for (int a = 0; a < D; ++a) {
            const int e = a * N + i;
            fsum[a] += fe[a];
            double pr = 0.0;
            if (in_lds) {
                for (int w = 0; w < share; ++w) pr += Fb[(size_t)w * fs + ip + a];
            } else if (pairs) {
                pr = fo[e];
            }
            const double phys = fe[a] + pr;
            double spring = 0.0;
            if (!exchange_bead)
                spring = r.k * (disp_fast(xv[a], xprev[e], pbc, r.L, invL_s) + disp_fast(xv[a], xnext[e], pbc, r.L, invL_s));
            fo[e] = exchange_bead ? phys : spring + phys;
        }
    }
    if (fpart) {
#pragma unroll
        for (int a = 0; a < D; ++a) {
            const double t = wave_total(fsum[a]);
            if (lane == 0) fpart[((size_t)b * share + sub) * D + a] = t;
        }
    }
}

template <int D, int KIND>
static __global__ void __launch_bounds__(SPLIT_THREADS, 4) k_split_forces(SplitPtrs sp, const int2* __restrict__ map,
                                                                        int only_noise, int mode) {
    extern __shared__ __align__(16) double smem[];
    const int2 m = map[blockIdx.x];
    const int ri = uni(m.x), id = uni(m.y);
    const StepArgs s = sp.steps[ri];   // (a copy: stores through it would make every use a load)
    const int N = s.fa.N, P = s.fa.P;
    const int nx = only_noise || !s.fa.bosonic ? 0 : xw_grid(N), nn = step_noise_groups(s, D);
    if (id < nx) {
        step_recursions<D, SPLIT_THREADS>(s, xw_ring_place(s.pub, N, id, smem), smem);
    } else if (id < nx + nn) {
        if (mode != STEP_FORCES) step_noise<D, SPLIT_THREADS>(s, mode, id - nx, smem);
    } else {
        split_slice<D, KIND>(sp.bp.reps[ri], sp.bp, smem, id - nx - nn, sp.share, split_slice_lds(N, D) <= sp.lds, s.fpart);
    }
}

template <int D>
static __global__ void __launch_bounds__(SPLIT_THREADS) k_split_integrate(SplitPtrs sp, const int2* __restrict__ map,
                                                                           int mode) {
    const int2 m = map[blockIdx.x];
    const StepArgs s = sp.steps[uni(m.x)];
    if (blockIdx.x == 0 && threadIdx.x == 0 && mode <= STEP_FULL) *s.ctr += 1;
    step_integrate<D>(s, mode, uni(m.y));
}

template <int D>
static __global__ void __launch_bounds__(256) k_split_settle(BatchPtrs bp) {
    const int ri = blockIdx.x;
    const RepDesc& r = bp.reps[ri];
    double* cmp = bp.cmp + 8 * (size_t)ri;
    const int n = r.P * D * r.N;
    double* p = bp.p + r.off_x;
    double cm[D];
#pragma unroll
    for (int a = 0; a < D; ++a) cm[a] = cmp[a];
    for (int e = threadIdx.x; e < n; e += blockDim.x) p[e] -= cm[elem_axis<D>(e, r.N)];
    __syncthreads();
    if (threadIdx.x < 8) cmp[threadIdx.x] = 0.0;
}

template <int D>
static void forces_d(const SplitPtrs& sp, int kind, bool forces, int mode, hipStream_t s) {
    const dim3 grid(forces ? sp.nforces : sp.nnoise), blk(SPLIT_THREADS);
    if (grid.x == 0) return;
    const int2* map = forces ? sp.forces_map : sp.noise_map;
    const int only = forces ? 0 : 1;
    switch (kind) {
    case POT_HARMONIC: hipLaunchKernelGGL((k_split_forces<D, POT_HARMONIC>), grid, blk, sp.lds, s, sp, map, only, mode); break;
    case POT_DIPOLE: hipLaunchKernelGGL((k_split_forces<D, POT_DIPOLE>), grid, blk, sp.lds, s, sp, map, only, mode); break;
    case POT_AZIZ: hipLaunchKernelGGL((k_split_forces<D, POT_AZIZ>), grid, blk, sp.lds, s, sp, map, only, mode); break;
    default: hipLaunchKernelGGL((k_split_forces<D, POT_FREE>), grid, blk, sp.lds, s, sp, map, only, mode); break;
    }
}

hipError_t launch_split_forces(const SplitPtrs& sp, int D, int kind, bool forces, int mode, hipStream_t s) {
    switch (D) {
    case 1: forces_d<1>(sp, kind, forces, mode, s); break;
    case 2: forces_d<2>(sp, kind, forces, mode, s); break;
    default: forces_d<3>(sp, kind, forces, mode, s); break;
    }
    return hipGetLastError();
}

hipError_t launch_split_integrate(const SplitPtrs& sp, int D, int mode, hipStream_t s) {
    const dim3 grid(mode == STEP_OPEN ? sp.nopen : sp.nfull), blk(SPLIT_THREADS);
    const int2* map = mode == STEP_OPEN ? sp.open_map : sp.full_map;
    switch (D) {
    case 1: hipLaunchKernelGGL(k_split_integrate<1>, grid, blk, 0, s, sp, map, mode); break;
    case 2: hipLaunchKernelGGL(k_split_integrate<2>, grid, blk, 0, s, sp, map, mode); break;
    default: hipLaunchKernelGGL(k_split_integrate<3>, grid, blk, 0, s, sp, map, mode); break;
    }
    return hipGetLastError();
}

hipError_t launch_split_settle(const BatchPtrs& bp, int D, int nrep, hipStream_t s) {
    switch (D) {
    case 1: hipLaunchKernelGGL(k_split_settle<1>, dim3(nrep), dim3(256), 0, s, bp); break;
    case 2: hipLaunchKernelGGL(k_split_settle<2>, dim3(nrep), dim3(256), 0, s, bp); break;
    default: hipLaunchKernelGGL(k_split_settle<3>, dim3(nrep), dim3(256), 0, s, bp); break;
    }
    return hipGetLastError();
}

}  // namespace pimdb
