// slice_groups.hpp -- pair forces of a single system with Newton's third law:
// every bead's particles in groups of 128, a workgroup per (bead, group).
//
// Reference: Simulation::updatePhysicalForces (src/simulation.cpp:428-455).
//
// Why.  bead_forces_tile (forces.hpp) evaluates every ordered pair: N=256, P=64
// helium spent 29.6 us a step in forces beside recursions of 19.3, N=1000, P=32
// 126 beside 54.  Its workgroups (64 rows, one to a compute unit) are also twice
// as many as these, so their last round over the card is nearly empty more
// often.  What bounds these: vector issue, 36 us for the 33 steps per wave of
// N=1000 (four waves a SIMD, 2 x 83 issue slots of 4 cycles a step).  A whole
// Langevin step, both with pair_grad_image: N=256, P=64 39.7 -> 25.3 us, N=500,
// P=32 63.6 -> 35.7, N=1000, P=32 159 -> 79 and P=64 257 -> 120; without exchange
// N=1000, P=4 54.8 -> 21.3, N=300, P=4 25.2 -> 17.1.
//
// Work.  Group g meets itself and, of the other G - 1 groups on a ring, those
// at distances 1 .. (G-1)/2 ahead, and for even G half of the pairs with the
// group opposite: rows l of the one and columns l + s of the other, offsets
// s = 0..31 by the lower group, 32..63 (seen from the other side, 1..32) by
// the higher.  So all workgroups do the same work, and each unordered pair is
// met once.  The work is a sequence of steps, two rows per lane against one
// column each, in segments
//   tile A with itself, tile B with itself (17 steps each: SliceWalk's
//   diagonal tile, pairs.hpp), rows l and l+32 of A against B (32 steps),
//   then A and B against one tile of another group (64 steps; 32 opposite),
// cut evenly over the waves, and over several workgroups ("parts") at segment
// bounds: for the beads of the last round over the card, which whole groups
// would leave nearly empty, or for all where they are too few to fill it.
//
// Sums.  A wave accumulates its rows, and the columns of the group's own
// tiles, in an LDS array of its own, and every other column tile in a slot of
// its own; the waves' arrays are then added in wave order, so the result does
// not depend on timing.  The rows become f (with the external and spring
// forces); the columns go to cpart[distance - 1], one value per particle and
// distance, and the rows of part p > 0 to cpart[G/2 + p - 1].  The reader of f
// adds these (step_integrate, k_pair_sum).
#pragma once

#include "device_common.hpp"
#include "forces.hpp"
#include "pairs.hpp"

namespace pimdb {

constexpr int GROUP = 2 * PTILE;
constexpr int GROUP_WAVES = FORCE_WAVES;
// Particles above which groups are used: one group is half idle (N=128, P=64
// without exchange 17.7 us a step against 16.9 by tiles of 64 rows).
constexpr int GROUP_MIN = GROUP;
constexpr int GROUP_PARTS = 4;  // parts at most
constexpr int GROUP_OWN = 17 + 17 + 32;   // steps of a group with itself

struct PairGroups {
    int G, kslots;      // groups (0: bead_forces_tile), LDS slots per wave
    int b1, q1, q2;     // parts per group: q1 for beads below b1, q2 for the others
    double* cpart;      // [slots][P][D][N]
    __host__ __device__ int parts(int b) const { return b < b1 ? q1 : q2; }
    __host__ __device__ int slots(int b) const { return G ? G / 2 + parts(b) - 1 : 0; }   // those of bead b
    __host__ __device__ int max_slots(int P) const { return b1 < P ? slots(P - 1) : slots(0); }   // (q1 <= q2)
    __host__ __device__ int groups_of(int P) const { return G * (b1 * q1 + (P - b1) * q2); }      // workgroups
};

// Segments of a group with others, their first steps, and a part's first segment.
__host__ __device__ inline int group_segments(int G) { return G - 1 + (G % 2 == 0 ? 1 : 0); }
__host__ __device__ inline int group_seg_start(int G, int e) {
    const int n = 2 * ((G - 1) / 2);
    return e <= n ? PTILE * e : PTILE * n + (PTILE / 2) * (e - n);
}
__host__ __device__ inline int group_seg_at(int G, int step) {   // the segment that a step belongs to
    const int n = 2 * ((G - 1) / 2);
    return step < PTILE * n ? step / PTILE : n + (step - PTILE * n) / (PTILE / 2);
}
__host__ __device__ inline int group_part_first(int G, int parts, int p) {
    const int n = group_segments(G);
    if (p <= 0) return 0;
    if (p >= parts) return n;
    const int at = (GROUP_OWN + group_seg_start(G, n)) * p / parts - GROUP_OWN;
    return at <= 0 ? 0 : (at + PTILE / 2 >= group_seg_start(G, n) ? n : group_seg_at(G, at + PTILE / 2));
}
// A part's steps: segments [e0, e1) behind `own` steps of the group with itself.
struct GroupPart {
    int e0, e1, own, first, steps;   // first: group_seg_start(e0)
    __host__ __device__ GroupPart(int G, int parts, int p)
        : e0(group_part_first(G, parts, p)), e1(group_part_first(G, parts, p + 1)), own(p == 0 ? GROUP_OWN : 0),
          first(group_seg_start(G, e0)), steps(own + group_seg_start(G, e1) - first) {}
    __host__ __device__ int lo(int w) const { return steps * w / GROUP_WAVES; }
    // first segment of wave w (its slot 0), given that it has one
    __host__ __device__ int wave_seg(int G, int w) const {
        const int at = lo(w) - own;
        return group_seg_at(G, first + (at > 0 ? at : 0));
    }
};
// LDS slots per wave: the most segments that a wave meets.
inline int group_kslots(int G, int parts) {
    int k = 0;
    for (int p = 0; p < parts; ++p) {
        const GroupPart gp(G, parts, p);
        for (int w = 0; w < GROUP_WAVES; ++w) {
            const int hi = gp.lo(w + 1) - gp.own;
            if (hi <= 0 || gp.lo(w + 1) == gp.lo(w)) continue;
            const int n = group_seg_at(G, gp.first + hi - 1) - gp.wave_seg(G, w) + 1;
            k = n > k ? n : k;
        }
    }
    return k;
}
__host__ __device__ inline size_t group_lds_doubles(int D, int kslots) {
    return (size_t)GROUP_WAVES * pair_fstride(D) * (GROUP + kslots * PTILE);
}

// One wave's walk: rows in registers, columns rotating (pairs.hpp).
template <int D, int KIND, int IMG>
struct GroupWalk {
    gbl_cdptr xs;
    int N;
    const ImageGrad<D, KIND, IMG>& wg;
    int lane;
    double xj[D];
    int jd;   // LDS byte address of the column's sums; negative: no column

    // Particle i's position, and whether it takes part: not beyond the slice, nor,
    // with a cutoff, where a coordinate is not finite, since no distance to it is
    // below the cutoff.  The position of one that does not is finite, since the
    // sums take its products with 0 (a step of N=256, P=64 27.3 -> 27.6 us, the state
    // read every 50).
    __device__ __forceinline__ bool load(int i, double (&x)[D]) const {
        bool ok = i < N;
        double t = 0.0;
#pragma unroll
        for (int a = 0; a < D; ++a) {
            x[a] = xs[a * N + (ok ? i : 0)];
            t += x[a] - x[a];   // (0 or NaN)
        }
        ok = ok && (wg.pp.cutoff < 0.0 || t == 0.0);
#pragma unroll
        for (int a = 0; a < D; ++a) x[a] = ok ? x[a] : 0.0;
        return ok;
    }
    __device__ __forceinline__ void rotate() {
#pragma unroll
        for (int a = 0; a < D; ++a) xj[a] = lane_rotate(xj[a]);
        jd = lane_rotate(jd);
    }
    __device__ __forceinline__ void pairs(const double (&xa)[D], const double (&xb)[D], double (&ra)[D],
                                          double (&rb)[D], bool acta, bool actb) {
        double da[D], db[D], ga = 0.0, gb = 0.0;
        const bool ina = wg(xa, xj, da, ga) && acta;
        const bool inb = wg(xb, xj, db, gb) && actb;
        if (ina || inb) {
            if (!ina) ga = 0.0;
            if (!inb) gb = 0.0;
            lds_double* Fj = (lds_double*)(size_t)(unsigned)jd;
#pragma unroll
            for (int a = 0; a < D; ++a) {
                ra[a] = fma(-ga, da[a], ra[a]);
                rb[a] = fma(-gb, db[a], rb[a]);
                __hip_atomic_fetch_add(&Fj[a], fma(ga, da[a], gb * db[a]), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
    }
    // rows ia and ib against tile J (its first particle j0, sums at Fc),
    // offsets [s0, s1).  DIAG: the tile with itself, offsets 0 .. 16.
    template <bool DIAG>
    __device__ __forceinline__ void segment(int ia, int ib, lds_double* fa, lds_double* fb, int j0, lds_double* Fc,
                                            int s0, int s1) {
        double xa[D], xb[D], ra[D] = {}, rb[D] = {};
        const bool oka = load(ia, xa), okb = load(ib, xb);
        const int c = (lane + s0) & (PTILE - 1);
        jd = load(j0 + c, xj) ? (int)(unsigned)(size_t)(Fc + c * pair_fstride(D)) : -1;
        for (int s = s0; s < s1; ++s) {
            const bool ok = jd >= 0;
            bool acta = oka && ok, actb = okb && ok;
            if constexpr (DIAG) {
                if (s == 0) {
                    acta = false;
                    actb = actb && lane < PTILE / 2;
                }
                if (s == PTILE / 4) actb = false;
            }
            pairs(xa, xb, ra, rb, acta, actb);
            rotate();
        }
#pragma unroll
        for (int a = 0; a < D; ++a) {
            if (oka) __hip_atomic_fetch_add(&fa[a], ra[a], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (okb) __hip_atomic_fetch_add(&fb[a], rb[a], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    }
};

// One wave's steps [lo, hi) of a part.  R: the wave's sums of the group's own
// particles [GROUP][S]; slots: [kslots][PTILE][S].
template <int D, int KIND, int IMG>
__device__ __forceinline__ void group_walk(const double* xs, int N, const ImageGrad<D, KIND, IMG>& wg, int g, int G,
                                           const GroupPart& gp, int lo, int hi, int lane, lds_double* R,
                                           lds_double* slots) {
    constexpr int S = pair_fstride(D);
    GroupWalk<D, KIND, IMG> w{(gbl_cdptr)xs, N, wg, lane, {}, 0};
    const int i0 = g * GROUP, l2 = (lane + PTILE / 2) & (PTILE - 1);
    const int nB = i0 + PTILE;   // tile B's first particle
    if (lo < gp.own) {
        for (int t = 0; t < 2; ++t) {
            const int a = lo - 17 * t > 0 ? lo - 17 * t : 0, b = hi - 17 * t < 17 ? hi - 17 * t : 17;
            if (a < b && i0 + t * PTILE < N) {
                lds_double* Rt = R + t * PTILE * S;
                w.template segment<true>(i0 + t * PTILE + lane, i0 + t * PTILE + l2, Rt + lane * S, Rt + l2 * S,
                                         i0 + t * PTILE, Rt, a, b);
            }
        }
        const int a = lo - 34 > 0 ? lo - 34 : 0, b = hi - 34 < 32 ? hi - 34 : 32;
        if (a < b && nB < N)
            w.template segment<false>(i0 + lane, i0 + l2, R + lane * S, R + l2 * S, nB, R + PTILE * S, a, b);
    }
    if (hi <= gp.own || hi <= lo) return;
    const int from = gp.first + (lo > gp.own ? lo - gp.own : 0), to = gp.first + hi - gp.own;
    const int nfull = 2 * ((G - 1) / 2);
    int at = from;
    for (int e = group_seg_at(G, from); at < to; ++e, slots += PTILE * S) {
        const int start = group_seg_start(G, e), end = min(to, group_seg_start(G, e + 1));
        const int d = e < nfull ? 1 + e / 2 : G / 2, h = g + d < G ? g + d : g + d - G;
        const int shift = e >= nfull && h < g ? 1 : 0;
        const int j0 = h * GROUP + ((e - (e < nfull ? 0 : nfull)) & 1) * PTILE;
#pragma unroll
        for (int a = 0; a < S; ++a) slots[a * PTILE + lane] = 0.0;
        __builtin_amdgcn_wave_barrier();
        if (j0 < N)
            w.template segment<false>(i0 + lane, nB + lane, R + lane * S, R + (PTILE + lane) * S, j0, slots,
                                      at - start + shift, end - start + shift);
        at = end;
    }
}

// Workgroup id of pg.groups_of(P): the forces of one part of one group of one
// bead, by 1024 threads: as bead_forces_tile, with the pair forces of other
// workgroups' rows and of other parts left in pg.cpart.
template <int D, int KIND>
__device__ __forceinline__ void group_forces(const ForceArgs& fa, const PairGroups& pg, int id, const double* __restrict__ x,
                                             double* __restrict__ f, double* __restrict__ fext,
                                             double* __restrict__ fpart, double* smem) {
    constexpr int S = pair_fstride(D);
    const int N = fa.N, P = fa.P, G = pg.G;
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
    const int n1 = G * pg.b1 * pg.q1, at = id < n1 ? id : id - n1, parts = id < n1 ? pg.q1 : pg.q2;
    const int part = at % parts, bg = at / parts, g = bg % G, b = bg / G + (id < n1 ? 0 : pg.b1);
    const size_t bs = (size_t)D * N;
    const double* xb = x + bs * b;
    const GroupPart gp(G, parts, part);
    lds_double* R0 = (lds_double*)smem;
    lds_double* slots0 = R0 + GROUP_WAVES * GROUP * S;
    lds_double* R = R0 + wave * GROUP * S;
    for (int e = lane; e < GROUP * S; e += WAVE) R[e] = 0.0;
    __builtin_amdgcn_wave_barrier();
    {
        const PairParams pp = make_pair_params(fa.L, fa.pbc, fa.cutoff, fa.cut2, fa.int_k, fa.strength);
        lds_double* slots = slots0 + (size_t)wave * pg.kslots * PTILE * S;
        const int lo = gp.lo(wave), hi = gp.lo(wave + 1);
        auto walk = [&](auto img) {
            constexpr int IMG = decltype(img)::value;
            group_walk<D, KIND, IMG>(xb, N, ImageGrad<D, KIND, IMG>{pp, image_params<KIND, IMG>(pp)}, g, G, gp, lo, hi,
                                     lane, R, slots);
        };
        switch (pair_image(pp)) {
        case 0: walk(std::integral_constant<int, 0>()); break;
        case 1: walk(std::integral_constant<int, 1>()); break;
        default: walk(std::integral_constant<int, 2>()); break;
        }
    }
    __syncthreads();
    // tasks 0 and 1: the rows of tiles A and B; then the column tiles
    const int ntask = 2 + gp.e1 - gp.e0;
    for (int task = wave; task < ntask; task += GROUP_WAVES) {
        double sum[D];
#pragma unroll
        for (int a = 0; a < D; ++a) sum[a] = 0.0;
        if (task >= 2) {
            const int e = gp.e0 + task - 2, nfull = 2 * ((G - 1) / 2);
            const int d = e < nfull ? 1 + e / 2 : G / 2, h = g + d < G ? g + d : g + d - G;
            const int j = h * GROUP + ((e - (e < nfull ? 0 : nfull)) & 1) * PTILE + lane;
            const int s0 = gp.own + group_seg_start(G, e) - gp.first, s1 = gp.own + group_seg_start(G, e + 1) - gp.first;
            if (j >= N) continue;
            for (int w = 0; w < GROUP_WAVES; ++w) {
                const int lo = gp.lo(w), hi = gp.lo(w + 1);
                if (hi <= s0 || lo >= s1 || hi == lo) continue;
                const lds_double* c = slots0 + ((size_t)w * pg.kslots + (e - gp.wave_seg(G, w))) * PTILE * S + lane * S;
#pragma unroll
                for (int a = 0; a < D; ++a) sum[a] += c[a];
            }
#pragma unroll
            for (int a = 0; a < D; ++a) pg.cpart[((size_t)(d - 1) * P + b) * bs + (size_t)a * N + j] = sum[a];
            continue;
        }
        const int i = g * GROUP + task * PTILE + lane;
        const bool mine = i < N;
#pragma unroll
        for (int w = 0; w < GROUP_WAVES; ++w) {
#pragma unroll
            for (int a = 0; a < D; ++a) sum[a] += R0[(w * GROUP + task * PTILE + lane) * S + a];
        }
        if (part > 0) {
            if (mine) {
#pragma unroll
                for (int a = 0; a < D; ++a)
                    pg.cpart[((size_t)(G / 2 + part - 1) * P + b) * bs + (size_t)a * N + i] = sum[a];
            }
            continue;
        }
        double fe[D];
#pragma unroll
        for (int a = 0; a < D; ++a) fe[a] = 0.0;
        if (mine) row_forces<D>(fa, b, i, x, sum, f, fext, fe);
        if (fpart && g * 2 + task < (N + FORCE_TILE - 1) / FORCE_TILE) {
            const int nt = (N + FORCE_TILE - 1) / FORCE_TILE;
#pragma unroll
            for (int a = 0; a < D; ++a) {
                const double s = wave_total(fe[a]);
                if (lane == 0) fpart[((size_t)b * nt + g * 2 + task) * D + a] = s;
            }
        }
    }
}

// The slots' sum into f (and fext), for readers of f that do not add them.
static __global__ void __launch_bounds__(256) k_pair_sum(size_t n, size_t bs, PairGroups pg,
                                                  double* __restrict__ f, double* __restrict__ fext) {
    const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    double s = 0.0;
    for (int k = 0, m = pg.slots((int)(e / bs)); k < m; ++k) s += pg.cpart[k * n + e];
    f[e] += s;
    if (fext) fext[e] += s;
}

}  // namespace pimdb
