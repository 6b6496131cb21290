// batch_split.hpp -- the two-kernel form of a batched MD step (steps.hpp with
// many replicas per launch), for batches that the persistent kernel (batch.hpp,
// one workgroup per replica) would leave the card idle or unevenly loaded with.
#pragma once

#include <hip/hip_runtime.h>

#include "batch.hpp"
#include "steps.hpp"

namespace pimdb {

// Threads of a workgroup of either kernel.
constexpr int SPLIT_THREADS = 256;
constexpr int SPLIT_WAVES = SPLIT_THREADS / WAVE;

// A workgroup's part of a forces launch: its replica and its index among the
// replica's workgroups (recursions first, then noise, then slices).
struct SplitPtrs {
    BatchPtrs bp;
    const StepArgs* steps;       // per replica
    const int2* forces_map;      // (replica, index) of every workgroup of k_split_forces
    const int2* noise_map;       // of the noise workgroups alone (an opening half)
    const int2* full_map;        // of k_split_integrate after forces
    const int2* open_map;        // and of an opening half
    int nforces, nnoise, nfull, nopen;
    size_t lds;                  // dynamic LDS of k_split_forces
    int share;                   // waves per slice: 1, 2 or 4
};

// LDS bytes of a slice workgroup: the force arrays of its waves and the tile
// order.  A replica whose slices exceed a workgroup's LDS accumulates them in
// device memory (pairs.hpp, slice_pair_forces; share 1).
__host__ __device__ inline size_t split_slice_lds(int N, int D) {
    return sizeof(double) * ((size_t)SPLIT_WAVES * pair_fstride(D) * N + N);
}
// Slice workgroups of a replica.
__host__ __device__ inline int split_slices(int P, int share) { return (P * share + SPLIT_WAVES - 1) / SPLIT_WAVES; }

// Launches on s: the forces of every replica (forces false: only the noise)
// with the noise of the integration of this mode, and that integration.
hipError_t launch_split_forces(const SplitPtrs& sp, int D, int kind, bool forces, int mode, hipStream_t s);
hipError_t launch_split_integrate(const SplitPtrs& sp, int D, int mode, hipStream_t s);
// p -= the momentum still pending from the persistent kernel's last O-step.
hipError_t launch_split_settle(const BatchPtrs& bp, int D, int nrep, hipStream_t s);

}  // namespace pimdb
