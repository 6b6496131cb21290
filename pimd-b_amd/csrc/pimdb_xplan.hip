// pimdb_xplan.hip -- the exchange on caller-provided device arrays: the
// forward V_B kernel chain and its hand-written adjoint, for the autograd
// harness (pimd-b_amd/pimdb_amd/autograd.py).
#include <hip/hip_runtime.h>

#include <string>

#include "pimdb_gpu.h"
#include "ctx_common.hpp"

using namespace pimdb;

struct pimdb_xplan {
    int N = 0, D = 0, pbc = 0;
    double bt = 0.0, k = 0.0, L = 0.0;
    double *V = nullptr, *Vb = nullptr, *Shi = nullptr, *Slo = nullptr;
    unsigned long long* pub = nullptr;   // the recursions' published values (k_exchange_wide)
    double* ws = nullptr;   // the recursions' workspace in device memory, when it exceeds LDS
    int* status = nullptr;
};

// Enqueues the recursions.
static int xplan_recursions(pimdb_xplan* pl, const double* x1, const double* xP, hipStream_t s) {
    launch_exchange_recursions(pl->D, pl->N, pl->bt, pl->k, pl->pbc, pl->L, x1, xP, pl->V, pl->Vb, pl->Shi, pl->Slo,
                               pl->pub, pl->ws, pl->status, s);
    return hipGetLastError() == hipSuccess ? PIMDB_OK : PIMDB_E_HIP;
}

// Waits for the stream and looks at the overflow flag (pinned host memory).
static int xplan_finish(pimdb_xplan* pl, hipStream_t s) {
    if (hipStreamSynchronize(s) != hipSuccess) return PIMDB_E_HIP;
    if (const int st = *(volatile int*)pl->status) {
        *(volatile int*)pl->status = 0;
        if (empty_published(pl->pub, xw_pub_words(pl->N), s) != hipSuccess) return PIMDB_E_HIP;
        return lost_wait(st) ? PIMDB_E_HIP : PIMDB_E_NONFINITE;
    }
    return PIMDB_OK;
}

// Beads given with any strides into SoA [2][D][N].
template <int D>
static __global__ void __launch_bounds__(256) k_gather_beads(int N, BeadView x1, BeadView xP, double* __restrict__ xc) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= D * N) return;
    xc[e] = x1.at(e / N, e % N);
    xc[(size_t)D * N + e] = xP.at(e / N, e % N);
}

// A forward pass's record: V and Vb [N+1], the prefix sums [N] + [N], the beads [2][D][N].
struct Saved {
    double *V, *Vb, *Shi, *Slo, *xc;
    Saved(double* p, int N) : V(p), Vb(p + N + 1), Shi(p + 2 * (size_t)(N + 1)), Slo(Shi + N), xc(Slo + N) {}
};

extern "C" {

int pimdb_xplan_create(int natoms, int ndim, double beta_t, double spring_k, int pbc, double size,
                       pimdb_xplan** out) {
    if (!out || natoms < 1 || ndim < 1 || ndim > 3 || !(beta_t > 0.0) || (pbc && !(size > 0.0))) return PIMDB_E_ARG;
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return PIMDB_E_HIP;
    pimdb_xplan* pl = new pimdb_xplan();
    pl->N = natoms; pl->D = ndim; pl->pbc = pbc; pl->bt = beta_t; pl->k = spring_k; pl->L = size;
    // one allocation: V, Vb, the prefix sums, then the recursions' published
    // values or, for a ring that exceeds a workgroup's LDS, their workspace
    const size_t N = natoms, head = 4 * N + 2;
    const bool wide = exchange_wide(natoms, ndim);
    const size_t rest = wide ? 8 * xw_pub_words(natoms) : 2 * rec_lds_bytes(natoms, ndim);
    pl->status = status_pool().take();
    if (!pl->status || hipMalloc((void**)&pl->V, head * sizeof(double) + rest) != hipSuccess ||
        (wide && hipMemset(pl->V + head, 0xFF, rest) != hipSuccess)) {
        pimdb_xplan_destroy(pl);
        return PIMDB_E_HIP;
    }
    pl->Vb = pl->V + N + 1;
    pl->Shi = pl->Vb + N + 1;
    pl->Slo = pl->Shi + N;
    if (wide) pl->pub = (unsigned long long*)(pl->V + head);
    else pl->ws = pl->V + head;
    (void)hipStreamSynchronize(nullptr);   // the fills are done before a call on any stream
    *out = pl;
    return PIMDB_OK;
}

void pimdb_xplan_destroy(pimdb_xplan* pl) {
    if (!pl) return;
    (void)hipDeviceSynchronize();
    if (pl->V) (void)hipFree(pl->V);
    status_pool().give(pl->status);
    delete pl;
}

int pimdb_xplan_test_lost_wait(pimdb_xplan* pl) {
    if (!pl) return PIMDB_E_ARG;
    if (fill_published(pl->pub, xw_pub_words(pl->N), nullptr) != hipSuccess) return PIMDB_E_HIP;
    *(volatile int*)pl->status = LOST_WAIT;
    return xplan_finish(pl, nullptr);
}

int pimdb_xplan_forward(pimdb_xplan* pl, const double* x1, const double* xP, double* VB, double* V, double* Vb,
                        void* stream) {
    if (!pl || !x1 || !xP) return PIMDB_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    int rc = xplan_recursions(pl, x1, xP, s);
    if (rc) return rc;
    const int N = pl->N;
    if (VB && hipMemcpyAsync(VB, pl->V + N, sizeof(double), hipMemcpyDeviceToDevice, s) != hipSuccess) return PIMDB_E_HIP;
    if (V && hipMemcpyAsync(V, pl->V, (N + 1) * sizeof(double), hipMemcpyDeviceToDevice, s) != hipSuccess) return PIMDB_E_HIP;
    if (Vb && hipMemcpyAsync(Vb, pl->Vb, (N + 1) * sizeof(double), hipMemcpyDeviceToDevice, s) != hipSuccess) return PIMDB_E_HIP;
    return xplan_finish(pl, s);
}

int pimdb_xplan_vb_grad(pimdb_xplan* pl, const double* x1, const double* xP, double* grad, void* stream) {
    if (!pl || !x1 || !xP || !grad) return PIMDB_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    int rc = xplan_recursions(pl, x1, xP, s);
    if (rc) return rc;
    const int N = pl->N;
    dim3 grid((2 * N + 3) / 4), block(256);
    switch (pl->D) {
    case 1: hipLaunchKernelGGL(k_exchange_vb_grad<1>, grid, block, 0, s, N, pl->bt, pl->k, pl->pbc, pl->L, pl->Shi, pl->Slo, pl->V, pl->Vb, x1, xP, grad); break;
    case 2: hipLaunchKernelGGL(k_exchange_vb_grad<2>, grid, block, 0, s, N, pl->bt, pl->k, pl->pbc, pl->L, pl->Shi, pl->Slo, pl->V, pl->Vb, x1, xP, grad); break;
    default: hipLaunchKernelGGL(k_exchange_vb_grad<3>, grid, block, 0, s, N, pl->bt, pl->k, pl->pbc, pl->L, pl->Shi, pl->Slo, pl->V, pl->Vb, x1, xP, grad); break;
    }
    if (hipGetLastError() != hipSuccess) return PIMDB_E_HIP;
    return xplan_finish(pl, s);
}

long long pimdb_xplan_saved_doubles(const pimdb_xplan* pl) {
    return pl ? 2 * ((long long)pl->N + 1) + 2 * (long long)pl->N + 2 * (long long)pl->D * pl->N : 0;
}

int pimdb_xplan_forward_saved(pimdb_xplan* pl, const double* x1, long long s1n, long long s1d, const double* xP,
                              long long sPn, long long sPd, double* VB, double* saved, void* stream) {
    if (!pl || !x1 || !xP || !VB || !saved) return PIMDB_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    const int N = pl->N, D = pl->D;
    const Saved sv(saved, N);
    const BeadView v1{x1, s1d, s1n}, vP{xP, sPd, sPn};
    if (exchange_wide(N, D)) {
        launch_exchange_wide(D, N, pl->bt, pl->k, pl->pbc, pl->L, v1, vP, sv.V, sv.Vb, VB, sv.Shi, sv.Slo, sv.xc, pl->pub,
                             pl->status, s);
    } else {
        const dim3 grid((unsigned)((D * N + 255) / 256)), blk(256);
        switch (D) {
        case 1: hipLaunchKernelGGL(k_gather_beads<1>, grid, blk, 0, s, N, v1, vP, sv.xc); break;
        case 2: hipLaunchKernelGGL(k_gather_beads<2>, grid, blk, 0, s, N, v1, vP, sv.xc); break;
        default: hipLaunchKernelGGL(k_gather_beads<3>, grid, blk, 0, s, N, v1, vP, sv.xc); break;
        }
        launch_exchange_recursions(D, N, pl->bt, pl->k, pl->pbc, pl->L, sv.xc, sv.xc + (size_t)D * N, sv.V, sv.Vb, sv.Shi,
                                   sv.Slo, pl->pub, pl->ws, pl->status, s);
        if (hipMemcpyAsync(VB, sv.V + N, sizeof(double), hipMemcpyDeviceToDevice, s) != hipSuccess) return PIMDB_E_HIP;
    }
    if (hipGetLastError() != hipSuccess) return PIMDB_E_HIP;
    return xplan_finish(pl, s);
}

int pimdb_xplan_backward_saved(pimdb_xplan* pl, const double* saved, const double* scale, double* d1, double* dP,
                               void* stream) {
    if (!pl || !saved || !d1 || !dP) return PIMDB_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    const int N = pl->N;
    const Saved sv(const_cast<double*>(saved), N);
    dim3 grid((2 * N + 3) / 4), block(256);
    switch (pl->D) {
    case 1: hipLaunchKernelGGL(k_exchange_backward<1>, grid, block, 0, s, N, pl->bt, pl->k, pl->pbc, pl->L, sv.Shi, sv.Slo, sv.V, sv.Vb, sv.xc, scale, d1, dP); break;
    case 2: hipLaunchKernelGGL(k_exchange_backward<2>, grid, block, 0, s, N, pl->bt, pl->k, pl->pbc, pl->L, sv.Shi, sv.Slo, sv.V, sv.Vb, sv.xc, scale, d1, dP); break;
    default: hipLaunchKernelGGL(k_exchange_backward<3>, grid, block, 0, s, N, pl->bt, pl->k, pl->pbc, pl->L, sv.Shi, sv.Slo, sv.V, sv.Vb, sv.xc, scale, d1, dP); break;
    }
    return hipGetLastError() == hipSuccess ? PIMDB_OK : PIMDB_E_HIP;
}

}  // extern "C"
