// Integrator kernels of the mole-based reactor with the sparse preconditioner
// and GMRES (IdealGasConstPressureMoleReactor; N = K + 1 <= 128).
#include "bdf_integrator.hpp"

namespace cg {

namespace {
__global__ void reset_mole_queue(int* q) { *q = 0; }
}  // namespace

template <int NS, bool kGen>
__global__ __launch_bounds__(64) void bdf_advance_mole(BdfArgs a) {
    bdf_advance_body<NS, SparseLdsLinSys<NS>, double, kGen, false, true>(a);
}

int bdf_mole_ns(int N) { return N <= 64 ? 1 : (N <= 128 ? 2 : (N <= 256 ? 4 : -1)); }

size_t bdf_mole_lds_bytes(const DevMech& m, int N, int nnz) {
    const int ns = bdf_mole_ns(N);
    return (bdf_scratch_doubles(m.K, ns, true) + SparseLdsLinSys<1>::lds_doubles(nnz, ns)) * sizeof(double);
}

template <bool kGen>
static const void* mole_kernel(int N) {
    switch (bdf_mole_ns(N)) {
        case 1: return reinterpret_cast<const void*>(&bdf_advance_mole<1, kGen>);
        case 2: return reinterpret_cast<const void*>(&bdf_advance_mole<2, kGen>);
        case 4: return reinterpret_cast<const void*>(&bdf_advance_mole<4, kGen>);
        default: return nullptr;
    }
}

const void* bdf_mole_kernel_ptr(const DevMech& m, int N) {
    return m.gen_end > 0 ? mole_kernel<true>(N) : mole_kernel<false>(N);
}

hipError_t bdf_mole_launch(BdfArgs a, int grid, size_t lds, hipStream_t stream) {
    const void* kernel = bdf_mole_kernel_ptr(a.mech, a.neq_norm);
    if (!kernel) return hipErrorInvalidValue;
    hipLaunchKernelGGL(reset_mole_queue, dim3(1), dim3(1), 0, stream, a.queue);
    void* args[] = {&a};
    return hipLaunchKernel(kernel, dim3(grid), dim3(64), args, lds, stream);
}

}  // namespace cg
