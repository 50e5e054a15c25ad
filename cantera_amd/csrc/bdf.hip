// Integrator dispatch: picks the kernel variant for the mechanism size.
#include "bdf_integrator.hpp"

namespace cg {

const void* bdf_kernel_r16(bool, bool, bool);
const void* bdf_kernel_r32(bool, bool, bool);
const void* bdf_kernel_lr56(bool, bool, bool);
const void* bdf_kernel_lr64(bool, bool, bool);
const void* bdf_kernel_l2(bool, bool, bool);
const void* bdf_kernel_gr56(bool, bool, bool);
const void* bdf_kernel_gr64(bool, bool, bool);

namespace {
__global__ void reset_queue_kernel(int* q) { *q = 0; }
}  // namespace

// 16, 32: iteration matrix in registers (one row per lane).
// 56, 64: iteration matrix kept in LDS, factored and solved in registers.
// 2: iteration matrix in LDS, state spread over 2 slots per lane.
int bdf_variant(int N) {
    if (N <= 16) return 16;
    if (N <= 32) return 32;
    if (N <= 56) return 56;
    if (N <= 64) return 64;
    if (N <= 128) return 2;
    return -1;
}

// register policies keep 64 reciprocal pivots after the factors
size_t bdf_lu_elems(int N, int ld) {
    const int v = bdf_variant(N);
    if (v == 56 || v == 64) return static_cast<size_t>(v + 1) * kWave;
    if (v == 16 || v == 32) return static_cast<size_t>(N) * ld + kWave;
    return static_cast<size_t>(N) * ld;
}

size_t bdf_lds_bytes(const DevMech& m, int ld, bool fp32, bool global) {
    const int v = bdf_variant(m.N);
    const int ns = (v == 2) ? 2 : 1;
    size_t bytes = bdf_scratch_doubles(m.K, ns) * sizeof(double);
    if (v == 2) {
        bytes += static_cast<size_t>(kWave) * ns * (sizeof(double) + sizeof(int));
        bytes += static_cast<size_t>(m.N) * ld * (fp32 ? 4 : 8);
    } else if ((v == 56 || v == 64) && !global) {
        bytes += static_cast<size_t>(v + 1) * kWave * (fp32 ? 4 : 8) + 2 * kWave * sizeof(int);
    }
    return bytes;
}

const void* bdf_kernel_ptr(const DevMech& m, bool fp32, bool global, bool sens) {
    const bool gen = m.gen_end > 0;
    switch (bdf_variant(m.N)) {
        case 16: return bdf_kernel_r16(fp32, sens, gen);
        case 32: return bdf_kernel_r32(fp32, sens, gen);
        case 56: return global ? bdf_kernel_gr56(fp32, sens, gen) : bdf_kernel_lr56(fp32, sens, gen);
        case 64: return global ? bdf_kernel_gr64(fp32, sens, gen) : bdf_kernel_lr64(fp32, sens, gen);
        case 2: return bdf_kernel_l2(fp32, sens, gen);
        default: return nullptr;
    }
}

hipError_t bdf_launch(BdfArgs a, bool fp32, bool global, int grid, size_t lds, hipStream_t stream) {
    const void* kernel = bdf_kernel_ptr(a.mech, fp32, global, a.nsens > 0);
    if (!kernel) return hipErrorInvalidValue;
    hipLaunchKernelGGL(reset_queue_kernel, dim3(1), dim3(1), 0, stream, a.queue);
    void* args[] = {&a};
    return hipLaunchKernel(kernel, dim3(grid), dim3(64), args, lds, stream);
}

}  // namespace cg
