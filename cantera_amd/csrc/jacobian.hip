// Batched analytic reactor Jacobians d(ydot)/dy of IdealGasConstPressureReactor
// states, the quantity Reactor::finiteDifferenceJacobian approximates
// (src/zeroD/Reactor.cpp:233-276 builds it column by column from eval()).
//
// Input layout as for the batched rates: T[n], P[n], Y[k*n + s] (species-major).
// Output: J[s*N*N + r*N + c], row-major per state, in the reactor's state order
// [m, T, Y_0..Y_{K-1}].  ydot does not depend on the reactor mass (dY/dt and
// dT/dt scale with V/m = 1/rho), so the state is taken with m = 1 kg and the m
// row and column are zero.
//
// For mechanisms that jac_tile.hip does not take (more than 62 species, or
// reactions that need the general code).
//
// One wavefront per state: the Jacobian assembly (two RHS evaluations, at the
// state and with T + dT, then the per-reaction derivatives), in LDS when it
// fits, else in the state's output block.  Two wavefronts per SIMD: the
// elementary passes go two side by side (three spill 19 registers).  One
// n-dodecane state 147 -> 100 us and 12,000 of them 4.59 -> 4.18 ms with the
// passes over the matrix in blocks (reactor_jacobian).
#include <hip/hip_runtime.h>

#include "bdf.hpp"
#include "wave_jac.hpp"

namespace cg {

namespace {

// kLdsJ: assemble J in LDS (FP64 LDS atomics for the per-reaction terms), then
// write it out with coalesced stores; otherwise assemble it in place in HBM
// (L2 atomics) -- used when N x N doubles do not fit next to the scratch.
// The assembly is inlined here, where the scratch and the matrix are known to
// be LDS: as an out-of-line function taking them through pointer arguments it
// used flat loads, stores and atomics for every access, and its callee-saved
// registers went to scratch memory.
// OT: element type of the output (double, or float for CG_FP32: the FP64
// assembly rounded once at the store, which halves the HBM bytes written).
template <int NS, bool kLdsJ, typename OT, bool kGen>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void jac_batch_kernel(DevMech m, long n, const double* __restrict__ T,
                                                       const double* __restrict__ P, const double* __restrict__ Y,
                                                       OT* __restrict__ J) {
    const int lane = lane_id();
    ScratchLayout L;
    int off = species_doubles(m.K);
    L.yb = off;  off += kWave * NS;
    L.F = off;   off += kWave * NS;
    L.Y0 = off;  off += kWave * NS;
    L.F0 = off;  off += kWave * NS;
    L.W2 = off;  off += 2 * m.K;
    const Scratch<kGen> S = scratch_view<kGen>(L, kernarg_mech());
    double* Jl = lds_base() + off;
    const int NN = m.N * m.N;
    const XcdStates xs(n);
    for (long st = xs.lo; st < xs.hi; st += xs.step) {
        const double Ts = T[st];
        const double Ps = uni(P[st]);
        double y[NS], f[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int i = lane + kWave * s;
            double v = 0.0;
            if (i < m.K) v = Y[static_cast<size_t>(i) * n + st];
            else if (i == m.K) v = Ts;
            else if (i == m.K + 1) v = 1.0;
            y[s] = v;
            if (i < m.N) S.yb[i] = v;
        }
        wave_sync();
#pragma unroll
        for (int s = 0; s < NS; s++) f[s] = 0.0;   // not read: the Jacobian takes its own base RHS
        OT* Jg = J + static_cast<size_t>(st) * NN;
        if constexpr (kLdsJ) {
            reactor_jacobian<NS, true, true, 2>(m, S, Ps, y, f, Jl);
            for (int e = lane; e < NN; e += kWave) Jg[e] = static_cast<OT>(Jl[e]);
            wave_sync();
        } else {
            static_assert(sizeof(OT) == sizeof(double), "in-place assembly needs a double output");
            reactor_jacobian<NS, true, true, 2>(m, S, Ps, y, f, Jg);
        }
    }
}

}  // namespace

// J goes to LDS for one state slot per lane (N <= 64); larger systems assemble in HBM
static bool jac_in_lds(int ns) { return ns == 1; }

size_t jac_lds_bytes(const DevMech& m, int ns) {
    size_t d = static_cast<size_t>(kWave) * ns * 4 + species_doubles(m.K) + 2 * m.K;
    if (jac_in_lds(ns)) d += static_cast<size_t>(m.N) * m.N;
    return d * sizeof(double);
}

// up to 62 species: only mechanisms with general reactions come here
const void* jac_kernel_ptr(const DevMech& m, int ns, bool f32) {
    if (ns == 1) return f32 ? reinterpret_cast<const void*>(&jac_batch_kernel<1, true, float, true>)
                            : reinterpret_cast<const void*>(&jac_batch_kernel<1, true, double, true>);
    if (ns != 2 || f32) return nullptr;
    return m.gen_end > 0 ? reinterpret_cast<const void*>(&jac_batch_kernel<2, false, double, true>)
                         : reinterpret_cast<const void*>(&jac_batch_kernel<2, false, double, false>);
}

hipError_t jac_launch(DevMech m, int ns, bool f32, long n, const double* T, const double* P, const double* Y, void* J,
                      int grid, size_t lds, hipStream_t stream) {
    const void* kernel = jac_kernel_ptr(m, ns, f32);
    if (!kernel) return hipErrorInvalidValue;
    void* args[] = {&m, &n, &T, &P, &Y, &J};
    return hipLaunchKernel(kernel, dim3(grid), dim3(64), args, lds, stream);
}

}  // namespace cg
