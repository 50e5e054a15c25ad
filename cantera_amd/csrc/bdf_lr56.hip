// Integrator kernels with the iteration matrix kept in LDS, factored and solved in registers (32 < N <= 56).
#include "bdf_integrator.hpp"

namespace cg {

template <typename MT, bool kGen, bool kSens>
__global__ __launch_bounds__(64) void bdf_advance_lr56(BdfArgs a) {
    bdf_advance_body<1, LdsRegLinSys<56, MT>, MT, kGen, kSens>(a);
}

template <bool kGen>
static const void* kernel(bool fp32, bool sens) {
    if (sens) return reinterpret_cast<const void*>(&bdf_advance_lr56<double, kGen, true>);
    return fp32 ? reinterpret_cast<const void*>(&bdf_advance_lr56<float, kGen, false>)
                : reinterpret_cast<const void*>(&bdf_advance_lr56<double, kGen, false>);
}

// sens: the FP64 kernel that also integrates sensitivities; gen: the mechanism
// has reactions of the general code
const void* bdf_kernel_lr56(bool fp32, bool sens, bool gen) {
    return gen ? kernel<true>(fp32, sens) : kernel<false>(fp32, sens);
}

}  // namespace cg
