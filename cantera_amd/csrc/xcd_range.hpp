// Which of n work items a workgroup takes, for batches whose neighbouring items
// share cache lines.  Plain C++: the kernels include it through
// wave_kinetics.hpp, a host program can check it.
#pragma once

#ifdef __HIPCC__
#define CG_XCD_INLINE __host__ __device__ __forceinline__
#else
#define CG_XCD_INLINE inline
#endif

namespace cg {

// Workgroups are dispatched to the 8 XCDs round-robin (blockIdx % 8), and each
// XCD has its own L2: XCD x takes one contiguous range of the items, its
// workgroups stride through it, so the states sharing a line meet in one L2
// instead of eight.  The first n % 8 XCDs, which also have the extra workgroups
// of a grid that is no multiple of 8, take one item more: a grid of n workgroups
// has one item each.  (With the ranges cut at x n / 8, one workgroup of 513 took
// two: rates of 4,097 gri30 states 55 us, now 34; 30 n-dodecane Jacobians 280,
// now 150.)  Every item is visited exactly once for any grid of at least 8
// workgroups (plain grid-stride order otherwise).
struct XcdRange {
    long lo, hi, step;
    CG_XCD_INLINE XcdRange(long n, long G, long b) {
        if (G < 8) {
            lo = b; hi = n; step = G;
            return;
        }
        const long x = b % 8, q = n / 8, r = n % 8;
        lo = q * x + (x < r ? x : r) + b / 8;
        hi = q * (x + 1) + (x + 1 < r ? x + 1 : r);
        step = (G - x + 7) / 8;              // workgroups on XCD x
    }
};

}  // namespace cg
