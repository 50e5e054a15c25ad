// Linear-system policy of the mole-reactor integrator: the preconditioner
// M = I - gamma J on the fill pattern of sparse_lu.hpp, factored without
// pivoting in LDS (right-looking: per elimination step, the L column scaled by
// the pivot, then the step's independent updates a_ij -= l_ik u_kj spread
// over the lanes) and applied by the two triangular solves.  The factors
// persist in the reactor's global slot between calls, as the dense policies
// keep theirs.
#pragma once
#include "bdf.hpp"
#include "wave_kinetics.hpp"

namespace cg {

// the integrator kernel's one parameter in the kernel-argument segment
using KernargArgsSp = const __attribute__((address_space(4))) BdfArgs;
__device__ __forceinline__ KernargArgsSp* kernarg_bdf_args() {
    return (KernargArgsSp*)__builtin_amdgcn_kernarg_segment_ptr();
}

// GMRES scratch of the mole integrator kept after the factors in LDS
constexpr int kGmMaxl = 5;                      // SPGMR Krylov dimension (SUNDIALS default, no restarts)
// layout: Hessenberg (row i, column l at i * kGmMaxl + l), Givens rotations
// (c, s per column), then 8 counters (lin_iters, prec_solves, jt products,
// linear convergence failures, lin_rhs_evals)
constexpr int kGmH = 0;
constexpr int kGmRot = (kGmMaxl + 1) * kGmMaxl;
constexpr int kGmCnt = kGmRot + 2 * kGmMaxl;
constexpr int kGmDoubles = kGmCnt + 8;

template <int NS>
struct SolveVec {
    double v[NS];
};

// b <- M^-1 b, rows lane-distributed in internal order.  The vector stays in
// registers in elimination order, row i in lane i % 64, slot i / 64: a step is
// readlane -> FMA, and a step's factor entries, one per lane through the slot
// tables (the slot that holds 0 where the pattern has none), do not depend on
// it: table rows are loaded two blocks of columns ahead, their values one
// block ahead.  (Column by column with the vector in LDS, every step waited
// for its list bounds, indices, values and a barrier in turn.)
template <int NS>
__device__ __noinline__ SolveVec<NS> sparse_solve(KernargArgsSp* a, int off_lu, int off_x, int N, SolveVec<NS> b) {
    N = uni(N);
    const double* lu = lds_base() + uni(off_lu);
    double* x = lds_base() + uni(off_x);
    const int lane = lane_id();
    constexpr int W = kWave * NS, kB = 8;
    const int* __restrict__ iperm = a->sp.iperm;
    const int* __restrict__ diag = a->sp.diag;
    int ip[NS];
    double rd[NS], y[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int i = lane + kWave * s, ic = min(i, N - 1);
        ip[s] = iperm[ic];
        rd[s] = lu[diag[ic]];
    }
    wave_sync();
#pragma unroll
    for (int s = 0; s < NS; s++)
        if (lane + kWave * s < N) x[ip[s]] = b.v[s];
    wave_sync();
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int i = lane + kWave * s;
        rd[s] = (i < N) ? 1.0 / rd[s] : 1.0;
        y[s] = (i < N) ? x[i] : 0.0;
    }
    // slots of columns k0, k0 + dir, ... (clamped into the table)
    auto slots = [&](const unsigned short* __restrict__ tab, int k0, int dir, unsigned (&ix)[kB][NS]) {
#pragma unroll
        for (int c = 0; c < kB; c++) {
            const unsigned short* row = tab + static_cast<size_t>(min(max(k0 + dir * c, 0), N - 1)) * W + lane;
#pragma unroll
            for (int s = 0; s < NS; s++) ix[c][s] = row[kWave * s];
        }
    };
    auto values = [&](const unsigned (&ix)[kB][NS], double (&v)[kB][NS]) {
#pragma unroll
        for (int c = 0; c < kB; c++)
#pragma unroll
            for (int s = 0; s < NS; s++) v[c][s] = lu[ix[c][s]];
    };
    const unsigned short* __restrict__ fwd = a->sp.fwd;
    const unsigned short* __restrict__ bwd = a->sp.bwd;
#pragma unroll
    for (int t = 0; t < NS; t++) {
        const int kend = min(N, kWave * (t + 1));
        if (kWave * t < kend) {
            unsigned ix[kB][NS];
            double v[kB][NS];
            slots(fwd, kWave * t, 1, ix);
            values(ix, v);
            slots(fwd, kWave * t + kB, 1, ix);
            for (int k0 = kWave * t; k0 < kend; k0 += kB) {
                double nv[kB][NS];
                values(ix, nv);
                slots(fwd, k0 + 2 * kB, 1, ix);
#pragma unroll
                for (int c = 0; c < kB; c++)
                    if (k0 + c < kend) {
                        const double yk = readlane_f64(y[t], k0 + c - kWave * t);
#pragma unroll
                        for (int s = t; s < NS; s++) y[s] -= v[c][s] * yk;
                    }
#pragma unroll
                for (int c = 0; c < kB; c++)
#pragma unroll
                    for (int s = 0; s < NS; s++) v[c][s] = nv[c][s];
            }
        }
    }
#pragma unroll
    for (int t = NS - 1; t >= 0; t--) {
        const int klo = kWave * t, khi = min(N, kWave * (t + 1)) - 1;
        if (khi >= klo) {
            unsigned ix[kB][NS];
            double v[kB][NS];
            slots(bwd, khi, -1, ix);
            values(ix, v);
            slots(bwd, khi - kB, -1, ix);
            for (int k0 = khi; k0 >= klo; k0 -= kB) {
                double nv[kB][NS];
                values(ix, nv);
                slots(bwd, k0 - 2 * kB, -1, ix);
#pragma unroll
                for (int c = 0; c < kB; c++)
                    if (k0 - c >= klo) {
                        const double xk = readlane_f64(y[t] * rd[t], k0 - c - klo);
#pragma unroll
                        for (int s = 0; s <= t; s++) y[s] -= v[c][s] * xk;
                    }
#pragma unroll
                for (int c = 0; c < kB; c++)
#pragma unroll
                    for (int s = 0; s < NS; s++) v[c][s] = nv[c][s];
            }
        }
    }
#pragma unroll
    for (int s = 0; s < NS; s++)
        if (lane + kWave * s < N) x[lane + kWave * s] = y[s] * rd[s];
    wave_sync();
#pragma unroll
    for (int s = 0; s < NS; s++) b.v[s] = (lane + kWave * s < N) ? x[ip[s]] : 0.0;
    wave_sync();
    return b;
}

// M factored in place; 0 on a zero pivot.  Step k scales the L column by the
// pivot, then its updates, which are independent, go kU per lane: 8 bytes of
// schedule each, loaded one batch ahead across step boundaries (the lists of
// consecutive steps follow each other), as are the next column's slots.
template <int kU>
__device__ __noinline__ int sparse_factor(KernargArgsSp* a, int off_lu, int N) {
    N = uni(N);
    double* lu = lds_base() + uni(off_lu);
    const int lane = lane_id();
    const int* __restrict__ lptr = a->sp.lptr;
    const int* __restrict__ lslot = a->sp.lslot;
    const int* __restrict__ optr = a->sp.optr;
    const uint2* __restrict__ ops = reinterpret_cast<const uint2*>(a->sp.ops);
    const int* __restrict__ diag = a->sp.diag;
    const int nops = optr[N], nl = lptr[N];
    auto batch = [&](int base, uint2 (&u)[kU]) {
#pragma unroll
        for (int b = 0; b < kU; b++) u[b] = ops[max(min(base + lane + kWave * b, nops - 1), 0)];
    };
    uint2 u[kU];
    batch(0, u);
    int ls = nl > 0 ? lslot[min(lane, nl - 1)] : 0;
    int l0 = 0, o0 = 0;
    for (int k = 0; k < N; k++) {
        const int l1 = lptr[k + 1], o1 = optr[k + 1], dk = diag[k];
        if (l0 == l1) continue;                    // nothing below the pivot
        const double piv = lu[dk];
        if (piv == 0.0) return 0;
        for (int t = l0 + lane; t < l1; t += kWave) {
            const int q = (t < l0 + kWave) ? ls : lslot[t];
            lu[q] = lu[q] / piv;
        }
        ls = lslot[min(l1 + lane, nl - 1)];
        wave_sync();
        for (int base = o0; base < o1; base += kWave * kU) {
            uint2 nu[kU];
            batch(min(base + kWave * kU, o1), nu);
            double c[kU], l[kU], r[kU];
#pragma unroll
            for (int b = 0; b < kU; b++) {
                c[b] = lu[u[b].x & 0xffffu];
                l[b] = lu[u[b].x >> 16];
                r[b] = lu[u[b].y];
            }
#pragma unroll
            for (int b = 0; b < kU; b++)
                if (base + lane + kWave * b < o1) lu[u[b].x & 0xffffu] = c[b] - l[b] * r[b];
#pragma unroll
            for (int b = 0; b < kU; b++) u[b] = nu[b];
        }
        wave_sync();
        l0 = l1;
        o0 = o1;
    }
    return lu[diag[N - 1]] != 0.0 ? 1 : 0;
}

template <int NS>
struct SparseLdsLinSys {
    double* lu;   // nnz values, then 0 (the slot of entries that the pattern lacks)
    double* x;    // kWave * NS: solve workspace
    double* gm;   // kGmDoubles: Hessenberg, rotations, least-squares rhs, counters

    __device__ __forceinline__ static int nnz() { return kernarg_bdf_args()->sp.nnz; }
    __host__ __device__ __forceinline__ static int lu_doubles(int nnz_) { return (nnz_ + 2) & ~1; }
    __host__ __device__ __forceinline__ static size_t lds_doubles(int nnz_, int ns) {
        return static_cast<size_t>(lu_doubles(nnz_)) + static_cast<size_t>(kWave) * ns + kGmDoubles;
    }
    __device__ __forceinline__ void init(double* base, int) {
        lu = base;
        x = base + lu_doubles(nnz());
        gm = x + kWave * NS;
        if (lane_id() == 0) lu[nnz()] = 0.0;
        wave_sync();
    }
    __device__ __forceinline__ void bind(double*, int*) {}
    // blocks of 8 values per lane, their loads in flight together
    __device__ __forceinline__ void restore(const double* __restrict__ save, const int*, int) {
        const int nz = nnz();
        int p = lane_id();
        for (; p + 7 * kWave < nz; p += 8 * kWave) {
            double t[8];
#pragma unroll
            for (int b = 0; b < 8; b++) t[b] = save[p + kWave * b];
#pragma unroll
            for (int b = 0; b < 8; b++) lu[p + kWave * b] = t[b];
        }
        for (; p < nz; p += kWave) lu[p] = save[p];
        wave_sync();
    }
    __device__ __forceinline__ void save(double* save, int*, int) {
        const int nz = nnz();
        for (int p = lane_id(); p < nz; p += kWave) save[p] = lu[p];
    }
    // M = I - gamma J (AdaptivePreconditioner: m_identity - m_gamma * J)
    __device__ __forceinline__ void form(const double* __restrict__ J, int N, double gamma) {
        KernargArgsSp* a = kernarg_bdf_args();
        const int nz = a->sp.nnz;
        const int lane = lane_id();
        wave_sync();
        int p = lane;
        for (; p + 7 * kWave < nz; p += 8 * kWave) {
            double t[8];
#pragma unroll
            for (int b = 0; b < 8; b++) t[b] = J[p + kWave * b];
#pragma unroll
            for (int b = 0; b < 8; b++) lu[p + kWave * b] = -gamma * t[b];
        }
        for (; p < nz; p += kWave) lu[p] = -gamma * J[p];
        wave_sync();
        for (int k = lane; k < N; k += kWave) lu[a->sp.diag[k]] += 1.0;
        wave_sync();
    }
    __device__ __forceinline__ int off_lu() const { return static_cast<int>(lu - lds_base()); }
    // false on a zero pivot
    __device__ __forceinline__ bool factor(int N) { return sparse_factor<4>(kernarg_bdf_args(), off_lu(), N) != 0; }
    // b <- M^{-1} b (lane-distributed, internal order)
    __device__ __forceinline__ void solve(double (&b)[NS], int N) {
        SolveVec<NS> t;
#pragma unroll
        for (int s = 0; s < NS; s++) t.v[s] = b[s];
        t = sparse_solve<NS>(kernarg_bdf_args(), off_lu(), static_cast<int>(x - lds_base()), N, t);
#pragma unroll
        for (int s = 0; s < NS; s++) b[s] = t.v[s];
    }
};

}  // namespace cg
