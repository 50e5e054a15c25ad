// Batched net production rates (Kinetics::getNetProductionRates,
// src/kinetics/Kinetics.cpp:447-457) over many independent states.
//
// Layout: species-major SoA in HBM, Y[k*n + s] and wdot[k*n + s].  One
// wavefront evaluates one state at a time (grid-stride over states): lane k
// loads Y_k, the wavefront runs the species, reaction and production passes
// with its scratch in LDS, and lane k stores wdot_k.  Consecutive states go to
// neighbouring wavefronts, so the 64-byte lines of Y and wdot (8 states of one
// species) are shared through L2.  The LDS scratch is small (a few KB), so many
// wavefronts per CU hide the latency of the table loads and transcendentals.
// kF32: the rate constants' transcendentals in FP32 (see eval_reaction).
#include <hip/hip_runtime.h>

#include "bdf.hpp"
#include "wave_kinetics.hpp"

namespace cg {

// From this many states on, several states per wavefront.  Below, the tiles
// leave SIMDs empty and one state per wavefront ends sooner (us, one state /
// tiles: gri30 2,048 states 21 / 34, 4,095 28 / 34, 6,144 35 / 36; n-dodecane
// 2,048 26 / 29, 4,095 38 / 31).  A mechanism of one pass of reactions has
// nothing to gain from 64 lanes a state and is past that point once two
// wavefronts per SIMD, all that the general code's registers allow, are full
// (h2o2 2,048 14 / 15, 3,072 16 / 15; 7 pressure-dependent reactions 2,048
// 20 / 19, 3,072 28 / 19).
constexpr long kRatesWideMin = 4096, kRatesWideMinSmall = 2049;
constexpr int kRatesSmall = 64;   // reactions
// LDS of a wavefront with 8 states: 8 wavefronts share a CU (two per SIMD, as
// their registers allow); larger mechanisms take 4 states
constexpr size_t kRatesWideLds = 160 * 1024 / 8;

namespace {

// At most 168 VGPRs, so that three wavefronts share a SIMD (latency-bound
// kernel; without the bound the allocator settles at 169 for NS = 1).  The
// general code would spill 30 of them: two wavefronts there (7
// pressure-dependent reactions, 2,048 states: 24 -> 20 us).
template <int NS, bool kF32, bool kGen>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kGen ? 2 : 3))) void rates_kernel(
    DevMech m, long n, const double* __restrict__ T, const double* __restrict__ P, const double* __restrict__ Y,
    double* __restrict__ wdot) {
    const int lane = lane_id();
    Scratch<kGen> S{};
    bind_species(S, kernarg_mech());
    const XcdStates xs(n);
    for (long st = xs.lo; st < xs.hi; st += xs.step) {
        const double Ts = uni(T[st]);
        const double Ps = uni(P[st]);
        double yk[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int k = lane + kWave * s;
            yk[s] = (k < m.K) ? Y[static_cast<size_t>(k) * n + st] : 0.0;
        }
        GasState g;
        SpeciesRegs<NS> sr;
        species_pass<NS, true>(m, S, Ts, Ps, yk, g, sr);
        production_rates<NS, kF32, false, 2>(m, S, g, sr);
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int k = lane + kWave * s;
            if (k < m.K) wdot[static_cast<size_t>(k) * n + st] = sr.wdot[s];
        }
        wave_sync();
    }
}

// S states per wavefront, 64 / S lanes per state (lane = s + S j, j the lane's
// reaction of a pass), for batches that fill the GPU.
//
// Evaluated one state per wavefront, 64 lanes add their rates of progress to
// the same 53 accumulators (gri30) at once: radicals occur in a third of the
// reactions, and LDS adds to one address take turns.  The kernel above is bound
// by that (2.6k cycles of a CU per gri30 state), and its falloff code runs for
// 64 lanes to serve 29.  With S = 8 only 8 lanes share an accumulator, 50
// falloff and three-body reactions take 7 passes of 8 states instead of one of
// each, and a tile reads and writes whole 64-byte lines.  1,048,576 gri30
// states: 4.50 -> 2.44 ms (FP64 VALU at 62% of its issue rate: 872
// instructions a state); S = 16 leaves room for 7 wavefronts per CU (3.02 ms),
// S = 4 has more lanes per accumulator (2.83 ms).  30,011 n-dodecane states,
// FP32 constants: 213 -> 138 us with S = 4, 141 us with S = 8.  1/W_bar and [M]
// are summed in the reference's order, as in the kernel above.
template <int S, bool kF32>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void rates_wide_kernel(
    DevMech m, long n, const double* __restrict__ T, const double* __restrict__ P, const double* __restrict__ Y,
    double* __restrict__ wdot) {
    constexpr int G = 64 / S;
    const int lane = lane_id(), s = lane % S, j = lane / S;
    const int rows = m.K + kDummyWide;
    LaneView<S> lv;
    lv.pair0 = 16u * s;
    lv.wd = lds_base() + 2 * S * rows + s;
    const SpeciesColumn<S> C{lds_base() + 2 * s}, MU{lds_base() + 2 * s + 1};
    const long tiles = (n + S - 1) / S;
    for (int k = m.K + j; k < rows; k += G) {   // sentinel rows
        C[k] = 1.0;
        MU[k] = 0.0;
    }
    const XcdStates xs(tiles);
    for (long tile = xs.lo; tile < xs.hi; tile += xs.step) {
        const long st = tile * S + s, sc = min(st, n - 1);   // a ragged tile's spare lanes repeat the last state
        GasState g;
        g.T = T[sc];
        const double Ps = P[sc];
        for (int k = j; k < m.K; k += G) {
            C[k] = Y[static_cast<size_t>(k) * n + sc] * m.rmw[k];
            lv.wd[S * k] = 0.0;
        }
        wave_sync();
        double sum = 0.0;
        {
            int k = 0;
            for (; k + 8 <= m.K; k += 8) {
                double t[8];
#pragma unroll
                for (int b = 0; b < 8; b++) t[b] = C[k + b];
#pragma unroll
                for (int b = 0; b < 8; b++) sum += t[b];
            }
            for (; k < m.K; k++) sum += C[k];
        }
        wave_sync();
        // as species_pass
        g.RT = g.T * kGasConstant;
        g.recipT = 1.0 / g.T;
        g.mmw = 1.0 / sum;
        g.dens = Ps * g.mmw / g.RT;
        g.ctot = g.dens / g.mmw;
        g.pressure = kGasConstant * g.ctot * g.T;
        // ln T, ln(P/RT), ln(P/Pref): one each for the first three lanes of a state
        const double lg = log(j == 0 ? g.T : (j == 1 ? g.ctot : g.pressure * m.rpref));
        g.logT = __shfl(lg, s);
        g.logC0 = __shfl(lg, s + S);
        const double lnp = __shfl(lg, s + 2 * S);
        double tt[6];
        tt[0] = g.T;
        tt[1] = g.T * g.T;
        tt[2] = tt[1] * g.T;
        tt[3] = tt[2] * g.T;
        tt[4] = g.recipT;
        tt[5] = g.logT;
        for (int k = j; k < m.K; k += G) {
            double cp, h, sR, g0;
            nasa7(m.nasa + 16 * k, g.T, tt, cp, h, sR, g0);
            C[k] = C[k] * g.dens;
            MU[k] = g0 + lnp;
        }
        wave_sync();
        int q = 0;
        for (; q < m.n_gen; q += G) {   // non-standard reactions
            const int p = q + j;
            if (p >= m.I) continue;
            RxnRegs x;
            load_rxn(m, p, x);
            double kpd = 0.0;
            if (x.flags & 64) kpd = plog_rate(m.pdd + x.fo, log(g.pressure), g.logT, g.recipT);
            else if (x.flags & 128) kpd = cheb_rate(m.pdd + x.fo, log10(g.pressure), g.recipT);
            RxnVals v;
            eval_reaction<kF32, S>(m, p, g, C, MU, x, kpd, v);
            const double r = v.ropf - v.ropr;
            const double* gs = (x.gen >= 0) ? m.gend + 12 * x.gen : m.gend;
            const bool rgen = x.flags & 8, pgen = x.flags & 16;
#pragma unroll
            for (int e = 0; e < kMaxSide; e++)
                if (e < x.nr) atomicAdd(&lv.wd[S * x.rk[e]], -(rgen ? gs[4 + e] : 1.0) * r);
#pragma unroll
            for (int e = 0; e < kMaxSide; e++)
                if (e < x.np) atomicAdd(&lv.wd[S * x.pk[e]], (pgen ? gs[8 + e] : 1.0) * r);
        }
        standard_passes<3, kF32, false, S>(m, m.rsw, lv, C, g, j, q, m.n_nonplain, m.I, -1, 1.0);
        wave_sync();
        if (st < n)
            for (int k = j; k < m.K; k += G) wdot[static_cast<size_t>(k) * n + st] = lv.wd[S * k];
        wave_sync();
    }
}

// Net production rates at the output states of a reactor batch (one record
// per reactor: the interpolated state [Y, T, m] after the 6 Nordsieck columns,
// then the control block with P, or V for a constant-volume reactor).
template <int NS, bool kGen>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kGen ? 2 : 3))) void reactor_rates_kernel(
    DevMech m, long n, const double* __restrict__ rec, size_t stride, int cv, double* __restrict__ wdot) {
    const int lane = lane_id();
    Scratch<kGen> S{};
    bind_species(S, kernarg_mech());
    constexpr int NP = kWave * NS;
    const XcdStates xs(n);
    for (long st = xs.lo; st < xs.hi; st += xs.step) {
        const double* rr = rec + static_cast<size_t>(st) * stride;
        const double Ts = uni(rr[6 * NP + m.K]);
        const double mass = uni(rr[6 * NP + m.K + 1]);
        const double pv = uni(rr[7 * NP + C_P]);
        double yk[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int k = lane + kWave * s;
            yk[s] = (k < m.K) ? rr[6 * NP + k] : 0.0;
        }
        GasState g;
        SpeciesRegs<NS> sr;
        species_pass<NS, true>(m, S, Ts, cv ? 0.0 : pv, yk, g, sr, cv ? mass / pv : 0.0);
        production_rates<NS, false, false, 2>(m, S, g, sr);
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int k = lane + kWave * s;
            if (k < m.K) wdot[static_cast<size_t>(k) * n + st] = sr.wdot[s];
        }
        wave_sync();
    }
}

}  // namespace

template <bool kGen>
static const void* reactor_rates_kernel_of(int ns) {
    if (ns == 1) return reinterpret_cast<const void*>(&reactor_rates_kernel<1, kGen>);
    if (ns == 2) return reinterpret_cast<const void*>(&reactor_rates_kernel<2, kGen>);
    return nullptr;
}

const void* reactor_rates_kernel_ptr(const DevMech& m, int ns) {
    return m.gen_end > 0 ? reactor_rates_kernel_of<true>(ns) : reactor_rates_kernel_of<false>(ns);
}

hipError_t reactor_rates_launch(DevMech m, int ns, long n, const double* rec, size_t stride, int cv, double* wdot,
                                int grid, size_t lds, hipStream_t stream) {
    const void* kernel = reactor_rates_kernel_ptr(m, ns);
    if (!kernel) return hipErrorInvalidValue;
    void* args[] = {&m, &n, &rec, &stride, &cv, &wdot};
    return hipLaunchKernel(kernel, dim3(grid), dim3(64), args, lds, stream);
}

// state slots per lane: 1, 2, or 4 for 128 < K + 2 <= 256
template <bool kF32, bool kGen>
static const void* rates_kernel_of(int ns) {
    if (ns == 1) return reinterpret_cast<const void*>(&rates_kernel<1, kF32, kGen>);
    return ns == 2 ? reinterpret_cast<const void*>(&rates_kernel<2, kF32, kGen>)
                   : reinterpret_cast<const void*>(&rates_kernel<4, kF32, kGen>);
}

template <bool kF32>
static const void* rates_kernel_of(bool gen, int ns, int wide) {
    if (wide == 8) return reinterpret_cast<const void*>(&rates_wide_kernel<8, kF32>);
    if (wide == 4) return reinterpret_cast<const void*>(&rates_wide_kernel<4, kF32>);
    return gen ? rates_kernel_of<kF32, true>(ns) : rates_kernel_of<kF32, false>(ns);
}

size_t reactor_rates_lds_bytes(const DevMech& m) { return static_cast<size_t>(species_doubles(m.K)) * sizeof(double); }

static size_t wide_lds(int K, int S) { return static_cast<size_t>(24) * S * (K + kDummyWide); }

RatesPlan rates_plan(const DevMech& m, int ns, bool f32, long n) {
    RatesPlan p{};
    if (n >= (m.I <= kRatesSmall ? kRatesWideMinSmall : kRatesWideMin))
        p.wide = wide_lds(m.K, 8) <= kRatesWideLds ? 8 : 4;
    if (p.wide) {
        p.lds = wide_lds(m.K, p.wide);
        p.items = (n + p.wide - 1) / p.wide;
    } else {
        p.lds = reactor_rates_lds_bytes(m);
        p.items = n;
    }
    const bool gen = m.gen_end > 0;
    p.kernel = f32 ? rates_kernel_of<true>(gen, ns, p.wide) : rates_kernel_of<false>(gen, ns, p.wide);
    return p;
}

hipError_t rates_launch(const RatesPlan& p, DevMech m, long n, const double* T, const double* P, const double* Y,
                        double* wdot, int grid, hipStream_t stream) {
    void* args[] = {&m, &n, &T, &P, &Y, &wdot};
    return hipLaunchKernel(p.kernel, dim3(grid), dim3(64), args, p.lds, stream);
}

}  // namespace cg
