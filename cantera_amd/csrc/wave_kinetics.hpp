// Wavefront-cooperative gas kinetics for one state at a time: lanes over
// species for thermo and concentrations, lanes over reactions for rate
// constants, equilibrium constants and rates of progress, which they add to the
// species' net production rates in LDS.  Shared by the batched rate kernels and
// the per-reactor BDF integrator.
//
// Reference algorithm (file:line in the Cantera sources):
//   BulkKinetics::updateROP            src/kinetics/BulkKinetics.cpp:457-545
//   Kinetics::getNetProductionRates    src/kinetics/Kinetics.cpp:447-457
//   StoichManagerN multiply rules      include/cantera/kinetics/StoichManager.h:147-366
//   ThirdBodyCalc::update/multiply     include/cantera/kinetics/ThirdBodyCalc.h:75-91
//   ArrheniusRate::evalFromStruct      include/cantera/kinetics/Arrhenius.h:196-198
//   FalloffRate::evalFromStruct        include/cantera/kinetics/Falloff.h:154-176
//   TroeRate::updateTemp / F           src/kinetics/Falloff.cpp:283-300
//   NasaPoly1/NasaPoly2                include/cantera/thermo/NasaPoly1.h:83-122, NasaPoly2.h:105-111
//   IdealGasConstPressureReactor::eval src/zeroD/IdealGasConstPressureReactor.cpp:46-110
//
// Internal state order on the device is [Y_0 .. Y_{K-1}, T, m]: component i
// lives in lane i % 64, register slot i / 64, so species k is owned by the
// lane that also owns Y_k (no cross-lane moves between thermo and state).
#pragma once
#include <hip/hip_runtime.h>

#include "mech.hpp"
#include "xcd_range.hpp"

namespace cg {

constexpr double kGasConstant = 6.02214076e26 * 1.380649e-23;  // ct_defs.h:84-123
constexpr double kSmallNumber = 1e-300;
constexpr double kBigNumber = 1e300;
constexpr int kWave = 64;

__device__ __forceinline__ int lane_id() { return static_cast<int>(threadIdx.x) & (kWave - 1); }

// 64-bit DPP move (both halves) with the given control; all lanes valid for
// quad_perm and row_ror controls.
template <int kCtrl>
__device__ __forceinline__ double dpp_f64(double x) {
    const long long u = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(u & 0xffffffffll), kCtrl, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(u >> 32), kCtrl, 0xf, 0xf, false);
    return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned int>(lo));
}

// The value unchanged, but opaque to the optimiser: it cannot trace it back to
// the load that produced it (used to stop selects between array elements from
// being turned into a load through a selected pointer).
__device__ __forceinline__ double opaque(double x) {
    asm("" : "+v"(x));
    return x;
}

__device__ __forceinline__ double readlane_f64(double v, int l) {
    const long long x = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane(static_cast<int>(x & 0xffffffffll), l);
    const int hi = __builtin_amdgcn_readlane(static_cast<int>(x >> 32), l);
    return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned int>(lo));
}

// 64-bit DPP move (both halves) with the given control.
template <int kCtrl>
__device__ __forceinline__ unsigned long long dpp_u64(unsigned long long x) {
    const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(x & 0xffffffffull), kCtrl, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(x >> 32), kCtrl, 0xf, 0xf, false);
    return (static_cast<unsigned long long>(static_cast<unsigned int>(hi)) << 32) | static_cast<unsigned int>(lo);
}

__device__ __forceinline__ unsigned long long readlane_u64(unsigned long long x, int l) {
    const unsigned int lo = __builtin_amdgcn_readlane(static_cast<int>(x & 0xffffffffull), l);
    const unsigned int hi = __builtin_amdgcn_readlane(static_cast<int>(x >> 32), l);
    return (static_cast<unsigned long long>(hi) << 32) | lo;
}

// Wavefront max of an unsigned 64-bit key: within each row of 16 lanes by
// quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_ror:4, row_ror:8; then over
// the four rows through lanes 0, 16, 32, 48.  Returns the (uniform) maximum.
__device__ __forceinline__ unsigned long long wave_max_u64(unsigned long long x) {
    unsigned long long y;
    y = dpp_u64<0xB1>(x);  x = y > x ? y : x;
    y = dpp_u64<0x4E>(x);  x = y > x ? y : x;
    y = dpp_u64<0x124>(x); x = y > x ? y : x;
    y = dpp_u64<0x128>(x); x = y > x ? y : x;
    unsigned long long m = readlane_u64(x, 0);
    const unsigned long long m1 = readlane_u64(x, 16), m2 = readlane_u64(x, 32), m3 = readlane_u64(x, 48);
    m = m1 > m ? m1 : m;
    m = m2 > m ? m2 : m;
    m = m3 > m ? m3 : m;
    return m;
}

// Wavefront sum, the same value in every lane: within each row of 16 lanes by
// DPP (quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_ror:4, row_ror:8), then the
// four row sums through lanes 0, 16, 32, 48 (fixed order, so every lane and
// every call with the same inputs gives the same result).
__device__ __forceinline__ double wave_sum(double v) {
    v += dpp_f64<0xB1>(v);
    v += dpp_f64<0x4E>(v);
    v += dpp_f64<0x124>(v);
    v += dpp_f64<0x128>(v);
    return (readlane_f64(v, 0) + readlane_f64(v, 16)) + (readlane_f64(v, 32) + readlane_f64(v, 48));
}
__device__ __forceinline__ float wave_sumf(float v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}
__device__ __forceinline__ double wave_max(double v) {
    v = fmax(v, dpp_f64<0xB1>(v));
    v = fmax(v, dpp_f64<0x4E>(v));
    v = fmax(v, dpp_f64<0x124>(v));
    v = fmax(v, dpp_f64<0x128>(v));
    return fmax(fmax(readlane_f64(v, 0), readlane_f64(v, 16)), fmax(readlane_f64(v, 32), readlane_f64(v, 48)));
}

// Order LDS traffic between the lanes of one wavefront.  Every kernel here
// runs one wavefront per workgroup, so the workgroup barrier is a cheap,
// compiler-visible ordering point (a wavefront-scope fence alone does not stop
// plain LDS loads from moving above another lane's stores).
__device__ __forceinline__ void wave_sync() { __syncthreads(); }

// make a value that all lanes hold identically explicitly wave-uniform
__device__ __forceinline__ double uni(double x) {
    long long v = __double_as_longlong(x);
    int lo = __builtin_amdgcn_readfirstlane(static_cast<int>(v & 0xffffffffLL));
    int hi = __builtin_amdgcn_readfirstlane(static_cast<int>(v >> 32));
    return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned int>(lo));
}
__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ float uni(float x) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x))); }

// broadcast element k of a lane-distributed vector (k wave-uniform)
template <int NS, typename T>
__device__ __forceinline__ T bcast(const T (&v)[NS], int k) {
    const int s = k >> 6;
    T src = v[0];
#pragma unroll
    for (int t = 1; t < NS; t++)
        if (s == t) src = v[t];
    if constexpr (sizeof(T) == 8) {
        long long x = __double_as_longlong(src);
        int lo = __builtin_amdgcn_readlane(static_cast<int>(x & 0xffffffffLL), k & 63);
        int hi = __builtin_amdgcn_readlane(static_cast<int>(x >> 32), k & 63);
        return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned int>(lo));
    } else {
        return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(src), k & 63));
    }
}

// Items of this workgroup of a one-dimensional grid.  States are stored
// species-major: the 8 states of a 64-byte line are neighbours.
struct XcdStates : XcdRange {
    __device__ __forceinline__ explicit XcdStates(long n) : XcdRange(n, gridDim.x, blockIdx.x) {}
};

// The mechanism of a kernel whose first parameter is a DevMech, or a struct
// that begins with one, addressed in the kernel-argument segment.  Out-of-line
// functions take this pointer rather than a reference to the kernel's copy of
// the argument: a reference would make the kernel keep that copy in scratch
// memory and read every field through it, while the kernel-argument segment is
// read with scalar loads.
using KernargMech = const __attribute__((address_space(4))) DevMech;
__device__ __forceinline__ KernargMech* kernarg_mech() {
    return (KernargMech*)__builtin_amdgcn_kernarg_segment_ptr();
}

// One member of the interleaved (C, mu) pairs of the scratch, which holds S
// states side by side (p: this lane's state).
template <int S = 1>
struct SpeciesColumn {
    double* p;
    __device__ __forceinline__ double& operator[](int k) const { return p[2 * S * k]; }
};

// Per-wave LDS scratch for one state evaluation.
struct WaveScratch {
    // K + kDummy pairs at the start of dynamic LDS: C [kmol/m^3] and mu/RT at
    // the state's pressure, (1, 0) from K on.  One 16-byte read serves a
    // species of a reaction's product and of its equilibrium constant, at the
    // address that the compact reaction record holds.
    SpeciesColumn<> C, MU;
    double* WD;    // K + kDummy production-rate accumulators, right behind the pairs
    double* yb;    // N (state broadcast)
    double* W2;    // 2K (Jacobian: wdot, D)
    double* F;     // N (right-hand side out)
    double* Y0;    // N (Jacobian expansion point)
    double* F0;    // N (right-hand side at Y0)
    KernargMech* mech;   // for out-of-line callees
};

// Reactions by lanes: a wavefront evaluates S states at once, 64 / S lanes per
// state, each lane one reaction of a pass.  State s owns column s of the
// scratch: rows of S pairs (C, mu) per species, then rows of S accumulators.
template <int S = 1>
struct LaneView {
    static constexpr int kStride = 64 / S;    // reactions per pass
    unsigned pair0;                           // byte offset of this state's pair in a row
    double* wd;                               // this state's accumulator in the first row
    // (C, mu/RT) and accumulator at a record's slot (16 x species)
    __device__ __forceinline__ double2 pair(unsigned slot) const;
    __device__ __forceinline__ double* acc(unsigned slot) const {
        return reinterpret_cast<double*>(reinterpret_cast<char*>(wd) + (slot * S >> 1));
    }
};

// The scratch of a kernel for mechanisms with reactions that need the general
// code (PLOG, Chebyshev, SRI, chemically activated, power-law orders): kGen.
// The kernels for the others hold none of that code.  With one kernel for both,
// the general passes a call behind a test of the mechanism, every kernel saved
// registers around a call that gri30, h2o2 and n-dodecane never make, and the
// Jacobian kernel of large mechanisms fell to one wavefront per SIMD.
template <bool kGen>
struct Scratch : WaveScratch {};

__host__ __device__ __forceinline__ int species_doubles(int K) { return 3 * (K + kDummy); }

// The same scratch as offsets (in doubles) from the start of dynamic LDS, for
// passing to out-of-line device functions: pointers rebuilt from the LDS base
// inside the callee keep the LDS address space (ds_* instructions).
struct ScratchLayout {
    int yb, W2, F, Y0, F0;
};

__device__ __forceinline__ double* lds_base() {
    extern __shared__ __attribute__((aligned(16))) double lds_raw[];
    return lds_raw;
}

template <int S>
__device__ __forceinline__ double2 LaneView<S>::pair(unsigned slot) const {
    return *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(lds_base()) + (S == 1 ? slot : slot * S + pair0));
}

__device__ __forceinline__ void bind_species(WaveScratch& S, KernargMech* mech) {
    S.mech = mech;
    S.C.p = lds_base();
    S.MU.p = lds_base() + 1;
    S.WD = lds_base() + 2 * (mech->K + kDummy);
}

template <bool kGen>
__device__ __forceinline__ Scratch<kGen> scratch_view(const ScratchLayout& L, KernargMech* mech) {
    double* b = lds_base();
    Scratch<kGen> S;
    bind_species(S, mech);
    S.yb = b + L.yb; S.W2 = b + L.W2; S.F = b + L.F; S.Y0 = b + L.Y0; S.F0 = b + L.F0;
    return S;
}

// Scalar thermodynamic state derived from (T, P, Y): setMassFractions_NoNorm +
// setState_TP (Phase.cpp:362-372; ThermoPhase.cpp:187-198; IdealGasPhase.h:338-354).
// c + a*b with the product rounded before the sum (no fused multiply-add):
// [M] = d C_tot + sum_k (e_k - d) C_k is accumulated exactly as the reference
// does (ThirdBodyCalc::update, ThirdBodyCalc.h:75-83), so a nearly cancelling
// [M] (a bath of an efficiency-0 species) rounds the same way.
__device__ __forceinline__ double add_mul_rn(double c, double a, double b) {
#pragma clang fp contract(off)
    return c + a * b;
}

struct GasState {
    double T, P, mmw, RT, dens, ctot, pressure, logT, recipT, logC0;
};

// Values one lane keeps for the species it owns (slot s = species lane + 64 s).
template <int NS>
struct SpeciesRegs {
    double ym[NS], hrt[NS], cpr[NS], wdot[NS];
};

template <typename R>
__device__ __forceinline__ void nasa7(const double* __restrict__ c16, double T, const double* tt, R& cp, R& h, R& s, R& g) {
    // both coefficient sets are loaded: chosen by address, the loads would wait
    // for tmid first, a second trip to memory
    double c[7];
    const bool low = T <= c16[7];
#pragma unroll
    for (int j = 0; j < 7; j++) {
        const double a = opaque(c16[j]), b = opaque(c16[8 + j]);
        c[j] = low ? a : b;
    }
    double ct0 = c[0];
    double ct1 = c[1] * tt[0];
    double ct2 = c[2] * tt[1];
    double ct3 = c[3] * tt[2];
    double ct4 = c[4] * tt[3];
    double cpv = ct0 + ct1 + ct2 + ct3 + ct4;
    double hv = ct0 + 0.5 * ct1 + 1.0 / 3.0 * ct2 + 0.25 * ct3 + 0.2 * ct4 + c[5] * tt[4];
    double sv = ct0 * tt[5] + ct1 + 0.5 * ct2 + 1.0 / 3.0 * ct3 + 0.25 * ct4 + c[6];
    cp = cpv;
    h = hv;
    s = sv;
    g = hv - sv;
}

// Per-reaction results.
struct RxnVals {
    double kf;     // forward rate constant (with falloff)
    double M;      // third-body concentration (1 if none)
    double rkcn;   // 1/Kc (0 if irreversible)
    double ropf, ropr;
};

// Reaction record unpacked into registers (static indexing only, so nothing
// spills to scratch).
struct RxnRegs {
    int flags, nr, np, tbo, tbn, fo, gen;
    int rk[kMaxSide], pk[kMaxSide];
};

__device__ __forceinline__ void load_rxn(const DevMech& m, int p, RxnRegs& x) {
    const int4* q = reinterpret_cast<const int4*>(m.ri + p);
    const int4 a = q[0], b = q[1], c = q[2];
    x.flags = a.x; x.nr = a.y; x.np = a.z; x.tbo = a.w;
    x.tbn = b.x; x.fo = b.y; x.gen = b.z;
    x.rk[0] = static_cast<short>(c.x & 0xffff); x.rk[1] = static_cast<short>(c.x >> 16);
    x.rk[2] = static_cast<short>(c.y & 0xffff); x.rk[3] = static_cast<short>(c.y >> 16);
    x.pk[0] = static_cast<short>(c.z & 0xffff); x.pk[1] = static_cast<short>(c.z >> 16);
    x.pk[2] = static_cast<short>(c.w & 0xffff); x.pk[3] = static_cast<short>(c.w >> 16);
}

// exp(x) without branches or special-case selects: x = n ln 2 + r, |r| <= ln(2)/2
// (both subtractions exact to the last bit through the fused multiply-adds),
// exp(r) = 1 + r + r^2 q(r) with q the degree-9 minimax polynomial of the
// relative error (3.7e-18, Remez exchange), scaled by v_ldexp, which gives
// infinity, subnormals and zero by itself.  Error below 0.92 ulp, below 0.62
// for 99% of 4 million arguments in [-700, 700] against extended precision.
// Arguments are finite (an infinite one gives NaN) and below 1e13 in magnitude.
constexpr double kLog2e = 1.4426950408889634;
constexpr double kLn2Hi = 0x1.62e42fefa39efp-1, kLn2Lo = 0x1.abc9e3b39803fp-56;
constexpr double kExpC[10] = {0x1.ad7f3cdbe6745p-26, 0x1.28ad9ef903086p-22, 0x1.71df25b30699dp-19,
                              0x1.a01999de1245bp-16, 0x1.a01a012a0f6c4p-13, 0x1.6c16c1843a8b2p-10,
                              0x1.1111111127d0fp-7,  0x1.5555555550834p-5,  0x1.55555555554f9p-3,
                              0x1.000000000000ap-1};
__device__ __forceinline__ double fast_exp(double x) {
    const double n = rint(x * kLog2e);
    double r = fma(n, -kLn2Hi, x);
    r = fma(n, -kLn2Lo, r);
    double q = kExpC[0];
#pragma unroll
    for (int j = 1; j < 10; j++) q = fma(q, r, kExpC[j]);
    q = fma(q, r, 1.0);
    q = fma(q, r, 1.0);
    return ldexp(q, static_cast<int>(n));
}

// M exponentials side by side, the same operations as fast_exp.  One wavefront
// per SIMD evaluates a chain of 13 dependent FMAs at its latency unless other
// chains fill the gaps, and the scheduler, which orders for register pressure,
// does one chain after the other (a library exp also copies each coefficient
// into the destination, v_mov + v_fmac); written out, M chains advance together
// with the coefficients in scalar registers.
template <int M>
__device__ __forceinline__ void fast_exp_n(double (&x)[M]);
template <>
__device__ __forceinline__ void fast_exp_n<2>(double (&x)[2]) {
    double n[2], q[2];
    asm(
        "v_mul_f64 %2, %0, %4\nv_mul_f64 %3, %1, %4\n"
        "v_rndne_f64 %2, %2\nv_rndne_f64 %3, %3\n"
        "v_fma_f64 %0, %2, %5, %0\nv_fma_f64 %1, %3, %5, %1\n"
        "v_fma_f64 %0, %2, %6, %0\nv_fma_f64 %1, %3, %6, %1\n"
        : "+v"(x[0]), "+v"(x[1]),
          "=&v"(n[0]), "=&v"(n[1])
        : "s"(kLog2e), "s"(-kLn2Hi), "s"(-kLn2Lo));
    asm(
        "v_fma_f64 %0, %2, %4, %5\nv_fma_f64 %1, %3, %4, %5\n"
        "v_fma_f64 %0, %0, %2, %6\nv_fma_f64 %1, %1, %3, %6\n"
        "v_fma_f64 %0, %0, %2, %7\nv_fma_f64 %1, %1, %3, %7\n"
        "v_fma_f64 %0, %0, %2, %8\nv_fma_f64 %1, %1, %3, %8\n"
        "v_fma_f64 %0, %0, %2, %9\nv_fma_f64 %1, %1, %3, %9\n"
        "v_fma_f64 %0, %0, %2, %10\nv_fma_f64 %1, %1, %3, %10\n"
        "v_fma_f64 %0, %0, %2, %11\nv_fma_f64 %1, %1, %3, %11\n"
        "v_fma_f64 %0, %0, %2, %12\nv_fma_f64 %1, %1, %3, %12\n"
        "v_fma_f64 %0, %0, %2, %13\nv_fma_f64 %1, %1, %3, %13\n"
        "v_fma_f64 %0, %0, %2, 1.0\nv_fma_f64 %1, %1, %3, 1.0\n"
        "v_fma_f64 %0, %0, %2, 1.0\nv_fma_f64 %1, %1, %3, 1.0\n"
        : "=&v"(q[0]), "=&v"(q[1])
        : "v"(x[0]), "v"(x[1]),
          "v"(kExpC[0]), "s"(kExpC[1]), "s"(kExpC[2]), "s"(kExpC[3]), "s"(kExpC[4]), "s"(kExpC[5]), "s"(kExpC[6]), "s"(kExpC[7]), "s"(kExpC[8]), "s"(kExpC[9]));
#pragma unroll
    for (int j = 0; j < 2; j++) x[j] = ldexp(q[j], static_cast<int>(n[j]));
}
template <>
__device__ __forceinline__ void fast_exp_n<4>(double (&x)[4]) {
    double n[4], q[4];
    asm(
        "v_mul_f64 %4, %0, %8\nv_mul_f64 %5, %1, %8\n"
        "v_mul_f64 %6, %2, %8\nv_mul_f64 %7, %3, %8\n"
        "v_rndne_f64 %4, %4\nv_rndne_f64 %5, %5\n"
        "v_rndne_f64 %6, %6\nv_rndne_f64 %7, %7\n"
        "v_fma_f64 %0, %4, %9, %0\nv_fma_f64 %1, %5, %9, %1\n"
        "v_fma_f64 %2, %6, %9, %2\nv_fma_f64 %3, %7, %9, %3\n"
        "v_fma_f64 %0, %4, %10, %0\nv_fma_f64 %1, %5, %10, %1\n"
        "v_fma_f64 %2, %6, %10, %2\nv_fma_f64 %3, %7, %10, %3\n"
        : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]),
          "=&v"(n[0]), "=&v"(n[1]), "=&v"(n[2]), "=&v"(n[3])
        : "s"(kLog2e), "s"(-kLn2Hi), "s"(-kLn2Lo));
    asm(
        "v_fma_f64 %0, %4, %8, %9\nv_fma_f64 %1, %5, %8, %9\n"
        "v_fma_f64 %2, %6, %8, %9\nv_fma_f64 %3, %7, %8, %9\n"
        "v_fma_f64 %0, %0, %4, %10\nv_fma_f64 %1, %1, %5, %10\n"
        "v_fma_f64 %2, %2, %6, %10\nv_fma_f64 %3, %3, %7, %10\n"
        "v_fma_f64 %0, %0, %4, %11\nv_fma_f64 %1, %1, %5, %11\n"
        "v_fma_f64 %2, %2, %6, %11\nv_fma_f64 %3, %3, %7, %11\n"
        "v_fma_f64 %0, %0, %4, %12\nv_fma_f64 %1, %1, %5, %12\n"
        "v_fma_f64 %2, %2, %6, %12\nv_fma_f64 %3, %3, %7, %12\n"
        "v_fma_f64 %0, %0, %4, %13\nv_fma_f64 %1, %1, %5, %13\n"
        "v_fma_f64 %2, %2, %6, %13\nv_fma_f64 %3, %3, %7, %13\n"
        "v_fma_f64 %0, %0, %4, %14\nv_fma_f64 %1, %1, %5, %14\n"
        "v_fma_f64 %2, %2, %6, %14\nv_fma_f64 %3, %3, %7, %14\n"
        "v_fma_f64 %0, %0, %4, %15\nv_fma_f64 %1, %1, %5, %15\n"
        "v_fma_f64 %2, %2, %6, %15\nv_fma_f64 %3, %3, %7, %15\n"
        "v_fma_f64 %0, %0, %4, %16\nv_fma_f64 %1, %1, %5, %16\n"
        "v_fma_f64 %2, %2, %6, %16\nv_fma_f64 %3, %3, %7, %16\n"
        "v_fma_f64 %0, %0, %4, %17\nv_fma_f64 %1, %1, %5, %17\n"
        "v_fma_f64 %2, %2, %6, %17\nv_fma_f64 %3, %3, %7, %17\n"
        "v_fma_f64 %0, %0, %4, 1.0\nv_fma_f64 %1, %1, %5, 1.0\n"
        "v_fma_f64 %2, %2, %6, 1.0\nv_fma_f64 %3, %3, %7, 1.0\n"
        "v_fma_f64 %0, %0, %4, 1.0\nv_fma_f64 %1, %1, %5, 1.0\n"
        "v_fma_f64 %2, %2, %6, 1.0\nv_fma_f64 %3, %3, %7, 1.0\n"
        : "=&v"(q[0]), "=&v"(q[1]), "=&v"(q[2]), "=&v"(q[3])
        : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]),
          "v"(kExpC[0]), "s"(kExpC[1]), "s"(kExpC[2]), "s"(kExpC[3]), "s"(kExpC[4]), "s"(kExpC[5]), "s"(kExpC[6]), "s"(kExpC[7]), "s"(kExpC[8]), "s"(kExpC[9]));
#pragma unroll
    for (int j = 0; j < 4; j++) x[j] = ldexp(q[j], static_cast<int>(n[j]));
}
template <>
__device__ __forceinline__ void fast_exp_n<6>(double (&x)[6]) {
    double n[6], q[6];
    asm(
        "v_mul_f64 %6, %0, %12\nv_mul_f64 %7, %1, %12\n"
        "v_mul_f64 %8, %2, %12\nv_mul_f64 %9, %3, %12\n"
        "v_mul_f64 %10, %4, %12\nv_mul_f64 %11, %5, %12\n"
        "v_rndne_f64 %6, %6\nv_rndne_f64 %7, %7\n"
        "v_rndne_f64 %8, %8\nv_rndne_f64 %9, %9\n"
        "v_rndne_f64 %10, %10\nv_rndne_f64 %11, %11\n"
        "v_fma_f64 %0, %6, %13, %0\nv_fma_f64 %1, %7, %13, %1\n"
        "v_fma_f64 %2, %8, %13, %2\nv_fma_f64 %3, %9, %13, %3\n"
        "v_fma_f64 %4, %10, %13, %4\nv_fma_f64 %5, %11, %13, %5\n"
        "v_fma_f64 %0, %6, %14, %0\nv_fma_f64 %1, %7, %14, %1\n"
        "v_fma_f64 %2, %8, %14, %2\nv_fma_f64 %3, %9, %14, %3\n"
        "v_fma_f64 %4, %10, %14, %4\nv_fma_f64 %5, %11, %14, %5\n"
        : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(x[4]), "+v"(x[5]),
          "=&v"(n[0]), "=&v"(n[1]), "=&v"(n[2]), "=&v"(n[3]), "=&v"(n[4]), "=&v"(n[5])
        : "s"(kLog2e), "s"(-kLn2Hi), "s"(-kLn2Lo));
    asm(
        "v_fma_f64 %0, %6, %12, %13\nv_fma_f64 %1, %7, %12, %13\n"
        "v_fma_f64 %2, %8, %12, %13\nv_fma_f64 %3, %9, %12, %13\n"
        "v_fma_f64 %4, %10, %12, %13\nv_fma_f64 %5, %11, %12, %13\n"
        "v_fma_f64 %0, %0, %6, %14\nv_fma_f64 %1, %1, %7, %14\n"
        "v_fma_f64 %2, %2, %8, %14\nv_fma_f64 %3, %3, %9, %14\n"
        "v_fma_f64 %4, %4, %10, %14\nv_fma_f64 %5, %5, %11, %14\n"
        "v_fma_f64 %0, %0, %6, %15\nv_fma_f64 %1, %1, %7, %15\n"
        "v_fma_f64 %2, %2, %8, %15\nv_fma_f64 %3, %3, %9, %15\n"
        "v_fma_f64 %4, %4, %10, %15\nv_fma_f64 %5, %5, %11, %15\n"
        "v_fma_f64 %0, %0, %6, %16\nv_fma_f64 %1, %1, %7, %16\n"
        "v_fma_f64 %2, %2, %8, %16\nv_fma_f64 %3, %3, %9, %16\n"
        "v_fma_f64 %4, %4, %10, %16\nv_fma_f64 %5, %5, %11, %16\n"
        "v_fma_f64 %0, %0, %6, %17\nv_fma_f64 %1, %1, %7, %17\n"
        "v_fma_f64 %2, %2, %8, %17\nv_fma_f64 %3, %3, %9, %17\n"
        "v_fma_f64 %4, %4, %10, %17\nv_fma_f64 %5, %5, %11, %17\n"
        "v_fma_f64 %0, %0, %6, %18\nv_fma_f64 %1, %1, %7, %18\n"
        "v_fma_f64 %2, %2, %8, %18\nv_fma_f64 %3, %3, %9, %18\n"
        "v_fma_f64 %4, %4, %10, %18\nv_fma_f64 %5, %5, %11, %18\n"
        "v_fma_f64 %0, %0, %6, %19\nv_fma_f64 %1, %1, %7, %19\n"
        "v_fma_f64 %2, %2, %8, %19\nv_fma_f64 %3, %3, %9, %19\n"
        "v_fma_f64 %4, %4, %10, %19\nv_fma_f64 %5, %5, %11, %19\n"
        "v_fma_f64 %0, %0, %6, %20\nv_fma_f64 %1, %1, %7, %20\n"
        "v_fma_f64 %2, %2, %8, %20\nv_fma_f64 %3, %3, %9, %20\n"
        "v_fma_f64 %4, %4, %10, %20\nv_fma_f64 %5, %5, %11, %20\n"
        "v_fma_f64 %0, %0, %6, %21\nv_fma_f64 %1, %1, %7, %21\n"
        "v_fma_f64 %2, %2, %8, %21\nv_fma_f64 %3, %3, %9, %21\n"
        "v_fma_f64 %4, %4, %10, %21\nv_fma_f64 %5, %5, %11, %21\n"
        "v_fma_f64 %0, %0, %6, 1.0\nv_fma_f64 %1, %1, %7, 1.0\n"
        "v_fma_f64 %2, %2, %8, 1.0\nv_fma_f64 %3, %3, %9, 1.0\n"
        "v_fma_f64 %4, %4, %10, 1.0\nv_fma_f64 %5, %5, %11, 1.0\n"
        "v_fma_f64 %0, %0, %6, 1.0\nv_fma_f64 %1, %1, %7, 1.0\n"
        "v_fma_f64 %2, %2, %8, 1.0\nv_fma_f64 %3, %3, %9, 1.0\n"
        "v_fma_f64 %4, %4, %10, 1.0\nv_fma_f64 %5, %5, %11, 1.0\n"
        : "=&v"(q[0]), "=&v"(q[1]), "=&v"(q[2]), "=&v"(q[3]), "=&v"(q[4]), "=&v"(q[5])
        : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(x[4]), "v"(x[5]),
          "v"(kExpC[0]), "s"(kExpC[1]), "s"(kExpC[2]), "s"(kExpC[3]), "s"(kExpC[4]), "s"(kExpC[5]), "s"(kExpC[6]), "s"(kExpC[7]), "s"(kExpC[8]), "s"(kExpC[9]));
#pragma unroll
    for (int j = 0; j < 6; j++) x[j] = ldexp(q[j], static_cast<int>(n[j]));
}
// 10^x, |x| moderate: x ln 10 in two parts
__device__ __forceinline__ double fast_exp10(double x) {
    const double h = x * 2.302585092994046;
    const double l = fma(x, 2.302585092994046, -h) + x * -2.1707562233822494e-16;
    const double e = fast_exp(h);
    return fma(e, l, e);
}

// Exponent of a Troe centre term, kept where fast_exp is defined: 1/T3 is
// infinite for Tsang, T2 is 1e100 in some mechanisms, T3 and T1 may be tiny and
// of either sign.  Beyond +-1e4 the exponential is infinite or 0 all the same.
__device__ __forceinline__ double troe_arg(double x) { return fmin(fmax(x, -1e4), 1e4); }

// Exponent of 1/K_c kept where fast_exp is defined (the NASA polynomials pass
// 1e13 at 1e7 K, a vanishing pressure makes it infinite): beyond +-1e5 the
// exponential is infinite or 0 all the same.  NaN goes to the upper end, that is
// to the cap of 1/K_c.
__device__ __forceinline__ double kc_arg(double x) { return fmax(fmin(x, 1e5), -1e5); }

// Transcendentals of the rate constants.  kF32: evaluated in FP32 (hardware
// exp2/log2 based) on FP64 arguments rounded to FP32, widened back to FP64;
// arguments whose result would leave the FP32 range take the FP64 function.
// The equilibrium constants never use these (their exp stays FP64).
template <bool kF32>
__device__ __forceinline__ double rate_exp(double arg) {
    if constexpr (kF32) {
        if (fabs(arg) < 80.0) return static_cast<double>(expf(static_cast<float>(arg)));
        return exp(arg);
    } else {
        return fast_exp(arg);
    }
}
template <bool kF32>
__device__ __forceinline__ double rate_log10(double x) {
    if constexpr (kF32) {
        if (x > 1e-35 && x < 1e35) return static_cast<double>(log10f(static_cast<float>(x)));
    }
    return log10(x);
}
template <bool kF32>
__device__ __forceinline__ double rate_exp10(double x) {
    if constexpr (kF32) {
        if (fabs(x) < 35.0) return static_cast<double>(exp10f(static_cast<float>(x)));
        return exp10(x);
    } else {
        return fast_exp10(x);
    }
}

// PLOG rate constant (PlogRate::updateFromStruct / evalFromStruct,
// include/cantera/kinetics/PlogRate.h:110-164).  Record r: ng, ln P[ng],
// first[ng], end[ng], then (A, b, Ea/R) per entry; groups 0 and ng-1 are the
// copies at ln P = -1000 and +1000.  The interval is [ln P[i-1], ln P[i]) with
// i the first group above ln P; each end takes ln(1e-300 + sum of the group's
// Arrhenius terms), and ln k is interpolated linearly in ln P.
__device__ __forceinline__ double plog_rate(const double* __restrict__ r, double logP, double logT, double recipT) {
    const int ng = static_cast<int>(r[0]);
    const double* lp = r + 1;
    const double* e = r + 1 + 3 * ng;
    int i = 1;
    while (i < ng - 1 && !(lp[i] > logP)) i++;
    double lk[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int q = i - 1 + h;
        double k = 1e-300;
        for (int j = static_cast<int>(r[1 + ng + q]); j < static_cast<int>(r[1 + 2 * ng + q]); j++)
            k += e[3 * j] * exp(e[3 * j + 1] * logT - e[3 * j + 2] * recipT);
        lk[h] = log(k);
    }
    const double rdp = 1.0 / (lp[i] - lp[i - 1]);
    return exp(lk[0] + (lk[1] - lk[0]) * (logP - lp[i - 1]) * rdp);
}

// Chebyshev rate constant (ChebyshevRate::updateFromStruct / evalFromStruct,
// include/cantera/kinetics/ChebyshevRate.h:133-171).  Record r: TrNum, TrDen,
// PrNum, PrDen, nT, nP, coefficients (nT x nP, row-major).  Each row is first
// reduced over the pressure polynomials, then the temperature series is summed
// with the same three-term recurrence, row by row.
__device__ __forceinline__ double cheb_rate(const double* __restrict__ r, double log10P, double recipT) {
    const int nT = static_cast<int>(r[4]), nP = static_cast<int>(r[5]);
    const double* c = r + 6;
    const double Pr = (2 * log10P + r[2]) * r[3];
    const double Tr = (2 * recipT + r[0]) * r[1];
    double logk = 0.0, Tm1 = Tr, Tn = 1.0;
    for (int i = 0; i < nT; i++) {
        double dot = c[i * nP];
        double Pm1 = Pr, Pn = 1.0;
        for (int j = 1; j < nP; j++) {
            const double Pp1 = 2 * Pr * Pn - Pm1;
            dot += Pp1 * c[i * nP + j];
            Pm1 = Pn;
            Pn = Pp1;
        }
        if (i == 0) {
            logk = dot;
        } else {
            const double Tp1 = 2 * Tr * Tn - Tm1;
            logk += Tp1 * dot;
            Tm1 = Tn;
            Tn = Tp1;
        }
    }
    return pow(10.0, logk);
}

// Rate constants of the PLOG and Chebyshev reactions at the gas state.  They
// come first in permuted order and number at most 64, so lane j evaluates
// reaction j once per state, before the reaction loop; the loop's first pass
// (lane j, reaction j) takes the value from the register.  Other lanes, and
// mechanisms without such reactions, return 0.
__device__ __forceinline__ double pdep_rate_lane(const DevMech& m, const GasState& g) {
    double k = 0.0;
    if (m.n_pd > 0) {
        const int lane = lane_id();
        if (lane < m.n_pd) {
            const int flags = m.ri[lane].flags;
            const int fo = m.ri[lane].fo;
            k = (flags & 64) ? plog_rate(m.pdd + fo, log(g.pressure), g.logT, g.recipT)
                             : cheb_rate(m.pdd + fo, log10(g.pressure), g.recipT);
        }
    }
    return k;
}

// SRI falloff function at reduced pressure pr (SriRate::updateTemp and F,
// Falloff.cpp:389-403); fo[3..7] = a, b, c, d, e.  Out of line: SRI reactions
// are rare, and inlined this code enlarges every caller's register frame.
__device__ __noinline__ double sri_falloff(const double* __restrict__ fo, double T, double pr) {
    double w = fo[3] * exp(-fo[4] / T);
    if (fo[5] != 0.0) w += exp(-T / fo[5]);
    const double lpr = log10(fmax(pr, kSmallNumber));
    return pow(w, 1.0 / (1.0 + lpr * lpr)) * (fo[6] * pow(T, fo[7]));
}

// sum_k (e_k - d) C_k over the explicit efficiencies of a reaction, in list
// order without fused multiply-adds.  Lists are padded to whole groups of
// kTbPad entries with efficiency 0, so a group's table loads, then its
// concentration loads, are all in flight together with no test against the
// list length.
template <int S>
__device__ __forceinline__ double efficiency_sum(const DevMech& m, SpeciesColumn<S> C, int tbo, int tbn) {
    double sum = 0.0;
    for (int j0 = 0; j0 == 0 || j0 < tbn; j0 += kTbPad) {
        int kk[kTbPad];
        double ee[kTbPad], cc[kTbPad];
#pragma unroll
        for (int b = 0; b < kTbPad; b++) {
            kk[b] = m.tbk[tbo + j0 + b];
            ee[b] = m.tbe[tbo + j0 + b];
        }
#pragma unroll
        for (int b = 0; b < kTbPad; b++) cc[b] = opaque(C[kk[b]]);
#pragma unroll
        for (int b = 0; b < kTbPad; b++) sum = add_mul_rn(sum, ee[b], cc[b]);
    }
    return sum;
}

// Evaluate reaction p (permuted index) at the gas state; C and MU live in LDS.
// kpd: this lane's pdep_rate_lane value (used for flags bit 6/7 only).
// kF32: rate constants (Arrhenius, falloff centre and blending) through the
// FP32 transcendentals above; everything else FP64.
// perturb: the reaction's rate multiplier (m_perturb, Kinetics::setMultiplier),
// applied to the forward rate of progress before the reverse one is formed.
template <bool kF32 = false, int S = 1>
__device__ __forceinline__ void eval_reaction(const DevMech& m, int p, const GasState& g,
                                              SpeciesColumn<S> C, SpeciesColumn<S> MU,
                                              const RxnRegs& x, double kpd, RxnVals& o, double perturb = 1.0) {
    const double4 rd = reinterpret_cast<const double4*>(m.rd)[p];
    const int type = (x.flags >> 1) & 3;
    const bool rev = x.flags & 1;
    double M = 1.0;
    if (x.flags & 32) {
        const double sum = efficiency_sum(m, C, x.tbo, x.tbn);
        M = add_mul_rn(sum, m.tbdef[p], g.ctot);
    }
    double kf;
    if (type <= kThreeBody) {
        // PLOG and Chebyshev constants (FP64 in both precisions) come from kpd
        kf = (x.flags & 192) ? kpd : rd.x * rate_exp<kF32>(rd.y * g.logT - rd.z * g.recipT);
    } else {
        const double* fo = m.fod + 8 * x.fo;
        const bool sri = x.flags & 256;
        double work = 0.0;
        if (type == kTroe && !sri) {
            // Troe (fo[7] = 0) and Tsang (Fcent = A + B T)
            double Fcent = (1.0 - fo[3]) * rate_exp<kF32>(troe_arg(-g.T * fo[4])) +
                           fo[3] * rate_exp<kF32>(troe_arg(-g.T * fo[5]));
            if (fo[6] != 0.0) Fcent += rate_exp<kF32>(troe_arg(-fo[6] / g.T));
            Fcent += fo[7] * g.T;
            work = rate_log10<kF32>(fmax(Fcent, kSmallNumber));
        }
        double rc_low = fo[0] * rate_exp<kF32>(fo[1] * g.logT - fo[2] * g.recipT);
        double rc_high = rd.x * rate_exp<kF32>(rd.y * g.logT - rd.z * g.recipT);
        double pr = M * rc_low / (rc_high + kSmallNumber);
        double F = 1.0;
        if (type == kTroe && sri) {
            F = sri_falloff(fo, g.T, pr);
        } else if (type == kTroe) {
            double lpr = rate_log10<kF32>(fmax(pr, kSmallNumber));
            double cc = -0.4 - 0.67 * work;
            double nn = 0.75 - 1.27 * work;
            double f1 = (lpr + cc) / (nn - 0.14 * (lpr + cc));
            double lgf = work / (1.0 + f1 * f1);
            F = rate_exp10<kF32>(lgf);
        }
        // FalloffRate::evalFromStruct (Falloff.h:154-176): Pr/(1+Pr) F k_inf, or
        // F/(1+Pr) k_0 for a chemically activated reaction
        const double fac = F / (1.0 + pr);
        kf = (x.flags & 512) ? fac * rc_low : (pr * fac) * rc_high;
    }
    o.kf = kf;
    o.M = M;
    // inverse equilibrium constant (BulkKinetics.cpp:465-484)
    double rkcn = 0.0;
    if (rev) {
        double dp = 0.0;
        if (x.flags & 16) {
            const double* gs = m.gend + 12 * x.gen;
#pragma unroll
            for (int j = 0; j < kMaxSide; j++)
                if (j < x.np) dp += gs[8 + j] * MU[x.pk[j]];
        } else {
            dp = MU[x.pk[0]];
            if (x.np > 1) dp += MU[x.pk[1]];
            if (x.np > 2) dp += MU[x.pk[2]];
        }
        double delta = dp;
        if (x.flags & 8) {
            const double* gs = m.gend + 12 * x.gen;
#pragma unroll
            for (int j = 0; j < kMaxSide; j++)
                if (j < x.nr) delta -= gs[4 + j] * MU[x.rk[j]];
        } else {
            double dr = MU[x.rk[0]];
            if (x.nr > 1) dr += MU[x.rk[1]];
            if (x.nr > 2) dr += MU[x.rk[2]];
            delta -= dr;
        }
        rkcn = fmin(fast_exp(kc_arg(delta - rd.w * g.logC0)), kBigNumber);
    }
    o.rkcn = rkcn;
    double ropf = kf * perturb;
    if (type == kThreeBody) ropf *= M;
    double ropr = ropf * rkcn;
    // concentration products with the reference's negative-concentration rules
    if (x.flags & 8) {
        const double* gs = m.gend + 12 * x.gen;
#pragma unroll
        for (int j = 0; j < kMaxSide; j++) {
            if (j < x.nr) {
                double order = gs[j];
                if (order != 0.0) {
                    double c = C[x.rk[j]];
                    ropf = (c > 0.0) ? ropf * pow(c, order) : 0.0;
                }
            }
        }
    } else {
        double a = C[x.rk[0]];
        if (x.nr == 1) {
            ropf *= a;
        } else if (x.nr == 2) {
            double b = C[x.rk[1]];
            ropf = (a < 0 && b < 0) ? 0.0 : ropf * (a * b);
        } else {
            double b = C[x.rk[1]], d = C[x.rk[2]];
            ropf = ((a < 0 && (b < 0 || d < 0)) || (b < 0 && d < 0)) ? 0.0 : ropf * (a * b * d);
        }
    }
    if (rev) {
        if (x.flags & 16) {
            const double* gs = m.gend + 12 * x.gen;
#pragma unroll
            for (int j = 0; j < kMaxSide; j++) {
                if (j < x.np) {
                    double c = C[x.pk[j]];
                    ropr = (c > 0.0) ? ropr * pow(c, gs[8 + j]) : 0.0;
                }
            }
        } else {
            double a = C[x.pk[0]];
            if (x.np == 1) {
                ropr *= a;
            } else if (x.np == 2) {
                double b = C[x.pk[1]];
                ropr = (a < 0 && b < 0) ? 0.0 : ropr * (a * b);
            } else {
                double b = C[x.pk[1]], d = C[x.pk[2]];
                ropr = ((a < 0 && (b < 0 || d < 0)) || (b < 0 && d < 0)) ? 0.0 : ropr * (a * b * d);
            }
        }
    }
    o.ropf = ropf;
    o.ropr = ropr;
}

// ---- standard reactions (RxnS), straight-line ---------------------------------
//
// One wavefront evaluates one state, so nothing but independent work in the
// same instruction stream hides the latency of the table loads, the LDS reads
// and the exponential's chain of dependent FMAs.  These functions therefore
// have no branches: unused entries read the sentinel slot, selects are made on
// values that the compiler cannot trace back to their loads (it turns a select
// on a computed product into a branch around it, and everything after waits
// there), and B reactions per lane are evaluated side by side.

// x of two reactants/products negative: the rate of progress is 0
// (the C1/C2/C3 rules of StoichManager.h:147-366; the sentinel's 1 is never negative)
__device__ __forceinline__ double zero_if_two_negative(double v, double a, double b, double d) {
    const bool na = a < 0, nb = b < 0, nd = d < 0;
    const bool two = (na & nb) | ((na | nb) & nd);
    v = opaque(v);
    return two ? 0.0 : v;
}

struct StdRxn {
    uint4 q;
    double4 rd;     // A, b, Ea/R, dn
    __device__ __forceinline__ void load(const DevMech& m, const RxnS* rs, int p) {
        q = reinterpret_cast<const uint4*>(rs)[p];
        rd = reinterpret_cast<const double4*>(m.rd)[p];
    }
    __device__ __forceinline__ unsigned slot(int e) const {   // entry e: r0 r1 r2 p0 p1 p2 p3
        const unsigned w = e < 2 ? q.x : (e < 4 ? q.y : (e < 6 ? q.z : q.w));
        return (e & 1) ? w >> 16 : w & 0xffffu;
    }
    __device__ __forceinline__ bool reversible() const { return q.w & 0x10000u; }
    __device__ __forceinline__ bool four_products() const { return q.w & 0x20000u; }
};

// exponent of 1/K_c from the pairs of the six entries
__device__ __forceinline__ double std_kc_arg(const StdRxn& x, double logC0, const double2 (&v)[6]) {
    const double dr = (v[0].y + v[1].y) + v[2].y;
    const double dp = (v[3].y + v[4].y) + v[5].y;
    return kc_arg((dp - dr) - x.rd.w * logC0);
}

// net rate of progress from the forward constant kf (perturbed, times [M] for a
// three-body reaction) and exp(std_kc_arg)
__device__ __forceinline__ double std_ropnet(const StdRxn& x, double kf, double ekc, const double2 (&v)[6]) {
    const double rkcn = fmin(ekc, kBigNumber);
    const double f = zero_if_two_negative(kf * (v[0].x * v[1].x * v[2].x), v[0].x, v[1].x, v[2].x);
    const double r =
        zero_if_two_negative(kf * rkcn * (v[3].x * v[4].x * v[5].x), v[3].x, v[4].x, v[5].x);
    return f - (x.reversible() ? r : 0.0);
}

// -r to the reactants' accumulators, +r to the products'
template <int S>
__device__ __forceinline__ void std_scatter(const LaneView<S>& v, const StdRxn& x, double r) {
#pragma unroll
    for (int e = 0; e < 3; e++) atomicAdd(v.acc(x.slot(e)), -r);
#pragma unroll
    for (int e = 3; e < 6; e++) atomicAdd(v.acc(x.slot(e)), r);
}

// B passes of elementary reactions: this lane's are p, p + 64 / S, ...
template <int B, bool kF32, bool kPert, int S>
__device__ __forceinline__ void plain_block(const DevMech& m, const RxnS* rs, const LaneView<S>& lv, const GasState& g,
                                            int p, int pert_rxn, double pert_v) {
    constexpr int kStride = LaneView<S>::kStride;
    StdRxn x[B];
#pragma unroll
    for (int b = 0; b < B; b++) x[b].load(m, rs, p + kStride * b);
    double2 v[B][6];
    double r[B], ex[2 * B];
#pragma unroll
    for (int b = 0; b < B; b++)
#pragma unroll
        for (int e = 0; e < 6; e++) v[b][e] = lv.pair(x[b].slot(e));
#pragma unroll
    for (int b = 0; b < B; b++) {
        ex[b] = x[b].rd.y * g.logT - x[b].rd.z * g.recipT;
        ex[B + b] = std_kc_arg(x[b], g.logC0, v[b]);
    }
    if constexpr (kF32) {
#pragma unroll
        for (int b = 0; b < B; b++) {
            ex[b] = rate_exp<true>(ex[b]);
            ex[B + b] = fast_exp(ex[B + b]);
        }
    } else {
        fast_exp_n(ex);
    }
    bool four = false;
#pragma unroll
    for (int b = 0; b < B; b++) {
        double kf = x[b].rd.x * ex[b];
        if constexpr (kPert) kf *= (p + kStride * b == pert_rxn) ? pert_v : 1.0;
        r[b] = std_ropnet(x[b], kf, ex[B + b], v[b]);
        four |= x[b].four_products();
    }
#pragma unroll
    for (int b = 0; b < B; b++) std_scatter(lv, x[b], r[b]);
    if (__any(four)) {
#pragma unroll
        for (int b = 0; b < B; b++) atomicAdd(lv.acc(x[b].slot(6)), r[b]);
    }
}

// One pass that may hold three-body, Lindemann, Troe/Tsang and elementary
// reactions: every lane runs the same code (the falloff part only if the pass
// has such a reaction), the type selects among the results.  The formulas are
// eval_reaction's.
template <bool kF32, bool kPert, int S>
__device__ __forceinline__ void falloff_pass(const DevMech& m, const RxnS* rs, const LaneView<S>& lv,
                                             SpeciesColumn<S> C, const GasState& g, int p, int pert_rxn,
                                             double pert_v) {
    StdRxn x;
    x.load(m, rs, p);
    const int4* qi = reinterpret_cast<const int4*>(m.ri + p);
    const int4 ia = qi[0], ib = qi[1];
    const double tbdef = m.tbdef[p];
    const int type = (ia.x >> 1) & 3;
    const double4* f4 = reinterpret_cast<const double4*>(m.fod + 8 * (ib.y < 0 ? m.n_fo : ib.y));
    const double4 fa = f4[0], fb = f4[1];   // A0, b0, Ea0/R, a | 1/T3, 1/T1, T2, B
    double2 v[6];
#pragma unroll
    for (int e = 0; e < 6; e++) v[e] = lv.pair(x.slot(e));
    const double M = add_mul_rn(efficiency_sum(m, C, ia.w, ib.x), tbdef, g.ctot);
    // the pass's six exponentials side by side
    double ex[6];
    ex[0] = x.rd.y * g.logT - x.rd.z * g.recipT;
    ex[1] = std_kc_arg(x, g.logC0, v);
    ex[2] = fa.y * g.logT - fa.z * g.recipT;
    ex[3] = troe_arg(-g.T * fb.x);
    ex[4] = troe_arg(-g.T * fb.y);
    ex[5] = troe_arg(-fb.z * g.recipT);
    const bool falloff = __any(type >= kLindemann);
    if constexpr (kF32) {
        ex[1] = fast_exp(ex[1]);
        ex[0] = rate_exp<true>(ex[0]);
        if (falloff)
#pragma unroll
            for (int j = 2; j < 6; j++) ex[j] = rate_exp<true>(ex[j]);
    } else if (falloff) {
        fast_exp_n(ex);
    } else {
        double e2[2] = {ex[0], ex[1]};
        fast_exp_n(e2);
        ex[0] = e2[0];
        ex[1] = e2[1];
    }
    double kf = x.rd.x * ex[0];
    if (falloff) {
        const double k0 = fa.x * ex[2];
        double Fcent = (1.0 - fa.w) * ex[3] + fa.w * ex[4];
        Fcent += (fb.z != 0.0) ? opaque(ex[5]) : 0.0;
        Fcent += fb.w * g.T;
        const double work = rate_log10<kF32>(fmax(Fcent, kSmallNumber));
        const double pr = M * k0 / (kf + kSmallNumber);
        const double lpr = rate_log10<kF32>(fmax(pr, kSmallNumber));
        const double cc = -0.4 - 0.67 * work;
        const double nn = 0.75 - 1.27 * work;
        const double f1 = (lpr + cc) / (nn - 0.14 * (lpr + cc));
        const double Ft = opaque(rate_exp10<kF32>(work / (1.0 + f1 * f1)));
        const double F = (type == kTroe) ? Ft : 1.0;
        const double kfo = opaque((pr * (F / (1.0 + pr))) * kf);
        kf = (type >= kLindemann) ? kfo : kf;
    }
    if constexpr (kPert) kf *= (p == pert_rxn) ? pert_v : 1.0;
    const double kM = opaque(kf * M);
    kf = (type == kThreeBody) ? kM : kf;
    const double r = std_ropnet(x, kf, ex[1], v);
    std_scatter(lv, x, r);
    if (__any(x.four_products())) atomicAdd(lv.acc(x.slot(6)), r);
}

// The standard reactions from `first` (a whole number of passes): falloff passes
// up to mid, elementary ones up to last, kBlock of these side by side.
template <int kBlock, bool kF32, bool kPert, int S>
__device__ __forceinline__ void standard_passes(const DevMech& m, const RxnS* rs, const LaneView<S>& lv,
                                                SpeciesColumn<S> C, const GasState& g, int lane, int first, int mid,
                                                int last, int pert_rxn, double pert_v) {
    constexpr int kStride = LaneView<S>::kStride;
    int q = first;
    for (; q < mid; q += kStride) falloff_pass<kF32, kPert, S>(m, rs, lv, C, g, q + lane, pert_rxn, pert_v);
    for (; q + (kBlock - 1) * kStride < last; q += kBlock * kStride)
        plain_block<kBlock, kF32, kPert, S>(m, rs, lv, g, q + lane, pert_rxn, pert_v);
    if constexpr (kBlock > 2)
        if (q + kStride < last) {
            plain_block<2, kF32, kPert, S>(m, rs, lv, g, q + lane, pert_rxn, pert_v);
            q += 2 * kStride;
        }
    if constexpr (kBlock > 1)
        if (q < last) plain_block<1, kF32, kPert, S>(m, rs, lv, g, q + lane, pert_rxn, pert_v);
}

// Gas state + per-species thermo, concentrations and chemical potentials.
// Y values: lane owns species lane + 64 s in yk[s].  Leaves C and MU in LDS.
// rho > 0: the state is (T, rho) instead of (T, P) (ThermoPhase::setState_TD);
// the pressure is then R T rho / Wbar.
// kSeqSum: 1/Wbar = sum_k Y_k/W_k summed in species order, as
// Phase::setMassFractions_NoNorm does (Phase.cpp:362-372), through S.WD (the
// batched rates and Jacobians, whose results are compared bit for bit);
// otherwise a wavefront tree sum (the integrator's right-hand side).
template <int NS, bool kSeqSum = false>
__device__ __forceinline__ void species_pass(const DevMech& m, const WaveScratch& S, double T, double P,
                                             const double (&yk)[NS], GasState& g, SpeciesRegs<NS>& sr,
                                             double rho = 0.0) {
    const int lane = lane_id();
    double sum = 0.0;
#pragma unroll
    for (int s = 0; s < NS; s++) {
        int k = lane + kWave * s;
        sr.ym[s] = (k < m.K) ? yk[s] * m.rmw[k] : 0.0;
        sum += sr.ym[s];
    }
    g.T = T;
    g.RT = T * kGasConstant;
    g.recipT = 1.0 / T;
    if constexpr (kSeqSum) {
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int k = lane + kWave * s;
            if (k < m.K) S.WD[k] = sr.ym[s];
        }
        wave_sync();
        sum = 0.0;
        int k = 0;
        for (; k + 8 <= m.K; k += 8) {   // the adds are a chain, the loads are not
            double t[8];
#pragma unroll
            for (int b = 0; b < 8; b++) t[b] = S.WD[k + b];
#pragma unroll
            for (int b = 0; b < 8; b++) sum += t[b];
        }
        for (; k < m.K; k++) sum += S.WD[k];
        wave_sync();
    } else {
        sum = uni(wave_sum(sum));
    }
    // rounded as the reference does (ThermoPhase.cpp, IdealGasPhase.h): a
    // nearly cancelling [M] amplifies the last bits of C_tot and C_k
    g.mmw = 1.0 / sum;
    g.dens = (rho > 0.0) ? rho : P * g.mmw / g.RT;
    g.ctot = g.dens / g.mmw;
    g.pressure = kGasConstant * g.ctot * T;
    g.P = (rho > 0.0) ? g.pressure : P;
    // ln T, ln(P/RT) and ln(P/Pref) in one evaluation, a lane each
    const double lg = log(lane == 0 ? T : (lane == 1 ? g.ctot : g.pressure * m.rpref));
    g.logT = readlane_f64(lg, 0);
    g.logC0 = readlane_f64(lg, 1);
    const double lnp = readlane_f64(lg, 2);
    double tt[6];
    tt[0] = T;
    tt[1] = T * T;
    tt[2] = tt[1] * T;
    tt[3] = tt[2] * T;
    tt[4] = g.recipT;
    tt[5] = g.logT;
#pragma unroll
    for (int s = 0; s < NS; s++) {
        int k = lane + kWave * s;
        sr.cpr[s] = 0.0;
        sr.hrt[s] = 0.0;
        if (k < m.K) {
            double cp, h, sR, g0;
            nasa7(m.nasa + 16 * k, T, tt, cp, h, sR, g0);
            sr.cpr[s] = cp;
            sr.hrt[s] = h;
            *reinterpret_cast<double2*>(lds_base() + 2 * k) = double2{sr.ym[s] * g.dens, g0 + lnp};
        }
    }
    // the sentinel slots of the compact records
    *reinterpret_cast<double2*>(lds_base() + 2 * (m.K + lane)) = double2{1.0, 0.0};
}

// The passes of 64 reactions that hold non-standard reactions (PLOG,
// Chebyshev, SRI, chemically activated, power-law orders), by the general code.
template <bool kF32, bool kPert>
__device__ __forceinline__ void general_passes(const DevMech& m, const WaveScratch& S, const GasState& g,
                                               int pert_rxn, double pert_v) {
    const int lane = lane_id();
    const double kpd = pdep_rate_lane(m, g);
    for (int p = lane; p < min(kWave * m.gen_end, m.I); p += kWave) {
        RxnRegs x;
        load_rxn(m, p, x);
        RxnVals v;
        if constexpr (kPert) eval_reaction<kF32>(m, p, g, S.C, S.MU, x, kpd, v, p == pert_rxn ? pert_v : 1.0);
        else eval_reaction<kF32>(m, p, g, S.C, S.MU, x, kpd, v);
        const double r = v.ropf - v.ropr;
        const double* gs = (x.gen >= 0) ? m.gend + 12 * x.gen : m.gend;
        const bool rgen = x.flags & 8, pgen = x.flags & 16;
#pragma unroll
        for (int j = 0; j < kMaxSide; j++)
            if (j < x.nr) atomicAdd(&S.WD[x.rk[j]], -(rgen ? gs[4 + j] : 1.0) * r);
#pragma unroll
        for (int j = 0; j < kMaxSide; j++)
            if (j < x.np) atomicAdd(&S.WD[x.pk[j]], (pgen ? gs[8 + j] : 1.0) * r);
    }
    wave_sync();
}

// Net production rates for the species each lane owns (after species_pass).
// Each reaction lane adds -nu' ropnet to its reactants and +nu'' ropnet to its
// products with LDS FP64 atomics (the species lists are already in registers),
// so no second pass over a gather table is needed; the summation order of a
// species' terms is the hardware's, not the reference's reaction order.
// kPert: reaction pert_rxn (permuted index) runs with rate multiplier pert_v.
// kBlock: elementary passes evaluated side by side.
template <int NS, bool kF32 = false, bool kPert = false, int kBlock = 3, bool kGen>
__device__ __forceinline__ void production_rates(const DevMech& m, const Scratch<kGen>& S, const GasState& g,
                                                 SpeciesRegs<NS>& sr, int pert_rxn = -1, double pert_v = 1.0) {
    const int lane = lane_id();
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int k = lane + kWave * s;
        if (k < m.K) S.WD[k] = 0.0;
    }
    wave_sync();
    if constexpr (kGen) general_passes<kF32, kPert>(m, S, g, pert_rxn, pert_v);
    standard_passes<kBlock, kF32, kPert, 1>(m, m.rs, LaneView<1>{0u, S.WD}, S.C, g, lane, kGen ? kWave * m.gen_end : 0,
                                            kWave * m.tb_end, m.I, pert_rxn, pert_v);
    wave_sync();
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int k = lane + kWave * s;
        sr.wdot[s] = (k < m.K) ? S.WD[k] : 0.0;
    }
}

// Scalars of the reactor energy equation kept for the Jacobian.
struct RhsScalars {
    double mass, vol, cp_mass, H;   // H = sum_k h_k wdot_k [J/m^3/s] (constant volume: c_v and u_k)
};

// IdealGasConstPressureReactor::eval (src/zeroD/IdealGasConstPressureReactor.cpp)
// or, with m.const_volume, IdealGasReactor::eval (src/zeroD/IdealGasReactor.cpp:50-117,
// closed rigid adiabatic: m c_v dT/dt = -sum_k u_k wdot_k V, u_k = h_k - R T),
// divided by the left-hand sides as ReactorNet::eval does: ydot for the lane's
// components (internal order).  y holds [Y_0..Y_{K-1}, T, m] distributed; P is
// the pressure, or the volume of a constant-volume reactor.
template <int NS, bool kPert = false, int kBlock = 3, bool kGen>
__device__ __forceinline__ void reactor_rhs(const DevMech& m, const Scratch<kGen>& S, double P, const double (&y)[NS],
                                            double (&f)[NS], GasState& g, SpeciesRegs<NS>& sr, RhsScalars& rs,
                                            int pert_rxn = -1, double pert_v = 1.0) {
    const int lane = lane_id();
#pragma unroll
    for (int s = 0; s < NS; s++) {
        int i = lane + kWave * s;
        if (i < m.N) S.yb[i] = y[s];
    }
    wave_sync();
    const double T = uni(S.yb[m.K]);
    const double mass = uni(S.yb[m.K + 1]);
    const bool cv = m.const_volume;
    species_pass<NS>(m, S, T, P, y, g, sr, cv ? mass / P : 0.0);
    production_rates<NS, false, kPert, kBlock>(m, S, g, sr, pert_rxn, pert_v);
    const double vol = cv ? P : mass / g.dens;
    const double hshift = cv ? 1.0 : 0.0;   // u_k / RT = h_k / RT - 1
    double e = 0.0, inner = 0.0;
#pragma unroll
    for (int s = 0; s < NS; s++) {
        int k = lane + kWave * s;
        if (k < m.K) {
            e += sr.wdot[s] * ((sr.hrt[s] - hshift) * g.RT) * vol;
            inner += sr.ym[s] * sr.cpr[s];
        }
    }
    e = uni(wave_sum(e));
    inner = uni(wave_sum(inner));
    // c_p (or c_v = (c_p,mole - R) / Wbar) per unit mass
    const double cp_mass = kGasConstant * (g.mmw * inner - hshift) / g.mmw;
    const double mcpdTdt = -e;
    rs.mass = mass;
    rs.vol = vol;
    rs.cp_mass = cp_mass;
    rs.H = e / vol;
#pragma unroll
    for (int s = 0; s < NS; s++) {
        int i = lane + kWave * s;
        double v = 0.0;
        if (i < m.K) v = (sr.wdot[s] * vol) * m.mw[i] / mass;
        else if (i == m.K) v = mcpdTdt / (mass * cp_mass);
        f[s] = v;
    }
}

// Out-of-line reactor RHS: state taken from S.yb (written by the caller),
// ydot written to S.F.  One copy of the kinetics code serves every call site of
// the integrator (smaller code, and the caller keeps little live across it).
template <int NS, bool kGen>
__device__ __noinline__ void rhs_call(KernargMech* mech, ScratchLayout L, double P) {
    const DevMech m = *(const DevMech*)mech;
    const Scratch<kGen> S = scratch_view<kGen>(L, mech);
    const int lane = lane_id();
    double y[NS], f[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int i = lane + kWave * s;
        y[s] = (i < m.N) ? S.yb[i] : 0.0;
    }
    GasState g;
    SpeciesRegs<NS> sr;
    RhsScalars rs;
    reactor_rhs<NS>(m, S, P, y, f, g, sr, rs);
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int i = lane + kWave * s;
        if (i < m.N) S.F[i] = f[s];
    }
    wave_sync();
}

// rhs_call with reaction pert_rxn (permuted index) at rate multiplier pert_v:
// the perturbed right-hand sides of the sensitivity difference quotients.
template <int NS, bool kGen>
__device__ __noinline__ void rhs_pert_call(KernargMech* mech, ScratchLayout L, double P, int pert_rxn, double pert_v) {
    const DevMech m = *(const DevMech*)mech;
    const Scratch<kGen> S = scratch_view<kGen>(L, mech);
    const int lane = lane_id();
    double y[NS], f[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int i = lane + kWave * s;
        y[s] = (i < m.N) ? S.yb[i] : 0.0;
    }
    GasState g;
    SpeciesRegs<NS> sr;
    RhsScalars rs;
    reactor_rhs<NS, true>(m, S, P, y, f, g, sr, rs, pert_rxn, pert_v);
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int i = lane + kWave * s;
        if (i < m.N) S.F[i] = f[s];
    }
    wave_sync();
}

// Loss frequencies lambda_k = d_k / C_k [1/s] at the state in S.yb (internal
// order, pressure P), left in S.W2[0..K): d_k = sum_i nu'_ki ropf_i +
// nu''_ki ropr_i is the destruction rate of species k
// (Kinetics::getDestructionRates, src/kinetics/Kinetics.cpp:435-445).  Used
// by the surrogate guard to turn a defect of species k into an error estimate.
template <int NS>
__device__ __noinline__ void loss_frequency_call(KernargMech* mech, ScratchLayout L, double P) {
    const DevMech m = *(const DevMech*)mech;
    const WaveScratch S = scratch_view<true>(L, mech);
    const int lane = lane_id();
    double y[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int i = lane + kWave * s;
        y[s] = (i < m.K) ? S.yb[i] : 0.0;
    }
    const double T = S.yb[m.K];
    GasState g;
    SpeciesRegs<NS> sr;
    species_pass<NS>(m, S, T, P, y, g, sr);
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int k = lane + kWave * s;
        if (k < m.K) S.WD[k] = 0.0;
    }
    wave_sync();
    const double kpd = pdep_rate_lane(m, g);
    for (int p = lane; p < m.I; p += kWave) {
        RxnVals v;
        RxnRegs x;
        load_rxn(m, p, x);
        eval_reaction(m, p, g, S.C, S.MU, x, kpd, v);
        const double* gs = (x.gen >= 0) ? m.gend + 12 * x.gen : m.gend;
        const bool rgen = x.flags & 8, pgen = x.flags & 16;
#pragma unroll
        for (int j = 0; j < kMaxSide; j++)
            if (j < x.nr) atomicAdd(&S.WD[x.rk[j]], (rgen ? gs[4 + j] : 1.0) * v.ropf);
#pragma unroll
        for (int j = 0; j < kMaxSide; j++)
            if (j < x.np) atomicAdd(&S.WD[x.pk[j]], (pgen ? gs[8 + j] : 1.0) * v.ropr);
    }
    wave_sync();
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int k = lane + kWave * s;
        if (k < m.K) S.W2[k] = S.WD[k] / fmax(S.C[k], 1e-300);
    }
    wave_sync();
}

}  // namespace cg
