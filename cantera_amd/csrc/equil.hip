// Batched chemical equilibrium of ideal-gas states at fixed (h, P) or (T, P)
// (ThermoPhase::equilibrate("HP" / "TP"), src/thermo/ThermoPhase.cpp, whose
// default solver for a single ideal-gas phase is the element-potential method
// of ChemEquil, src/equil/ChemEquil.cpp:329-337).
//
// Method: Gibbs-energy minimisation with element potentials, the Newton
// iteration of Gordon & McBride (NASA RP-1311, 1994, eqs. 2.24-2.27 for a gas
// phase) with its step control (eqs. 3.1-3.3).  Unknowns per iteration are the
// element potentials pi_e, dln n (n = total kmol per kg) and, for HP, dln T;
// species follow as dln n_j = -mu_j/RT + sum_e a_ej pi_e + dln n + h_j dln T.
// Elements absent from a state, and the species containing them, are left
// out.  Convergence: every correction below 1e-12 (species: relative to the
// total).
//
// Layout: inputs and outputs species-major as the batched rates (T[n], P[n],
// Y[k*n + s]).  One wavefront per state: lane k owns species k (slot s for
// k = lane + 64 s), with its element counts and, for one slot, its NASA
// coefficients in registers for the whole kernel.  The Newton matrix and right-hand side are entries of
// one contraction G = V^T diag(n) V over the species with V's columns the
// element counts, 1, h/RT, mu/RT and cp/R (E + 4 <= 12): V goes to LDS and
// v_mfma_f64_16x16x4f64 sums four species at a time.  The (E+2) x (E+2)
// system is solved row per lane in registers (solve_rows).  (As wavefront
// sums, 36 per iteration for 5 elements, with the system eliminated by one
// lane in LDS, 20,011 gri30 states took 3.7 ms; HBM traffic is the state in
// and out.)  Two wavefronts per SIMD in both registers and LDS: 12,000
// n-dodecane states TP 1.29 ms, HP 1.45 (one per SIMD 1.85 and 2.08, wavefront
// sums 1.53 and 2.03).
#include <hip/hip_runtime.h>

#include "bdf.hpp"
#include "wave_linalg.hpp"

namespace cg {

namespace {

constexpr int kEqMaxE = 8;
constexpr int kEqMaxNu = kEqMaxE + 2;
constexpr double kSize = 18.420681;       // ln(1e8): trace-species threshold of eq. 3.2
constexpr double kTraceLn = 9.2103404;    // ln(1e4)

// x <- A^-1 x, row q of A and of x in lane q < nu; false where A is singular.
// Gaussian elimination with the exact largest pivot of a column and with
// quotients by it (a product by the reciprocal and a correction by its
// remainder, so exact where the quotient is): an iterate of almost one species
// makes element rows multiples of each other, and a quotient keeps the zero that
// they cancel to.  With bare products by 1 / pivot and pivots compared in 58
// bits that zero became a pivot of rounding noise or not as it fell, and 0.07%
// of hydrogen mixtures at 200 to 500 K were refused that are not now.  20,011
// gri30 states 1.99 -> 1.93 ms (2.04 with divisions).
__device__ __forceinline__ bool solve_rows(double (&a)[kEqMaxNu], double& x, int nu) {
    const int lane = lane_id();
    bool open = lane < nu;   // not a pivot row yet
    int step = kEqMaxNu;     // the column that this lane's row is the pivot of
    double rdiag = 0.0;
    int owner[kEqMaxNu];
#pragma unroll
    for (int c = 0; c < kEqMaxNu; c++) {
        owner[c] = 0;
        if (c >= nu) continue;
        const double v = open ? fabs(a[c]) : -1.0;
        double top = fmax(v, dpp_f64<0xB1>(v));
        top = fmax(top, dpp_f64<0x4E>(top));
        top = fmax(top, dpp_f64<0x124>(top));
        top = readlane_f64(fmax(top, dpp_f64<0x128>(top)), 0);
        const unsigned long long same = __ballot(v == top);
        if (!(top > 0.0) || same == 0) return false;
        const int p = owner[c] = __builtin_ctzll(same);
        const double piv = readlane_f64(a[c], p);
        double rp = __builtin_amdgcn_rcp(piv);
        rp = fma(fma(-piv, rp, 1.0), rp, rp);
        rp = fma(fma(-piv, rp, 1.0), rp, rp);
        if (lane == p) {
            open = false;
            step = c;
            rdiag = rp;
        }
        const double q0 = a[c] * rp, q = fma(fma(-q0, piv, a[c]), rp, q0);
        const double f = open ? q : 0.0;
#pragma unroll
        for (int j = c + 1; j < kEqMaxNu; j++) a[j] -= f * readlane_f64(a[j], p);
        x -= f * readlane_f64(x, p);
    }
    double y = 0.0;
#pragma unroll
    for (int c = kEqMaxNu - 1; c >= 0; c--) {
        if (c >= nu) continue;
        const double xc = readlane_f64(x * rdiag, owner[c]);
        x -= (step < c ? a[c] : 0.0) * xc;
        y = lane == c ? xc : y;
    }
    x = y;
    return true;
}

template <int NS>
__global__ __launch_bounds__(64) void equil_kernel(DevMech m, long n, int hp, const double* __restrict__ Tin,
                                                   const double* __restrict__ Pin, const double* __restrict__ Yin,
                                                   double* __restrict__ Tout, double* __restrict__ Yout,
                                                   int* __restrict__ info, int max_iter) {
    // NASA coefficients in registers for one species per lane; for two they come
    // from L1 each time (28 registers a slot that made it one wavefront per SIMD)
    constexpr bool kHold = NS == 1;
    // columns of V: elements 0 .. E-1, then 1, h, mu, cp, then zero; odd strides,
    // so that a column of lanes and a row of columns are both free of bank
    // conflicts.  With 15.7 KB for two slots (20.6 with all 16 columns of the
    // product) LDS leaves room for two wavefronts per SIMD, as the registers do.
    constexpr int kCols = 13;
    __shared__ double Vs[kWave * NS * kCols];
    __shared__ double ns[kWave * NS];
    __shared__ double Gs[kCols * kCols];
    const int lane = lane_id();
    const int K = m.K, E = m.E;
    const int cOne = E, cH = E + 1, cMu = E + 2, cCp = E + 3;
    const int nu = E + 1 + (hp ? 1 : 0);
    // the lane's species
    double cl[kHold ? NS : 1][7], ch[kHold ? NS : 1][7], tmid[NS], el[NS][kEqMaxE], rmw[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int k = lane + kWave * s, kc = min(k, K - 1);
        const double* c16 = m.nasa + 16 * kc;
        if constexpr (kHold)
#pragma unroll
            for (int j = 0; j < 7; j++) {
                cl[s][j] = c16[j];
                ch[s][j] = c16[8 + j];
            }
        tmid[s] = c16[7];
        rmw[s] = m.rmw[kc];
#pragma unroll
        for (int e = 0; e < kEqMaxE; e++) el[s][e] = (k < K && e < E) ? m.comp[kc * E + e] : 0.0;
#pragma unroll
        for (int c = 0; c < kCols; c++) Vs[k * kCols + c] = 0.0;
#pragma unroll
        for (int e = 0; e < kEqMaxE; e++)
            if (e < E) Vs[k * kCols + e] = el[s][e];
        Vs[k * kCols + cOne] = 1.0;
        ns[k] = 0.0;
    }
    wave_sync();
    auto thermo = [&](int s, double T, double recipT, double logT, double& cp, double& h, double& g) {
        const bool low = T <= tmid[s];
        double c[7];
        const double* c7 = m.nasa + 16 * min(lane + kWave * s, K - 1) + (low ? 0 : 8);
#pragma unroll
        for (int j = 0; j < 7; j++) {
            if constexpr (kHold) c[j] = low ? cl[s][j] : ch[s][j];
            else c[j] = c7[j];
        }
        const double ct1 = c[1] * T, ct2 = c[2] * (T * T), ct3 = c[3] * (T * T * T), ct4 = c[4] * (T * T * T * T);
        cp = c[0] + ct1 + ct2 + ct3 + ct4;
        h = c[0] + 0.5 * ct1 + 1.0 / 3.0 * ct2 + 0.25 * ct3 + 0.2 * ct4 + c[5] * recipT;
        g = h - (c[0] * logT + ct1 + 0.5 * ct2 + 1.0 / 3.0 * ct3 + 0.25 * ct4 + c[6]);
    };
    const XcdStates xst(n);
    for (long st = xst.lo; st < xst.hi; st += xst.step) {
        const double T0 = uni(Tin[st]);
        const double P = uni(Pin[st]);
        // element amounts [kmol/kg] and specific enthalpy of the input state
        double hl = 0.0, ny[NS];
        const double rT0 = 1.0 / T0, lT0 = log(T0);
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int k = lane + kWave * s;
            ny[s] = 0.0;
            if (k < K) {
                double cp, h, g;
                ny[s] = Yin[static_cast<size_t>(k) * n + st] * rmw[s];
                thermo(s, T0, rT0, lT0, cp, h, g);
                hl += ny[s] * h;
            }
        }
        const double h0 = uni(wave_sum(hl)) * kGasConstant * T0;
        double b0[kEqMaxE];
        double bmax = 0.0;
#pragma unroll
        for (int e = 0; e < kEqMaxE; e++) {
            double v = 0.0;
            if (e < E) {
#pragma unroll
                for (int s = 0; s < NS; s++) v += el[s][e] * ny[s];
                v = uni(wave_sum(v));
            }
            b0[e] = v;
            bmax = fmax(bmax, v);
        }
        unsigned emask = 0;
#pragma unroll
        for (int e = 0; e < kEqMaxE; e++)
            if (e < E && b0[e] > 1e-14 * bmax) emask |= 1u << e;
        // this lane's row of the system: element, ln n or ln T; its
        // right-hand side b_q (elements)
        const bool elem = lane < E && ((emask >> lane) & 1u);
        const bool row_on = elem || lane == cOne || (hp && lane == cH);
        double bq0 = 0.0;
#pragma unroll
        for (int e = 0; e < kEqMaxE; e++) bq0 = (lane == e) ? b0[e] : bq0;
        bool act[NS];
        double lnn[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) {
            bool a = lane + kWave * s < K;
#pragma unroll
            for (int e = 0; e < kEqMaxE; e++)
                if (!((emask >> e) & 1u) && el[s][e] != 0.0) a = false;
            act[s] = a;
            lnn[s] = a ? log(0.1 / K) : 0.0;
        }
        double lnntot = log(0.1);
        double T = hp ? 3800.0 : T0;
        const double lnP = log(P / m.pref);
        int status = -1, it = 0;
        for (; it < max_iter; it++) {
            const double recipT = 1.0 / T, logT = log(T);
            double nj[NS], mu[NS], hj[NS];
#pragma unroll
            for (int s = 0; s < NS; s++) {
                double cp, h, g;
                thermo(s, T, recipT, logT, cp, h, g);
                hj[s] = act[s] ? h : 0.0;
                mu[s] = act[s] ? g + (lnn[s] - lnntot) + lnP : 0.0;
                nj[s] = act[s] ? fast_exp(lnn[s]) : 0.0;
                const int k = lane + kWave * s;
                Vs[k * kCols + cH] = hj[s];
                Vs[k * kCols + cMu] = mu[s];
                Vs[k * kCols + cCp] = act[s] ? cp : 0.0;
                ns[k] = nj[s];
            }
            const double ntot = fast_exp(lnntot);
            wave_sync();
            // lane l holds V(k, l % 16), k = 4 c + l / 16, as left and, times
            // n_k, as right operand; two accumulators break the chain
            mfma_d4 acc0 = {0.0, 0.0, 0.0, 0.0}, acc1 = {0.0, 0.0, 0.0, 0.0};
            {
                const int kq = lane >> 4, lr = min(lane & 15, kCols - 1);   // spare lanes: a zero column
                for (int k0 = 0; k0 < K; k0 += 8) {   // rows past K are zero
                    const int ka = k0 + kq, kb = k0 + 4 + kq;
                    const double va = Vs[ka * kCols + lr], na = ns[ka], vb = Vs[kb * kCols + lr], nb = ns[kb];
                    acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(va, na * va, acc0, 0, 0, 0);
                    acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(vb, nb * vb, acc1, 0, 0, 0);
                }
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (kq + 4 * r < kCols) Gs[(kq + 4 * r) * kCols + lr] = acc0[r] + acc1[r];
            }
            wave_sync();
            double a[kEqMaxNu];
            const int row = min(lane, nu - 1);
            const double sumn = uni(Gs[cOne * kCols + cOne]);
#pragma unroll
            for (int j = 0; j < kEqMaxNu; j++) {
                double v = Gs[row * kCols + min(j, nu - 1)];
                if (j == lane) {
                    v -= (lane == cOne) ? ntot : 0.0;
                    v += (lane == cH) ? Gs[cOne * kCols + cCp] : 0.0;
                }
                // an element that the state lacks: 1 on the diagonal, 0 elsewhere
                a[j] = (lane < nu && j < nu) ? (row_on ? v : (j == lane ? 1.0 : 0.0)) : 0.0;
            }
            double x;
            {
                const double gmu = Gs[row * kCols + cMu], gone = Gs[row * kCols + cOne];
                const double lead = elem ? bq0 : (lane == cOne ? ntot : h0 / (kGasConstant * T));
                x = row_on ? lead - gone + gmu : 0.0;
            }
            const bool ok = solve_rows(a, x, nu);
            if (!ok || __any(lane < nu && !(x == x))) { status = -3; break; }
            const double dlnN = readlane_f64(x, cOne), dlnT = hp ? readlane_f64(x, cH) : 0.0;
            double pi[kEqMaxE];
#pragma unroll
            for (int e = 0; e < kEqMaxE; e++) pi[e] = readlane_f64(x, e);
            double d[NS];
            double l_big = 0.0, l_conv = 0.0, l_lam2 = 1.0;
#pragma unroll
            for (int s = 0; s < NS; s++) {
                d[s] = 0.0;
                if (act[s]) {
                    double v = -mu[s] + dlnN + hj[s] * dlnT;
#pragma unroll
                    for (int e = 0; e < kEqMaxE; e++) v += (e < E) ? el[s][e] * pi[e] : 0.0;
                    d[s] = v;
                    const double lnx = lnn[s] - lnntot;
                    if (lnx > -kSize) {
                        l_big = fmax(l_big, v);
                        l_conv = fmax(l_conv, nj[s] / sumn * fabs(v));
                    } else if (v >= 0.0 && v - dlnN != 0.0) {
                        l_lam2 = fmin(l_lam2, fabs((-lnx - kTraceLn) / (v - dlnN)));
                    }
                }
            }
            wave_sync();
            const double big = fmax(fmax(5.0 * fabs(dlnT), 5.0 * fabs(dlnN)), uni(wave_max(l_big)));
            const double conv = fmax(fmax(fabs(dlnT), fabs(dlnN)), uni(wave_max(l_conv)));
            const double lam2 = -uni(wave_max(-l_lam2));
            double lam = fmin(1.0, lam2);
            if (big > 2.0) lam = fmin(lam, 2.0 / big);
#pragma unroll
            for (int s = 0; s < NS; s++)
                if (act[s]) lnn[s] += lam * d[s];
            lnntot += lam * dlnN;
            if (hp) T = fmin(fmax(T * fast_exp(lam * dlnT), 200.0), 6000.0);
            if (lam == 1.0 && conv < 1e-12) { status = 0; it++; break; }
        }
        double yo[NS], ysum = 0.0;
#pragma unroll
        for (int s = 0; s < NS; s++) {
            yo[s] = act[s] ? exp(lnn[s]) / rmw[s] : 0.0;
            ysum += yo[s];
        }
        ysum = uni(wave_sum(ysum));
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int k = lane + kWave * s;
            if (k < K) Yout[static_cast<size_t>(k) * n + st] = yo[s] / ysum;
        }
        if (lane == 0) {
            Tout[st] = T;
            if (info) info[st] = status == 0 ? it : status;
        }
        wave_sync();
    }
}

}  // namespace

hipError_t equil_launch(const DevMech& m, int ns, int hp, long n, const double* T, const double* P, const double* Y,
                        double* Tout, double* Yout, int* info, int max_iter, int grid, hipStream_t stream) {
    if (m.E > kEqMaxE) return hipErrorInvalidValue;
    if (ns == 1)
        hipLaunchKernelGGL((equil_kernel<1>), dim3(grid), dim3(64), 0, stream, m, n, hp, T, P, Y, Tout, Yout, info,
                           max_iter);
    else if (ns == 2)
        hipLaunchKernelGGL((equil_kernel<2>), dim3(grid), dim3(64), 0, stream, m, n, hp, T, P, Y, Tout, Yout, info,
                           max_iter);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

const void* equil_kernel_ptr(int ns) {
    return ns == 1 ? reinterpret_cast<const void*>(&equil_kernel<1>) : reinterpret_cast<const void*>(&equil_kernel<2>);
}

}  // namespace cg
