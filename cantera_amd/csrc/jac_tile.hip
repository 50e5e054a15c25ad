// Batched reactor Jacobians of small mechanisms (K <= 62, standard reactions
// only): the quantities and formulas of wave_jac.hpp without atomics on the
// matrix.
//
// One wavefront per state that scatters every reaction's derivatives into an
// LDS matrix (jacobian.hip) spends its time in LDS adds: 400 add instructions
// per gri30 state, each serialised over the lanes that meet in the rows of H,
// O, OH and H2O, and five states per CU compete for them (250k cycles of a SIMD
// each).  Here the derivatives d rop / d C of each reaction are stored once
// (1,275 numbers per gri30 state) and every matrix entry sums its own list of
// them (5.5k terms, prepared with the mechanism): plain loads and multiply-adds
// in a fixed order.  65,536 gri30 states: 6.65 -> 1.43 ms, 1.1 TB/s of the
// matrices themselves; with the lists uncut, a wavefront whose 64 lists wait
// for the diagonal of H (136 terms) made it 2.66 ms.
//
// A workgroup of 4 wavefronts takes kTile = 2 states:
//   1. wavefront w runs the species pass of evaluation w -- states 0 and 1 at
//      T, then at T + dT (the temperature column is a one-sided difference);
//   2. the passes of 16 reactions x 4 evaluations (LaneView<4>) go round the
//      wavefronts; each keeps its own production-rate accumulators, the base
//      evaluations' lanes store the derivatives;
//   3. rates and temperature difference, a wavefront per evaluation;
//   4. the entry lists, cut into pieces of 16 terms and sorted by length so that
//      neighbouring lanes run equally long, two states per table read;
//   5. row and column sums of the chain rule, then whole rows to HBM.
#include <hip/hip_runtime.h>

#include "bdf.hpp"
#include "wave_jac.hpp"

namespace cg {

namespace {

constexpr int kTile = 2, kEval = 4, kWaves = 4, kVec = 64;

// offsets in doubles of the workgroup's LDS
struct JacTileLayout {
    int pairs, dv, mat, vec, coef, total;
    __host__ __device__ JacTileLayout(int K, int nd, int ncoef, int nover) {
        const int rows = K + kDummyWide;
        pairs = 0;
        dv = pairs + 2 * kEval * rows;
        mat = dv + kTile * (nd + 1);
        // the accumulators of step 2 lie in the matrices' area
        const int acc = kWaves * kEval * rows, m = kTile * (K * K + nover);
        vec = mat + (acc > m ? acc : m);
        coef = vec + kVec * (4 * kTile + 3);
        total = coef + ncoef;
    }
};

// one reaction of one evaluation: rate of progress into lv's accumulators,
// derivatives (base evaluations only) into dv, the first slot of this lane's
// state
template <bool kFalloff>
__device__ __forceinline__ void deriv_pass(const DevMech& m, const JacTables& jt, const LaneView<kEval>& lv,
                                           SpeciesColumn<kEval> C, const GasState& g, int p, double* dv, bool base) {
    StdRxn x;
    x.load(m, m.rsw, p);
    const unsigned jd = jt.rxn[p];
    double2 v[6];
#pragma unroll
    for (int e = 0; e < 6; e++) v[e] = lv.pair(x.slot(e));
    double kf, ekc, M = 1.0, qk = 0.0;   // qk: d k / d [M]
    int type = kElementary;
    if constexpr (kFalloff) {
        const int4* qi = reinterpret_cast<const int4*>(m.ri + p);
        const int4 ia = qi[0], ib = qi[1];
        type = (ia.x >> 1) & 3;
        const double4* f4 = reinterpret_cast<const double4*>(m.fod + 8 * (ib.y < 0 ? m.n_fo : ib.y));
        const double4 fa = f4[0], fb = f4[1];
        M = add_mul_rn(efficiency_sum(m, C, ia.w, ib.x), m.tbdef[p], g.ctot);
        double ex[6];
        ex[0] = x.rd.y * g.logT - x.rd.z * g.recipT;
        ex[1] = std_kc_arg(x, g.logC0, v);
        ex[2] = fa.y * g.logT - fa.z * g.recipT;
        ex[3] = troe_arg(-g.T * fb.x);
        ex[4] = troe_arg(-g.T * fb.y);
        ex[5] = troe_arg(-fb.z * g.recipT);
        fast_exp_n(ex);
        ekc = ex[1];
        kf = x.rd.x * ex[0];
        qk = kf;
        if (__any(type >= kLindemann)) {
            const double k0 = fa.x * ex[2];
            double Fcent = (1.0 - fa.w) * ex[3] + fa.w * ex[4];
            Fcent += (fb.z != 0.0) ? opaque(ex[5]) : 0.0;
            Fcent += fb.w * g.T;
            const double lFc = log10(fmax(Fcent, kSmallNumber));
            const double pr = M * k0 / (kf + kSmallNumber);
            const double lpr = log10(fmax(pr, kSmallNumber));
            const double xx = lpr + (-0.4 - 0.67 * lFc), nn = 0.75 - 1.27 * lFc;
            const double den = nn - 0.14 * xx, f1 = xx / den, w = 1.0 + f1 * f1;
            const double Ft = opaque(fast_exp10(lFc / w));
            const double F = (type == kTroe) ? Ft : 1.0;
            const double dl = opaque(-lFc * 2.0 * f1 * (nn / (den * den)) / (w * w));
            const double dlogF = (type == kTroe && pr > kSmallNumber) ? dl : 0.0;
            const double rp = 1.0 / (1.0 + pr);
            const double k0p = k0 * kf / (kf + kSmallNumber);
            const double qf = opaque(k0p * F * rp * (rp + dlogF));
            const double kfo = opaque((pr * (F / (1.0 + pr))) * kf);
            qk = (type >= kLindemann) ? qf : qk;
            kf = (type >= kLindemann) ? kfo : kf;
        }
        const double kM = opaque(kf * M);
        kf = (type == kThreeBody) ? kM : kf;
    } else {
        double ex[2] = {x.rd.y * g.logT - x.rd.z * g.recipT, std_kc_arg(x, g.logC0, v)};
        fast_exp_n(ex);
        kf = x.rd.x * ex[0];
        ekc = ex[1];
    }
    const double r = std_ropnet(x, kf, ekc, v);
    std_scatter(lv, x, r);
    if (__any(x.four_products())) atomicAdd(lv.acc(x.slot(6)), r);
    // derivatives; a reaction's slots: reactants, products (reversible), [M]
    const double rkcn = x.reversible() ? fmin(ekc, kBigNumber) : 0.0;
    const int nr = (jd >> 16) & 7, np = (jd >> 19) & 7, d0 = jd & 0xffff;
    const double kr = -kf * rkcn;
    const double ab = v[0].x * v[1].x, de = v[3].x * v[4].x;
    const double dr[3] = {kf * (v[1].x * v[2].x), kf * (v[0].x * v[2].x), kf * ab};
    const double dp[3] = {kr * (v[4].x * v[5].x), kr * (v[3].x * v[5].x), kr * de};
    if (base) {
#pragma unroll
        for (int e = 0; e < 3; e++) {
            if (e < nr) dv[kTile * (d0 + e)] = dr[e];
            if (e < np) dv[kTile * (d0 + nr + e)] = dp[e];
        }
        if constexpr (kFalloff) {
            const double diff = ab * v[2].x - (x.reversible() ? opaque(rkcn * (de * v[5].x)) : 0.0);
            if (jd >> 22 & 1) dv[kTile * (d0 + nr + np)] = qk * diff;
        }
    }
}

// one term of an entry's list for both states
__device__ __forceinline__ void add_term(const double* coef, const double* dv, unsigned u, double& a0, double& a1) {
    const double c = coef[u >> 16];
    const double2 d = *reinterpret_cast<const double2*>(dv + kTile * (u & 0xffffu));
    a0 = fma(c, d.x, a0);
    a1 = fma(c, d.y, a1);
}

template <typename OT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void jac_tile_kernel(
    DevMech m, JacTables jt, long n, const double* __restrict__ T, const double* __restrict__ P,
    const double* __restrict__ Y, OT* __restrict__ J) {
    const int lane = lane_id(), w = static_cast<int>(threadIdx.x) >> 6;
    const int K = m.K, N = m.N, rows = K + kDummyWide;
    const JacTileLayout L(K, jt.nd, jt.ncoef, jt.nover);
    double* const lds = lds_base();
    double* const dv = lds + L.dv;
    double* const mat = lds + L.mat;
    double* const vec = lds + L.vec;
    double* const coef = lds + L.coef;
    double* const wv = vec + kVec * 4 * kTile;   // W_k, 1 / W_k, then the gas state of evaluation e at 16 e
    double* const gs = wv + 2 * kVec;
    const int ms = K * K + jt.nover;             // doubles between the two states' matrices
    if (threadIdx.x < kVec) {
        const double mw = m.mw[min(static_cast<int>(threadIdx.x), K - 1)];
        wv[threadIdx.x] = mw;
        wv[kVec + threadIdx.x] = 1.0 / mw;
    }
    for (int i = threadIdx.x; i < jt.ncoef; i += 256) coef[i] = jt.coef[i];
    for (int i = threadIdx.x; i < kEval * kDummyWide; i += 256)
        *reinterpret_cast<double2*>(lds + 2 * (kEval * K + i)) = double2{1.0, 0.0};
    if (threadIdx.x < kTile) dv[kTile * jt.nd + threadIdx.x] = 0.0;   // the padding entries' slot
    const long tiles = (n + kTile - 1) / kTile;
    const XcdStates xs(tiles);
    for (long tile = xs.lo; tile < xs.hi; tile += xs.step) {
        // 1. species pass of evaluation w: state w % 2, at T + dT for w >= 2
        const int ts = w % kTile;
        const long st = tile * kTile + ts, sc = min(st, n - 1);
        const double T0 = uni(T[sc]), Ps = uni(P[sc]);
        const double dT = kSqrtEps * T0;
        const double yk = (lane < K) ? Y[static_cast<size_t>(lane) * n + sc] : 0.0;
        GasState g;
        SpeciesRegs<1> sr;
        g.T = w < kTile ? T0 : T0 + dT;
        g.RT = g.T * kGasConstant;
        g.recipT = 1.0 / g.T;
        sr.ym[0] = (lane < K) ? yk * m.rmw[lane] : 0.0;
        g.mmw = 1.0 / uni(wave_sum(sr.ym[0]));
        g.dens = Ps * g.mmw / g.RT;
        g.ctot = g.dens / g.mmw;
        g.pressure = kGasConstant * g.ctot * g.T;
        const double lg = log(lane == 0 ? g.T : (lane == 1 ? g.ctot : g.pressure * m.rpref));
        g.logT = readlane_f64(lg, 0);
        g.logC0 = readlane_f64(lg, 1);
        const double lnp = readlane_f64(lg, 2);
        const double tt[6] = {g.T, g.T * g.T, g.T * g.T * g.T, g.T * g.T * g.T * g.T, g.recipT, g.logT};
        const int kc = min(lane, K - 1);
        double sR, g0;
        nasa7(m.nasa + 16 * kc, g.T, tt, sr.cpr[0], sr.hrt[0], sR, g0);
        if (lane < K) *reinterpret_cast<double2*>(lds + 2 * (kEval * lane + w)) = double2{sr.ym[0] * g.dens, g0 + lnp};
        if (lane == 0) {
            double* o = gs + 16 * w;
            o[0] = g.T; o[1] = g.logT; o[2] = g.recipT; o[3] = g.logC0; o[4] = g.ctot;
        }
        for (int i = lane; i < kEval * rows; i += kWave) mat[w * kEval * rows + i] = 0.0;
        __syncthreads();
        // 2. reactions
        {
            const int e = lane % kEval, j = lane / kEval;
            constexpr int G = LaneView<kEval>::kStride;
            const double* o = gs + 16 * e;
            GasState ge;
            ge.T = o[0]; ge.logT = o[1]; ge.recipT = o[2]; ge.logC0 = o[3]; ge.ctot = o[4];
            LaneView<kEval> lv;
            lv.pair0 = 16u * e;
            lv.wd = mat + w * kEval * rows + e;
            const SpeciesColumn<kEval> C{lds + 2 * e};
            double* const dve = dv + e % kTile;
            int q = w * G;
            for (; q < m.n_nonplain; q += kWaves * G) deriv_pass<true>(m, jt, lv, C, ge, q + j, dve, e < kTile);
            for (; q < m.I; q += kWaves * G) deriv_pass<false>(m, jt, lv, C, ge, q + j, dve, e < kTile);
        }
        __syncthreads();
        // 3. rates of evaluation w (fixed order over the wavefronts' shares)
        double wd = 0.0;
        if (lane < K)
#pragma unroll
            for (int u = 0; u < kWaves; u++) wd += mat[(u * rows + lane) * kEval + w];
        const double mw = m.mw[kc];
        const double hk = sr.hrt[0] * g.RT;
        const double vol = 1.0 / g.dens;
        const double cp = kGasConstant * (g.mmw * uni(wave_sum(sr.ym[0] * sr.cpr[0]))) / g.mmw;
        const double eT = uni(wave_sum(lane < K ? wd * hk * vol : 0.0));
        // right-hand side, [Y.., T] in lanes 0..K
        const double f = lane < K ? (wd * vol) * mw : (lane == K ? -eT / cp : 0.0);
        double* const hkv = vec + kVec * ts;                  // h_k
        double* const ckv = vec + kVec * (kTile + ts);        // (wdot_k - D_k) / C_tot
        double* const hjv = vec + kVec * (2 * kTile + ts);    // sum_k h_k JC_kj, then the T row
        double* const ftv = vec + kVec * (3 * kTile + ts);    // f(T + dT), then the T column
        if (w < kTile) {
            hkv[lane] = lane < K ? hk : 0.0;
        } else {
            ftv[lane] = f;
        }
        __syncthreads();
        if (w < kTile) ftv[lane] = (ftv[lane] - f) / dT;
        // 4. matrix entries
        for (int i = 0; i < jt.groups; i++) {
            const int2 seg = jt.seg[kWaves * i + w];   // first table row, rows
            const int pos = jt.pos[256 * i + threadIdx.x];
            const unsigned* t = jt.ell + static_cast<size_t>(seg.x) * kWave + lane;
            double a0 = 0.0, a1 = 0.0;
            int r = 0;
            for (; r + 4 <= seg.y; r += 4) {
                unsigned u[4];
#pragma unroll
                for (int b = 0; b < 4; b++) u[b] = t[(r + b) * kWave];
#pragma unroll
                for (int b = 0; b < 4; b++) add_term(coef, dv, u[b], a0, a1);
            }
            for (; r < seg.y; r++) add_term(coef, dv, t[r * kWave], a0, a1);
            if (pos != 0xffff) {
                mat[pos] = a0;
                mat[ms + pos] = a1;
            }
        }
        __syncthreads();
        // entries in several pieces
        if (w == kWaves - 1) {
            int over = K * K;
            for (int i0 = 0; i0 < jt.nsplit; i0 += kWave) {
                const int2 sp = i0 + lane < jt.nsplit ? jt.split[i0 + lane] : int2{0, 0};
                // exclusive scan of the piece counts
                int inc = sp.y;
#pragma unroll
                for (int d = 1; d < kWave; d <<= 1) {
                    const int o = __shfl_up(inc, d);
                    if (lane >= d) inc += o;
                }
                const int at = over + inc - sp.y;
                over += __shfl(inc, kWave - 1);
                double a0 = 0.0, a1 = 0.0;
                for (int t = 0; t < sp.y; t++) {
                    a0 += mat[at + t];
                    a1 += mat[ms + at + t];
                }
                if (sp.y > 0) {
                    mat[sp.x] += a0;
                    mat[ms + sp.x] += a1;
                }
            }
        }
        __syncthreads();
        // 5. chain rule to mass fractions at fixed T and P (reactor_jacobian)
        const double* A = mat + ts * ms;
        double D = 0.0;
        if (w < kTile) {
#pragma unroll 8
            for (int l = 0; l < K; l++) D += A[kc * K + l] * lds[2 * (kEval * l + ts)];
            if (lane < K) ckv[lane] = (wd - D) / g.ctot;
        } else {
            double s = 0.0;
#pragma unroll 8
            for (int k = 0; k < K; k++) s += hkv[k] * A[k * K + kc];
            hjv[lane] = s;
        }
        __syncthreads();
        if (w < kTile) {
            const double hD = uni(wave_sum(lane < K ? hk * D : 0.0));
            const double H = uni(wave_sum(lane < K ? hk * wd : 0.0));
            const double cpj = kGasConstant * sr.cpr[0] / mw;
            const double hj = hjv[lane];
            if (lane < K)
                hjv[lane] = -1.0 / (g.dens * cp) * ((g.dens * hj - g.mmw * hD + g.mmw * H) / mw - H * cpj / cp);
        }
        __syncthreads();
        // rows of state ts: wavefronts ts and ts + 2 take alternate rows
        if (st < n) {
            OT* const Js = J + static_cast<size_t>(st) * N * N;
            const int cj = min(max(lane - 2, 0), K - 1);
            const double wi = wv[kVec + cj];
            OT* o = Js + lane;
            if (w < kTile) {   // the mass row, then even species rows
                if (lane < N) o[0] = static_cast<OT>(0.0);
            } else if (lane < N) {   // the temperature row, then odd species rows
                o[N] = static_cast<OT>(lane >= 2 ? hjv[cj] : (lane == 1 ? ftv[K] : 0.0));
            }
#pragma unroll 4
            for (int k = w / kTile; k < K; k += kWaves / kTile) {
                const double jc = wv[k] * wi * (A[k * K + cj] + ckv[k]);
                const double jt1 = lane == 1 ? ftv[k] : 0.0;   // column 0 is zero at any state, column 1 d / dT
                if (lane < N) o[(k + 2) * N] = static_cast<OT>(lane >= 2 ? jc : jt1);
            }
        }
        __syncthreads();
    }
}

}  // namespace

size_t jac_tile_lds_bytes(const DevMech& m, const JacTables& jt) {
    return static_cast<size_t>(JacTileLayout(m.K, jt.nd, jt.ncoef, jt.nover).total) * sizeof(double);
}

const void* jac_tile_kernel_ptr(bool f32) {
    return f32 ? reinterpret_cast<const void*>(&jac_tile_kernel<float>)
               : reinterpret_cast<const void*>(&jac_tile_kernel<double>);
}

long jac_tile_items(long n) { return (n + kTile - 1) / kTile; }

hipError_t jac_tile_launch(const DevMech& m, const JacTables& jt, bool f32, long n, const double* T, const double* P,
                           const double* Y, void* J, int grid, size_t lds, hipStream_t stream) {
    if (f32)
        hipLaunchKernelGGL(jac_tile_kernel<float>, dim3(grid), dim3(256), lds, stream, m, jt, n, T, P, Y,
                           static_cast<float*>(J));
    else
        hipLaunchKernelGGL(jac_tile_kernel<double>, dim3(grid), dim3(256), lds, stream, m, jt, n, T, P, Y,
                           static_cast<double*>(J));
    return hipGetLastError();
}

}  // namespace cg
