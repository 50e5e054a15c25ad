// MLP surrogate kernels: BF16 MFMA GEMM with fused epilogues, features and
// targets from FP64 reactor states, loss, Adam.  See surrogate.hpp.
#include "surrogate.hpp"

#include "wave_kinetics.hpp"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <random>
#include <stdexcept>
#include <string>

namespace cg {

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// round to nearest even (v_cvt_pk_bf16_f32); NaN stays NaN
__device__ __forceinline__ uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f)); }

// GELU, tanh form (Hendrycks & Gimpel 2016), and its derivative.
constexpr float kGeluC = 0.7978845608028654f;   // sqrt(2/pi)
constexpr float kGeluA = 0.044715f;
// 0.5 (1 + tanh u) = 1 / (1 + exp(-2u)): one hardware exponential and one
// reciprocal (1 ulp each) instead of tanhf's ~30 instructions, which took
// longer than a 256-wide layer's matrix products.  With t = exp(-2|u|) and
// r = 1 / (1 + t), gelu(z) = max(z, 0) - |z| t r and the derivative of the
// gate is t r^2 times that of 2u, both without cancellation.  Over |z| <= 12,
// exponential and reciprocal each off by an ulp,
// the largest errors against 64 bits are 2.4e-7 and 3.8e-7 (with tanhf 4.7e-7
// and 1.2e-6), the RMS errors 4e-8 and 1e-7 (6e-8 and 1.9e-7).
constexpr float kGelu1 = 2.0f * kGeluC, kGelu3 = 2.0f * kGeluC * kGeluA, kLog2e = 1.4426950408889634f;
struct Gate { float t, r; };
__device__ __forceinline__ Gate gelu_gate(float z) {
    const float w = fabsf(z) * fmaf(z * z, kGelu3 * kLog2e, kGelu1 * kLog2e);   // 2|u| log2(e)
    const float t = __builtin_amdgcn_exp2f(-w);
    return {t, __builtin_amdgcn_rcpf(1.0f + t)};
}
__device__ __forceinline__ float gelu(float z) {
    const Gate g = gelu_gate(z);
    return fmaf(-fminf(fabsf(z), 1e30f), g.t * g.r, fmaxf(z, 0.0f));   // 1e30: no inf * 0
}
__device__ __forceinline__ float gelu_grad(float z) {
    const Gate g = gelu_gate(z);
    const float tr = g.t * g.r;
    return fmaf(z * (tr * g.r), fmaf(z * z, 3.0f * kGelu3, kGelu1), z >= 0.0f ? g.r : tr);
}

enum Epi { kFwdGelu, kFwdLinear, kBwdGelu };

struct EpiArgs {
    const float* bias;   // kFwdGelu / kFwdLinear: [N]
    float* zf;           // kFwdGelu: pre-activation out; kFwdLinear: fp32 out
    uint16_t* hb;        // kFwdGelu: gelu(z) as bf16; kBwdGelu: acc * gelu'(zin) as bf16
    const float* zin;    // kBwdGelu: pre-activation of the layer below
    int ldc;
};

constexpr int kTM = 64, kTN = 64, kTK = 32, kLdsK = kTK + 8;

// C(m, n) = sum_k A(m, k) B(n, k) over BF16 operands, FP32 accumulation.
// A(m, k) = A[m * K + k];  B(n, k) = B[n * K + k], for kBwdGelu B[k * N + n].
// Any size: the layers that gemm_direct and gemm_nt_bf16 do not take.
// 256 threads: a 64 x 64 tile of C per workgroup, 32 x 32 per wavefront as
// 2 x 2 MFMA 16x16x16 tiles; K staged through LDS in steps of 32.  Out-of-range
// rows / columns / k read as zero and are not stored.
template <int EPI>
__global__ __launch_bounds__(256) void gemm_bf16(int M, int N, int K, const uint16_t* __restrict__ A,
                                                 const uint16_t* __restrict__ B, EpiArgs e) {
    constexpr bool TB = EPI == kBwdGelu;
    __shared__ uint16_t As[kTM][kLdsK];
    __shared__ uint16_t Bs[kTN][kLdsK];
    const int t = threadIdx.x;
    const int lane = t & 63, w = t >> 6;
    const int m0 = blockIdx.x * kTM, n0 = blockIdx.y * kTN;
    const int wm = (w >> 1) * 32, wn = (w & 1) * 32;
    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < K; k0 += kTK) {
        // stage A (64 x 32) and B (64 x 32), 8 elements per thread each
        {
            const int r = t >> 2, kk = (t & 3) * 8;
            const int m = m0 + r;
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const int k = k0 + kk + q;
                As[r][kk + q] = (m < M && k < K) ? A[static_cast<size_t>(m) * K + k] : 0;
            }
        }
        if (!TB) {
            const int r = t >> 2, kk = (t & 3) * 8;
            const int n = n0 + r;
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const int k = k0 + kk + q;
                Bs[r][kk + q] = (n < N && k < K) ? B[static_cast<size_t>(n) * K + k] : 0;
            }
        } else {
            const int kk = t >> 3, rr = (t & 7) * 8;
            const int k = k0 + kk;
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const int n = n0 + rr + q;
                Bs[rr + q][kk] = (n < N && k < K) ? B[static_cast<size_t>(k) * N + n] : 0;
            }
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < kTK; ks += 16) {
            bf16x4 a[2], b[2];
            const int kq = ks + 4 * (lane >> 4);
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const uint16_t* pa = &As[wm + 16 * i + (lane & 15)][kq];
                const uint16_t* pb = &Bs[wn + 16 * i + (lane & 15)][kq];
                a[i] = bf16x4{static_cast<short>(pa[0]), static_cast<short>(pa[1]), static_cast<short>(pa[2]),
                              static_cast<short>(pa[3])};
                b[i] = bf16x4{static_cast<short>(pb[0]), static_cast<short>(pb[1]), static_cast<short>(pb[2]),
                              static_cast<short>(pb[3])};
            }
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
    // D(16x16) lane layout: row 4 * (lane / 16) + r, column lane % 16
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + wm + 16 * i + 4 * (lane >> 4) + r;
                const int n = n0 + wn + 16 * j + (lane & 15);
                if (m >= M || n >= N) continue;
                const float v = acc[i][j][r];
                const size_t o = static_cast<size_t>(m) * e.ldc + n;
                if (EPI == kFwdGelu) {
                    const float z = v + e.bias[n];
                    if (e.zf) e.zf[o] = z;      // pre-activation kept for training only
                    e.hb[o] = f2bf(gelu(z));
                } else if (EPI == kFwdLinear) {
                    e.zf[o] = v + e.bias[n];
                } else {
                    e.hb[o] = f2bf(v * gelu_grad(e.zin[o]));
                }
            }
}

// Features of row idx[r] (or r): T, ln P, ln max(Y_k, 1e-30), normalised and
// clipped to [-8, 8]; padding columns zero.
__global__ void features_kernel(int rows, const int* __restrict__ idx, int N, int K, const double* __restrict__ y,
                                const double* __restrict__ P, const double* __restrict__ norm, int in_p,
                                uint16_t* __restrict__ X) {
    const int r = blockIdx.x;
    if (r >= rows) return;
    const long s = idx ? idx[r] : r;
    const double* yr = y + s * N;
    for (int j = threadIdx.x; j < in_p; j += blockDim.x) {
        double f = 0.0;
        if (j == 0) f = yr[1];
        else if (j == 1) f = log(P[s]);
        else if (j < 2 + K) f = log(fmax(yr[j], 1e-30));
        float v = 0.f;
        if (j < 2 + K) {
            double z = (f - norm[j]) / norm[in_p + j];
            v = static_cast<float>(fmin(fmax(z, -8.0), 8.0));
        }
        X[static_cast<size_t>(r) * in_p + j] = f2bf(v);
    }
}

// Mean-squared error over the n_out valid outputs, gradient as BF16 operand.
// Targets are the increments d = (T1 - T0, Y1_k - Y0_k), compressed as
// asinh(d / s) (linear below the scale s, logarithmic above, so small and large
// increments get comparable relative accuracy), then standardised.  Each block
// leaves its part of the loss in loss[1 + block]; grad_sum_kernel adds them.
constexpr int kLossBlocks = 256;
__global__ __launch_bounds__(256) void loss_kernel(int rows, const int* __restrict__ idx, int N, int n_out, int in_p,
                                                   int out_p, const double* __restrict__ y0,
                                                   const double* __restrict__ y1, const double* __restrict__ norm,
                                                   const float* __restrict__ out, uint16_t* __restrict__ g,
                                                   double* __restrict__ loss) {
    __shared__ double part[256];
    double acc = 0.0;
    const double scale = 1.0 / (static_cast<double>(rows) * n_out);
    const double* mu = norm + 2 * in_p;
    const double* sd = mu + out_p;
    const double* sc = sd + out_p;
    const size_t total = static_cast<size_t>(rows) * out_p;
    for (size_t i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const int j = static_cast<int>(i % out_p);
        float gv = 0.f;
        if (j < n_out) {
            const size_t r = i / out_p, e = (idx ? idx[r] : r) * N + 1 + j;
            const float tgt = static_cast<float>((asinh((y1[e] - y0[e]) / sc[j]) - mu[j]) / sd[j]);
            const float d = out[i] - tgt;
            acc += static_cast<double>(d) * d;
            gv = static_cast<float>(2.0 * scale) * d;
        }
        g[i] = f2bf(gv);
    }
    part[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) part[threadIdx.x] += part[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) loss[1 + blockIdx.x] = part[0] * scale;
}

// Adam (Kingma & Ba 2015) with bias correction, then the BF16 weight copy.
__global__ void adam_kernel(size_t n, float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m1,
                            float* __restrict__ m2, uint16_t* __restrict__ wb, float lr, float c1, float c2) {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    for (size_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const float gi = g[i];
        const float a = b1 * m1[i] + (1.f - b1) * gi;
        const float b = b2 * m2[i] + (1.f - b2) * gi * gi;
        m1[i] = a;
        m2[i] = b;
        const float wi = w[i] - lr * (a / c1) / (sqrtf(b / c2) + eps);
        w[i] = wi;
        wb[i] = f2bf(wi);
    }
}

__global__ void to_bf16_kernel(size_t n, const float* __restrict__ w, uint16_t* __restrict__ wb) {
    for (size_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += static_cast<size_t>(gridDim.x) * blockDim.x)
        wb[i] = f2bf(w[i]);
}

// y1 = y0 + denormalised output; m carried over.  With the element table
// (comp != nullptr) the mass-fraction increments are projected onto the
// element-conserving subspace: with B_ek = a_ek / W_k and weights
// D_k = max(|Y0_k|, |Y0_k + dY_k|) + 1e-12, dY <- dY - D B^T (B D B^T)^-1 B dY,
// the correction of least D^-1-weighted norm, so species near zero hardly move
// and sum_k dY_k = 0 follows from element conservation.
//
// A wavefront takes R rows, 64 / R lanes per row: the E x E Gram matrix B D B^T
// and B dY are sums over the species in the lane's registers, added over a row's
// lanes, and each lane solves its row's (symmetric positive definite) system by
// elimination (an element absent from the mechanism's species has a zero row and
// gets lambda = 0).  Rows of y0 and of the output go through LDS, so HBM sees
// whole lines; the network output is FP32, so the decode is too (sinhf), the
// increments and the projection are FP64.
//
// R = 8: 65,536 gri30 rows in 38 us (with two lanes per row 65, with a wavefront
// per row 217), of which the 90 MB of rows are 18 at a copy's rate, one row in 6
// us instead of the 19 that two lanes need for 53 species.  R = 32 where 8 lanes
// have fewer than two species each (see launch_apply).  The loads of rows,
// outputs and tables are in flight together, and sinhf is spread over the 64
// lanes whatever the number of rows.  A row's result does not depend on R: the
// species form 8 classes, k mod 8, each summed in order, and the classes are
// added pairwise, ((0 + 1) + (2 + 3)) + ((4 + 5) + (6 + 7)), by one lane or
// across lanes.
constexpr int kMaxK = 128, kMaxE = 8, kClasses = 8;
template <int EM, int R>   // EM: elements, padded with zero rows
__global__ __launch_bounds__(64) void apply_kernel(int rows, int N, int K, const double* __restrict__ y0,
                                                   const float* __restrict__ out, const double* __restrict__ norm,
                                                   int in_p, int out_p, const double* __restrict__ comp,
                                                   const double* __restrict__ rmw, int E, double* __restrict__ y1) {
    constexpr int C = kClasses * R / 64;           // classes per lane: 1 or 4
    static_assert(C == 1 || C == 4, "rows per wavefront");
    extern __shared__ __attribute__((aligned(16))) double apply_lds[];
    const int ds = (K + 1) | 1;                    // odd row stride
    double* const ly = apply_lds;                  // rows of y0
    double* const lB = ly + R * N;                 // B_ek, species-major, EM each
    double* const ld = lB + EM * K;                // increments of T and Y before the projection
    const int lane = threadIdx.x, part = lane / R;
    const int r0 = blockIdx.x * R, nr = min(R, rows - r0);
    const bool project = comp && E >= 1 && E <= kMaxE;
    // the loads of all that goes to LDS are in flight together
    constexpr int kY = 8, kB = 8;
    const double* yr = y0 + static_cast<size_t>(r0) * N;
    const int ny = nr * N, nb = project ? K * EM : 0;
    auto b_entry = [&](int i) { return i % EM < E ? comp[i / EM * E + i % EM] * rmw[i / EM] : 0.0; };
    double vy[kY], vb[kB];
#pragma unroll
    for (int b = 0; b < kY; b++) vy[b] = yr[min(lane + 64 * b, ny - 1)];
#pragma unroll
    for (int b = 0; b < kB; b++) vb[b] = nb ? b_entry(min(lane + 64 * b, nb - 1)) : 0.0;
    const float* orow = out + static_cast<size_t>(r0) * out_p;
    const double* par = norm + 2 * in_p;           // mu, sd, sc
    const int n_out = K + 1, no = nr * n_out;      // output 0 is T, 1 + k species k
    for (int i0 = lane; i0 < no; i0 += 64 * 8) {
        float v[8];
        double mu[8], sd[8], sc[8];
        int at[8];
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const int i = min(i0 + 64 * b, no - 1);
            const int r = static_cast<int>(static_cast<unsigned>(i) / static_cast<unsigned>(n_out)), c = i - r * n_out;
            v[b] = orow[r * out_p + c];
            mu[b] = par[c];
            sd[b] = par[out_p + c];
            sc[b] = par[2 * out_p + c];
            at[b] = r * ds + c;
        }
#pragma unroll
        for (int b = 0; b < 8; b++)
            if (i0 + 64 * b < no)
                ld[at[b]] = sc[b] * static_cast<double>(sinhf(static_cast<float>(v[b] * sd[b] + mu[b])));
    }
#pragma unroll
    for (int b = 0; b < kY; b++)
        if (lane + 64 * b < ny) ly[lane + 64 * b] = vy[b];
    for (int i = lane + 64 * kY; i < ny; i += 64 * kY) {
#pragma unroll
        for (int b = 0; b < kY; b++) vy[b] = yr[min(i + 64 * b, ny - 1)];
#pragma unroll
        for (int b = 0; b < kY; b++)
            if (i + 64 * b < ny) ly[i + 64 * b] = vy[b];
    }
#pragma unroll
    for (int b = 0; b < kB; b++)
        if (lane + 64 * b < nb) lB[lane + 64 * b] = vb[b];
    for (int i = lane + 64 * kB; i < nb; i += 64) lB[i] = b_entry(i);
    __syncthreads();
    const int row = min(lane % R, nr - 1);         // spare lanes repeat the last row
    double* const y = ly + row * N;
    const double* const dy = ld + row * ds;
    auto weight = [&](int k, double d) { return fmax(fabs(y[2 + k]), fabs(y[2 + k] + d)) + 1e-12; };
    double lam[EM];
#pragma unroll
    for (int a = 0; a < EM; a++) lam[a] = 0.0;
    if (project) {
        double G[EM][EM + 1], H[EM][EM + 1];
        auto each = [&](auto&& f) {
#pragma unroll
            for (int a = 0; a < EM; a++)
#pragma unroll
                for (int b = a; b <= EM; b++) f(a, b);
        };
#pragma unroll
        for (int c = 0; c < C; c++) {
            double S[EM][EM + 1];
            each([&](int a, int b) { S[a][b] = 0.0; });
            for (int k = part * C + c; k < K; k += kClasses) {
                const double dY = dy[1 + k], D = weight(k, dY);
                double B[EM];
#pragma unroll
                for (int a = 0; a < EM; a++) B[a] = lB[k * EM + a];
#pragma unroll
                for (int a = 0; a < EM; a++) {
                    const double bd = B[a] * D;
#pragma unroll
                    for (int b = a; b < EM; b++) S[a][b] += bd * B[b];
                    S[a][EM] += B[a] * dY;
                }
            }
            if (c == 0) each([&](int a, int b) { G[a][b] = S[a][b]; });
            if (c == 1) each([&](int a, int b) { G[a][b] += S[a][b]; });
            if (c == 2) each([&](int a, int b) { H[a][b] = S[a][b]; });
            if (c == 3) each([&](int a, int b) { G[a][b] += H[a][b] + S[a][b]; });
        }
#pragma unroll
        for (int d = R; d < 64; d *= 2) each([&](int a, int b) { G[a][b] += __shfl_xor(G[a][b], d); });
        each([&](int a, int b) { if (b < EM) G[b][a] = G[a][b]; });
        // elimination without pivoting (SPD); zero rows give lambda = 0
        double rp[EM];
#pragma unroll
        for (int c = 0; c < EM; c++) {
            rp[c] = G[c][c] > 1e-300 ? 1.0 / G[c][c] : 0.0;
#pragma unroll
            for (int a = c + 1; a < EM; a++) {
                const double f = G[a][c] * rp[c];
#pragma unroll
                for (int b = c; b <= EM; b++) G[a][b] -= f * G[c][b];
            }
        }
#pragma unroll
        for (int c = EM - 1; c >= 0; c--) {
            double v = G[c][EM];
#pragma unroll
            for (int b = c + 1; b < EM; b++) v -= G[c][b] * lam[b];
            lam[c] = v * rp[c];
        }
    }
    __syncthreads();   // the spare lanes have read the last row
    if (lane % R < nr) {
        if (part == 0) y[1] += dy[0];
        for (int c = 0; c < C; c++)
            for (int k = part * C + c; k < K; k += kClasses) {
                const double d = dy[1 + k];
                double s = 0.0;
                if (project)
#pragma unroll
                    for (int a = 0; a < EM; a++) s += lB[k * EM + a] * lam[a];
                y[2 + k] += d - weight(k, d) * s;
            }
    }
    __syncthreads();
    double* const yo = y1 + static_cast<size_t>(r0) * N;
    for (int i = lane; i < nr * N; i += 64) yo[i] = ly[i];
}

// 32 rows per wavefront for small mechanisms (us per prediction of h2o2, 8 / 32
// rows: 8,192 rows 26 / 27, 11,904 28 / 28, 32,768 36 / 32, 65,536 51 / 42; gri30
// and n-dodecane the same with both at 65,536)
constexpr int kApplySmallK = 16, kApplyMany = 12288;
void launch_apply(int rows, int N, int K, const double* y0, const float* out, const double* norm, int in_p, int out_p,
                  const double* comp, const double* rmw, int E, double* y1, hipStream_t st) {
    const int em = E <= 5 ? 5 : kMaxE, R = em == 5 && K <= kApplySmallK && rows > kApplyMany ? 32 : 8;
    const size_t lds = static_cast<size_t>(R * N + em * K + R * ((K + 1) | 1)) * sizeof(double);
    auto* const k = R == 32 ? &apply_kernel<5, 32> : em == 5 ? &apply_kernel<5, 8> : &apply_kernel<kMaxE, 8>;
    hipLaunchKernelGGL(k, dim3((rows + R - 1) / R), dim3(64), lds, st, rows, N, K, y0, out, norm, in_p, out_p, comp,
                       rmw, E, y1);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) throw std::runtime_error(std::string("surrogate apply: ") + hipGetErrorString(e));
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Forward-layer GEMM, C = A B^T with A (M x K) and B (N x K) both row-major,
// on the gfx950 v_mfma_f32_16x16x32_bf16 (A/B lane layout: row lane % 16,
// k = 8 (lane / 16) .. +7; D: row 4 (lane / 16) + r, column lane % 16).
// 256 threads, a 128 x BN tile per workgroup, (64 x BN/2) per wavefront; K in
// steps of 32 through LDS with 16-byte global loads and LDS accesses, the next
// step's tile loaded into registers while the current one is multiplied.
// Requires K % 32 == 0, N % BN == 0, lda, ldb % 8 == 0 and 16-byte aligned A,
// B (as every buffer here is); rows >= M read zero and are not stored.
template <int BN, int EPI>
__global__ __launch_bounds__(256) void gemm_nt_bf16(int M, int N, int K, const uint16_t* __restrict__ A, int lda,
                                                    const uint16_t* __restrict__ B, int ldb, EpiArgs e) {
    constexpr int BM = 128, BK = 32, LK = BK + 8, WN = BN / 2, TJ = WN / 16, QB = BN / 64;
    __shared__ __attribute__((aligned(16))) uint16_t As[BM * LK];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[BN * LK];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;
    const int wm = (w >> 1) * 64, wn = (w & 1) * WN;
    f32x4 acc[4][TJ];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // chunk c = t + 256 q of a tile: row c / 4, k offset 8 (c % 4)
    const int kc = (t & 3) * 8, r0 = t >> 2, r1 = (t + 256) >> 2;
    const bool a0ok = m0 + r0 < M, a1ok = m0 + r1 < M;
    const uint16_t* pa0 = A + static_cast<size_t>(a0ok ? m0 + r0 : 0) * lda + kc;
    const uint16_t* pa1 = A + static_cast<size_t>(a1ok ? m0 + r1 : 0) * lda + kc;
    const uint16_t* pb0 = B + static_cast<size_t>(n0 + r0) * ldb + kc;
    const uint16_t* pb1 = B + static_cast<size_t>(n0 + (QB == 2 ? r1 : r0)) * ldb + kc;
    const uint4 zero{0u, 0u, 0u, 0u};
    uint4 ra0 = a0ok ? *reinterpret_cast<const uint4*>(pa0) : zero;
    uint4 ra1 = a1ok ? *reinterpret_cast<const uint4*>(pa1) : zero;
    uint4 rb0 = *reinterpret_cast<const uint4*>(pb0);
    uint4 rb1 = (QB == 2) ? *reinterpret_cast<const uint4*>(pb1) : zero;
    for (int k0 = 0; k0 < K; k0 += BK) {
        *reinterpret_cast<uint4*>(&As[r0 * LK + kc]) = ra0;
        *reinterpret_cast<uint4*>(&As[r1 * LK + kc]) = ra1;
        *reinterpret_cast<uint4*>(&Bs[r0 * LK + kc]) = rb0;
        if (QB == 2) *reinterpret_cast<uint4*>(&Bs[r1 * LK + kc]) = rb1;
        __syncthreads();
        if (k0 + BK < K) {
            const int k1 = k0 + BK;
            ra0 = a0ok ? *reinterpret_cast<const uint4*>(pa0 + k1) : zero;
            ra1 = a1ok ? *reinterpret_cast<const uint4*>(pa1 + k1) : zero;
            rb0 = *reinterpret_cast<const uint4*>(pb0 + k1);
            if (QB == 2) rb1 = *reinterpret_cast<const uint4*>(pb1 + k1);
        }
        bf16x8 a[4], b[TJ];
        const int ko = 8 * (lane >> 4);
#pragma unroll
        for (int i = 0; i < 4; i++) a[i] = *reinterpret_cast<const bf16x8*>(&As[(wm + 16 * i + (lane & 15)) * LK + ko]);
#pragma unroll
        for (int j = 0; j < TJ; j++) b[j] = *reinterpret_cast<const bf16x8*>(&Bs[(wn + 16 * j + (lane & 15)) * LK + ko]);
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + wm + 16 * i + 4 * (lane >> 4) + r;
                const int n = n0 + wn + 16 * j + (lane & 15);
                if (m >= M) continue;
                const float v = acc[i][j][r];
                const size_t o = static_cast<size_t>(m) * e.ldc + n;
                if (EPI == kFwdGelu) {
                    const float z = v + e.bias[n];
                    if (e.zf) e.zf[o] = z;      // pre-activation kept for training only
                    e.hb[o] = f2bf(gelu(z));
                } else {
                    e.zf[o] = v + e.bias[n];
                }
            }
}

// Four neighbouring columns of 8 rows of a row-major BF16 matrix as B operands
// (or A operands of a transposed product): each lane loads its own 8 rows
// (8 (lane / 16) ..) and columns (4 (lane % 16) ..), 8 bytes a row, and
// transposes the 8 x 4 block in registers with 16 byte permutes, so no LDS is
// needed.  Operand j then holds the columns 4 (lane % 16) + j of the tile.
struct Rows8 { uint2 r[8]; };
__device__ __forceinline__ bf16x8 column(const Rows8& v, int j) {
    union { uint32_t u[4]; bf16x8 b; } o;
    const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
#pragma unroll
    for (int q = 0; q < 4; q++)
        o.u[q] = j < 2 ? __builtin_amdgcn_perm(v.r[2 * q + 1].x, v.r[2 * q].x, sel)
                       : __builtin_amdgcn_perm(v.r[2 * q + 1].y, v.r[2 * q].y, sel);
    return o.b;
}

// Training's products over one batch, C = A B^T (kBwdGelu: A B): a 64 x 64 tile
// per workgroup, 16 rows x 64 columns per wavefront, operands straight from
// global memory into the MFMA lanes (layouts as above; column 4 (lane % 16) + j
// in operand j, so that results are stored 4 columns at a time).  A 4,096-row
// batch is 64 tiles of 128 x 128 for 256 CUs and only 8 k-steps long: one
// memory latency per k-step (20 us per layer) against one per KC k-steps here,
// all loads of the next KC in flight under the products of these (9 us forward
// and 7 us backward, where a tile's k-major operand was read 2 bytes at a time).
// Requires K % (32 KC) == 0, N % 16 == 0.
template <int KC, int EPI>
__global__ __launch_bounds__(256) void gemm_direct(int M, int N, int K, const uint16_t* __restrict__ A,
                                                   const uint16_t* __restrict__ B, EpiArgs e) {
    constexpr bool kTB = EPI == kBwdGelu;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, lr = lane & 15, lq = lane >> 4;
    const int m0 = blockIdx.x * 64 + 16 * w, n = blockIdx.y * 64 + 4 * lr;
    if (m0 >= M) return;
    const bool nok = n < N;
    const int nc = nok ? n : 0;
    const uint16_t* pa = A + static_cast<size_t>(min(m0 + lr, M - 1)) * K + 8 * lq;
    const uint16_t* pb = kTB ? B + static_cast<size_t>(8 * lq) * N + nc : B + static_cast<size_t>(nc) * K + 8 * lq;
    union Bk { Rows8 t; bf16x8 d[4]; };
    auto load = [&](int k0, bf16x8 (&a)[KC], Bk (&b)[KC]) {
#pragma unroll
        for (int c = 0; c < KC; c++) {
            const int k = k0 + 32 * c;
            a[c] = *reinterpret_cast<const bf16x8*>(pa + k);
            if constexpr (kTB) {
#pragma unroll
                for (int i = 0; i < 8; i++) b[c].t.r[i] = *reinterpret_cast<const uint2*>(pb + static_cast<size_t>(k + i) * N);
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) b[c].d[j] = *reinterpret_cast<const bf16x8*>(pb + static_cast<size_t>(j) * K + k);
            }
        }
    };
    bf16x8 a[KC];
    Bk b[KC];
    load(0, a, b);
    float4 z[4];   // kBwdGelu: pre-activations; otherwise the bias
#pragma unroll
    for (int r = 0; r < 4; r++)
        if constexpr (kTB)
            z[r] = *reinterpret_cast<const float4*>(e.zin + static_cast<size_t>(min(m0 + 4 * lq + r, M - 1)) * N + nc);
        else
            z[r] = *reinterpret_cast<const float4*>(e.bias + nc);
    f32x4 acc[4] = {};
    for (int k0 = 0; k0 < K; k0 += 32 * KC) {
        bf16x8 an[KC];
        Bk bn[KC];
        load(min(k0 + 32 * KC, K - 32 * KC), an, bn);
#pragma unroll
        for (int c = 0; c < KC; c++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                bf16x8 bj;
                if constexpr (kTB) bj = column(b[c].t, j);
                else bj = b[c].d[j];
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[c], bj, acc[j], 0, 0, 0);
            }
#pragma unroll
        for (int c = 0; c < KC; c++) { a[c] = an[c]; b[c] = bn[c]; }
    }
    if (!nok) return;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int m = m0 + 4 * lq + r;
        if (m >= M) continue;
        const size_t o = static_cast<size_t>(m) * N + n;
        float v[4] = {acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
        const float zz[4] = {z[r].x, z[r].y, z[r].z, z[r].w};
        union { uint16_t h[4]; uint2 u; } h;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (kTB) v[j] *= gelu_grad(zz[j]);
            else v[j] += zz[j];
            h.h[j] = f2bf(EPI == kFwdGelu ? gelu(v[j]) : v[j]);
        }
        if (!kTB && e.zf) *reinterpret_cast<float4*>(e.zf + o) = make_float4(v[0], v[1], v[2], v[3]);
        if (EPI != kFwdLinear) *reinterpret_cast<uint2*>(e.hb + o) = h.u;
    }
}

// Weight and bias gradients of every layer in one launch: dW = G^T H (fo x fi)
// and the column sums of G, over the rows [chunk z, chunk (z + 1)) of the batch,
// into split z's own copy of the parameters (grad_sum_kernel adds the copies).
// A 64 x 64 tile of one layer per workgroup; its wavefronts take every fourth
// 32 rows and are added through LDS.  Both operands are transposed in registers
// (Rows8), the next 32 rows loaded while these are multiplied.  Bias: the
// product with a column of ones, by the tiles of the first columns.
// (Layer by layer with atomics onto cleared gradients this was 20 launches and
// 160 us for 4,096 rows of 55 -> 4 x 256 -> 54, more than half of it 2-byte
// loads, the rest clears and column sums; now 16 us and 6 for the sum.)
constexpr int kGradTiles = 512;   // workgroups aimed at
struct GradArgs {
    int rows, chunk;
    int layer0;                        // the first layer of this launch
    size_t n_par;
    float* part;
    int first[18];                     // first tile of each layer, and their number
    int fo[17], fi[17];
    size_t oW[17], oB[17];
    const uint16_t* G[17];
    const uint16_t* H[17];
};
__global__ __launch_bounds__(256) void wgrad_kernel(GradArgs g) {
    __shared__ float sum[4][16][64];   // one row of tiles of each wavefront
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, lr = lane & 15, lq = lane >> 4;
    int l = g.layer0;
    while (static_cast<int>(blockIdx.x) >= g.first[l + 1]) l++;
    const int fo = g.fo[l], fi = g.fi[l], tile = blockIdx.x - g.first[l], tn = (fi + 63) / 64;
    const int m0 = tile / tn * 64, n0 = tile % tn * 64, m = m0 + 4 * lr, n = n0 + 4 * lr;
    const uint16_t* pg = g.G[l] + (m < fo ? m : 0);
    const uint16_t* ph = g.H[l] + (n < fi ? n : 0);
    const int r0 = blockIdx.y * g.chunk, r1 = min(g.rows, r0 + g.chunk);
    auto load = [&](int r, Rows8& a, Rows8& b) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int row = r + 8 * lq + i;
            const size_t q = min(row, g.rows - 1);
            a.r[i] = *reinterpret_cast<const uint2*>(pg + q * fo);
            b.r[i] = *reinterpret_cast<const uint2*>(ph + q * fi);
            if (row >= r1) a.r[i] = b.r[i] = make_uint2(0u, 0u);
        }
    };
    f32x4 acc[4][4] = {}, bias[4] = {};
    bf16x8 ones;
#pragma unroll
    for (int i = 0; i < 8; i++) ones[i] = static_cast<__bf16>(1.0f);
    Rows8 a, b;
    load(r0 + 32 * w, a, b);
    for (int r = r0 + 32 * w; r < r1; r += 128) {
        Rows8 an, bn;
        load(r + 128, an, bn);
        bf16x8 bj[4];
#pragma unroll
        for (int j = 0; j < 4; j++) bj[j] = column(b, j);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const bf16x8 ai = column(a, i);
#pragma unroll
            for (int j = 0; j < 4; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ai, bj[j], acc[i][j], 0, 0, 0);
            if (n0 == 0) bias[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ai, ones, bias[i], 0, 0, 0);
        }
        a = an;
        b = bn;
    }
    float* const part = g.part + static_cast<size_t>(blockIdx.y) * g.n_par;
    auto reduce = [&](const f32x4 (&v)[4], float (&o)[4]) {   // wavefront w: o[j] of register w
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) sum[w][4 * r + j][lane] = v[j][r];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 4; j++)
            o[j] = (sum[0][4 * w + j][lane] + sum[1][4 * w + j][lane]) + (sum[2][4 * w + j][lane] + sum[3][4 * w + j][lane]);
    };
    // operand i, register r of row group lq is row 4 (4 lq + r) + i of the tile
    const int mr = m0 + 4 * (4 * lq + w);
    float o[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        reduce(acc[i], o);
        if (mr < fo && n < fi)
            *reinterpret_cast<float4*>(part + g.oW[l] + static_cast<size_t>(mr + i) * fi + n) =
                make_float4(o[0], o[1], o[2], o[3]);
    }
    if (n0 == 0) {
        reduce(bias, o);
        if (mr < fo && lr == 0)
            *reinterpret_cast<float4*>(part + g.oB[l] + mr) = make_float4(o[0], o[1], o[2], o[3]);
    }
}

// grad = sum of the splits' copies in order, loss[0] = sum of the blocks' parts
__global__ __launch_bounds__(256) void grad_sum_kernel(size_t n, int splits, const float* __restrict__ part,
                                                       float* __restrict__ grad, double* __restrict__ loss) {
    const size_t i = 4 * (blockIdx.x * static_cast<size_t>(256) + threadIdx.x);
    if (i < n) {   // n is a multiple of 4
        float4 s = *reinterpret_cast<const float4*>(part + i);
#pragma unroll 8
        for (int z = 1; z < splits; z++) {
            const float4 v = *reinterpret_cast<const float4*>(part + z * n + i);
            s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
        }
        *reinterpret_cast<float4*>(grad + i) = s;
    }
    if (blockIdx.x) return;
    __shared__ double p[kLossBlocks];
    p[threadIdx.x] = loss[1 + threadIdx.x];
    __syncthreads();
    for (int h = kLossBlocks / 2; h > 0; h >>= 1) {
        if (static_cast<int>(threadIdx.x) < h) p[threadIdx.x] += p[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) loss[0] = p[0];
}

// Inference in one kernel: features, hidden layers and output layer for 64 rows
// per workgroup, with the activations (BF16) in LDS from layer to layer.
//
// Layer by layer through HBM, a 65,536 x 256 layer moved 100 MB for 8.6 GFLOP
// (50 us with its epilogue).  Here HBM sees the states once and the FP32
// outputs; the weights (450 KB for 55 -> 4 x 256 -> 54) are read by every
// workgroup through L2, each element by one wavefront only, straight into the
// B operand's lanes (16 bytes per lane and 16 x 32 tile), four k-steps ahead.
// Wavefront w computes columns 16 HT w .. of all rows: 4 x HT tiles of
// v_mfma_f32_16x16x32_bf16 (layouts as gemm_nt_bf16).  A layer's results stay
// in the accumulators until every wavefront has read its input, then replace it.
// hidden = 64 HT <= 256: 128 rows would need 128 accumulator registers and
// spill.  65,536 rows of the net above: 109 us against 255 us layer by layer
// (30 GFLOP: 26 us at a large product's rate); what is left over that is GELU,
// the FP64 logarithms of the features and the waits between layers.
struct MlpArgs {
    int rows, N, K, in_p, out_p, depth;
    const double* y;
    const double* P;
    const double* norm;
    const uint16_t* W;     // BF16 weights
    const float* par;      // FP32 parameters (biases)
    float* out;            // rows x out_p
    int oW[17], oB[17];
};

constexpr int kMlpRows = 64;

// KC k-steps of weights at a time, the next KC loaded while these are multiplied
template <int NT, int KC>
__device__ __forceinline__ void mlp_steps(const uint16_t* __restrict__ act, int ls, const uint16_t* __restrict__ W,
                                          int fi, int n0, f32x4 (&acc)[kMlpRows / 16][NT]) {
    const int lane = threadIdx.x & 63, lr = lane & 15, ko = 8 * (lane >> 4);
    const uint16_t* w = W + static_cast<size_t>(n0 + lr) * fi + ko;
    bf16x8 b[KC][NT];
#pragma unroll
    for (int c = 0; c < KC; c++)
#pragma unroll
        for (int j = 0; j < NT; j++) b[c][j] = *reinterpret_cast<const bf16x8*>(w + static_cast<size_t>(16 * j) * fi + 32 * c);
    for (int k0 = 0; k0 < fi; k0 += 32 * KC) {
        bf16x8 nb[KC][NT];
        const int kn = min(k0 + 32 * KC, fi - 32 * KC);
#pragma unroll
        for (int c = 0; c < KC; c++)
#pragma unroll
            for (int j = 0; j < NT; j++)
                nb[c][j] = *reinterpret_cast<const bf16x8*>(w + static_cast<size_t>(16 * j) * fi + kn + 32 * c);
#pragma unroll
        for (int c = 0; c < KC; c++)
#pragma unroll
            for (int i = 0; i < kMlpRows / 16; i++) {
                const bf16x8 a = *reinterpret_cast<const bf16x8*>(act + (16 * i + lr) * ls + k0 + 32 * c + ko);
#pragma unroll
                for (int j = 0; j < NT; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[c][j], acc[i][j], 0, 0, 0);
            }
#pragma unroll
        for (int c = 0; c < KC; c++)
#pragma unroll
            for (int j = 0; j < NT; j++) b[c][j] = nb[c][j];
    }
}

template <int NT>
__device__ __forceinline__ void mlp_layer(const uint16_t* __restrict__ act, int ls, const uint16_t* __restrict__ W,
                                          int fi, int n0, f32x4 (&acc)[kMlpRows / 16][NT]) {
#pragma unroll
    for (int i = 0; i < kMlpRows / 16; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (fi % 128 == 0) mlp_steps<NT, 4>(act, ls, W, fi, n0, acc);
    else mlp_steps<NT, 2>(act, ls, W, fi, n0, acc);   // a multiple of 64
}

template <int HT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void mlp_kernel(MlpArgs g) {
    extern __shared__ __attribute__((aligned(16))) double apply_lds[];
    uint16_t* const act = reinterpret_cast<uint16_t*>(apply_lds);
    constexpr int H = 64 * HT;
    const int ls = max(H, g.in_p) + 8;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, lr = lane & 15, lq = lane >> 4;
    const int r0 = blockIdx.x * kMlpRows;
    // features (see features_kernel): column c of a state gives feature 0 (T,
    // c = 1), 1 (ln P, in the place of the mass) or c.  Rows past the end keep
    // what LDS holds: a row of the operand reaches only its own row of the
    // result, and theirs are not stored (the features of 64 rows for a single row
    // of n-dodecane took 10 us)
    const int nr = min(kMlpRows, g.rows - r0), total = nr * g.N;
    for (int e0 = t; e0 < total; e0 += 4 * 256) {
        double x[4];
        int row[4], col[4];
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const int e = min(e0 + 256 * b, total - 1);
            row[b] = e / g.N;
            const int c = e - row[b] * g.N;
            col[b] = c < 2 ? 1 - c : c;
            const size_t s = static_cast<size_t>(r0 + row[b]);
            x[b] = c == 0 ? g.P[s] : g.y[s * g.N + c];
        }
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const double lx = log(col[b] == 1 ? x[b] : fmax(x[b], 1e-30));
            const double f = col[b] == 0 ? x[b] : lx;
            const double z = (f - g.norm[col[b]]) / g.norm[g.in_p + col[b]];
            act[row[b] * ls + col[b]] = f2bf(static_cast<float>(fmin(fmax(z, -8.0), 8.0)));
        }
    }
    for (int i = t; i < nr * (g.in_p - g.N); i += 256) {
        const int r = i / (g.in_p - g.N), c = i - r * (g.in_p - g.N);
        act[r * ls + g.N + c] = 0;
    }
    __syncthreads();
    for (int l = 0; l < g.depth; l++) {
        f32x4 acc[kMlpRows / 16][HT];
        const int n0 = 16 * HT * w;
        mlp_layer<HT>(act, ls, g.W + g.oW[l], l == 0 ? g.in_p : H, n0, acc);
        const float* bias = g.par + g.oB[l] + n0;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < HT; j++) {
            const float bj = bias[16 * j + lr];
#pragma unroll
            for (int i = 0; i < kMlpRows / 16; i++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    act[(16 * i + 4 * lq + r) * ls + n0 + 16 * j + lr] = f2bf(gelu(acc[i][j][r] + bj));
        }
        __syncthreads();
    }
    for (int c = 0; c < g.out_p; c += 64) {   // output layer, 16 columns per wavefront
        f32x4 acc[kMlpRows / 16][1];
        const int n0 = c + 16 * w;
        mlp_layer<1>(act, ls, g.W + g.oW[g.depth], H, n0, acc);
        const float bj = g.par[g.oB[g.depth] + n0 + lr];
#pragma unroll
        for (int i = 0; i < kMlpRows / 16; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = r0 + 16 * i + 4 * lq + r;
                if (row < g.rows) g.out[static_cast<size_t>(row) * g.out_p + n0 + lr] = acc[i][0][r] + bj;
            }
    }
}

void check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

// C = A B^T (kBwdGelu: A B) with A (M x K), every matrix contiguous.  Forward
// layers go to gemm_nt_bf16 once its larger tiles make 128 workgroups (16,384
// rows of 320: 93 us per prediction against 109 with gemm_direct; of 1,024: 175
// against 391; 1,024 rows of 1,024, 64 workgroups: 106 against 87).
template <int EPI>
void gemm(int M, int N, int K, const uint16_t* A, const uint16_t* B, const EpiArgs& e, hipStream_t s) {
    const int bn = N % 128 ? 64 : 128;
    if (K % 32) {
        hipLaunchKernelGGL((gemm_bf16<EPI>), dim3((M + kTM - 1) / kTM, (N + kTN - 1) / kTN), dim3(256), 0, s, M, N, K,
                           A, B, e);
    } else if (EPI == kBwdGelu || N % 64 || (M + 127) / 128 * (N / bn) < 128) {
        auto* const k = K % 128 == 0 ? &gemm_direct<4, EPI> : K % 64 == 0 ? &gemm_direct<2, EPI> : &gemm_direct<1, EPI>;
        hipLaunchKernelGGL(k, dim3((M + 63) / 64, (N + 63) / 64), dim3(256), 0, s, M, N, K, A, B, e);
    } else if constexpr (EPI != kBwdGelu) {
        auto* const k = bn == 128 ? &gemm_nt_bf16<128, EPI> : &gemm_nt_bf16<64, EPI>;
        hipLaunchKernelGGL(k, dim3((M + 127) / 128, N / bn), dim3(256), 0, s, M, N, K, A, K, B, K, e);
    }
    check(hipGetLastError(), "surrogate GEMM launch");
}

int pad64(int x) { return (x + 63) / 64 * 64; }

}  // namespace

SurrogateNet::SurrogateNet(int K, double dt, int hidden, int depth, uint64_t seed) {
    if (K < 1 || hidden < 16 || hidden % 16 || depth < 1 || depth > 16 || !(dt > 0))
        throw std::runtime_error("surrogate: bad shape (hidden must be a positive multiple of 16, 1 <= depth <= 16)");
    if (K > kMaxK) throw std::runtime_error("surrogate: at most 128 species");
    s_.K = K;
    s_.n_in = 2 + K;
    s_.n_out = 1 + K;
    s_.in_p = pad64(s_.n_in);
    s_.out_p = pad64(s_.n_out);
    s_.hidden = hidden;
    s_.depth = depth;
    dt_ = dt;
    rng_ = seed;
    size_t off = 0;
    for (int l = 0; l < s_.layers(); l++) {
        oW_.push_back(off);
        off += static_cast<size_t>(s_.fan_out(l)) * s_.fan_in(l);
        oB_.push_back(off);
        off += s_.fan_out(l);
    }
    n_par_ = off;
    // uniform(-1/sqrt(fan_in), 1/sqrt(fan_in)) weights, zero biases; padded
    // rows of the last layer zero (their gradients are zero, so they stay zero)
    std::vector<float> h(n_par_, 0.f);
    std::mt19937_64 g(seed);
    for (int l = 0; l < s_.layers(); l++) {
        const int fi = s_.fan_in(l), fo = s_.fan_out(l);
        const int real_in = (l == 0) ? s_.n_in : fi;
        const int real_out = (l == s_.depth) ? s_.n_out : fo;
        std::uniform_real_distribution<float> u(-1.f / std::sqrt(static_cast<float>(real_in)),
                                                1.f / std::sqrt(static_cast<float>(real_in)));
        for (int o = 0; o < real_out; o++)
            for (int i = 0; i < real_in; i++) h[oW_[l] + static_cast<size_t>(o) * fi + i] = u(g);
    }
    check(hipMalloc(&par_, n_par_ * 4), "hipMalloc(surrogate)");
    check(hipMalloc(&grad_, n_par_ * 4), "hipMalloc(surrogate)");
    check(hipMalloc(&m1_, n_par_ * 4), "hipMalloc(surrogate)");
    check(hipMalloc(&m2_, n_par_ * 4), "hipMalloc(surrogate)");
    check(hipMalloc(&wb_, n_par_ * 2), "hipMalloc(surrogate)");
    check(hipMalloc(&norm_, norm_len() * sizeof(double)), "hipMalloc(surrogate)");
    check(hipMalloc(&loss_, (1 + kLossBlocks) * sizeof(double)), "hipMalloc(surrogate)");
    check(hipMemcpy(par_, h.data(), n_par_ * 4, hipMemcpyHostToDevice), "hipMemcpy");
    check(hipMemset(m1_, 0, n_par_ * 4), "hipMemset");
    check(hipMemset(m2_, 0, n_par_ * 4), "hipMemset");
    std::vector<double> nm(norm_len(), 0.0);
    for (int j = 0; j < s_.in_p; j++) nm[s_.in_p + j] = 1.0;
    for (int j = 0; j < s_.out_p; j++) nm[2 * s_.in_p + s_.out_p + j] = 1.0;
    for (int j = 0; j < s_.out_p; j++) nm[2 * s_.in_p + 2 * s_.out_p + j] = 1.0;
    set_normalization(nm.data());
    sync_bf16(nullptr);
    check(hipDeviceSynchronize(), "surrogate init");
}

SurrogateNet::~SurrogateNet() {
    for (void* p : {static_cast<void*>(par_), static_cast<void*>(grad_), static_cast<void*>(m1_),
                    static_cast<void*>(m2_), static_cast<void*>(wb_), static_cast<void*>(norm_),
                    static_cast<void*>(loss_)})
        if (p) (void)hipFree(p);
}

void SurrogateNet::sync_bf16(hipStream_t s) {
    hipLaunchKernelGGL(to_bf16_kernel, dim3(256), dim3(256), 0, s, n_par_, par_, wb_);
    check(hipGetLastError(), "surrogate bf16 copy");
}

DeviceBuffer::~DeviceBuffer() {
    if (p_) (void)hipFree(p_);
}

void DeviceBuffer::reserve(size_t bytes) {
    if (bytes <= bytes_) return;
    void* old = p_;
    p_ = nullptr;
    bytes_ = 0;
    if (old) check(hipFree(old), "hipFree(surrogate)");
    check(hipMalloc(&p_, bytes), "hipMalloc(surrogate)");
    bytes_ = bytes;
}

// Gradient operands held at a time: one launch computes the weight gradients of
// as many layers as 256 MB of operands hold (all of them up to 123,361 rows of 4 x
// 256), at least two, for a layer's operand is made from the next one's.  With
// every layer's operand held, 1,048,576 rows of 16 x 1,024 had 30 GB more to find
// than with two.
constexpr size_t kHeldBytes = size_t{256} << 20;
int SurrogateNet::held_operands(int rows) const {
    const size_t n = kHeldBytes / (static_cast<size_t>(rows) * std::max(s_.out_p, s_.hidden) * 2);
    return static_cast<int>(std::min(std::max<size_t>(n, 2), static_cast<size_t>(s_.layers())));
}

void SurrogateNet::reserve_training(int rows) {
    const size_t r = static_cast<size_t>(rows), deep = static_cast<size_t>(s_.depth) * s_.hidden;
    act_.reserve(r * (s_.in_p + deep) * 2);
    pre_.reserve(r * deep * 4);
    out_.reserve(r * s_.out_p * 4);
    g_.reserve(held_operands(rows) * r * std::max(s_.out_p, s_.hidden) * 2);
    idx_.reserve(r * 4);
}

// H_0 = features (already in act_), H_{l+1} = gelu(H_l W_l^T + b_l), out = H_depth W^T + b
void SurrogateNet::forward(int rows, hipStream_t st) {
    const size_t r = static_cast<size_t>(rows);
    uint16_t* const act = act_.as<uint16_t>();
    for (int l = 0; l <= s_.depth; l++) {
        const int fi = s_.fan_in(l), fo = s_.fan_out(l);
        const uint16_t* H = (l == 0) ? act : act + r * (s_.in_p + static_cast<size_t>(l - 1) * s_.hidden);
        EpiArgs e{};
        e.bias = par_ + oB_[l];
        e.ldc = fo;
        if (l < s_.depth) {
            e.zf = pre_.as<float>() + r * static_cast<size_t>(l) * s_.hidden;
            e.hb = act + r * (s_.in_p + static_cast<size_t>(l) * s_.hidden);
            gemm<kFwdGelu>(rows, fo, fi, H, wb_ + oW_[l], e, st);
        } else {
            e.zf = out_.as<float>();
            gemm<kFwdLinear>(rows, fo, fi, H, wb_ + oW_[l], e, st);
        }
    }
}

// Weight and bias gradients of layers l0 .. l1 into grad_ (and loss_[0]); G(l): the
// gradient operand of layer l's outputs.
template <class F>
void SurrogateNet::weight_gradients(int rows, int l0, int l1, F&& G, hipStream_t st) {
    const size_t r = static_cast<size_t>(rows);
    GradArgs g{};
    g.rows = rows;
    g.layer0 = l0;
    const size_t base = oW_[l0];
    g.n_par = (l1 == s_.depth ? n_par_ : oW_[l1 + 1]) - base;
    for (int l = l0; l <= l1; l++) {
        g.fo[l] = s_.fan_out(l);
        g.fi[l] = s_.fan_in(l);
        g.oW[l] = oW_[l] - base;
        g.oB[l] = oB_[l] - base;
        g.G[l] = G(l);
        const uint16_t* act = act_.as<uint16_t>();
        g.H[l] = (l == 0) ? act : act + r * (s_.in_p + static_cast<size_t>(l - 1) * s_.hidden);
        g.first[l + 1] = g.first[l] + (g.fo[l] + 63) / 64 * ((g.fi[l] + 63) / 64);
    }
    // at most kGradTiles workgroups of at least 256 rows each (4,096 rows of
    // 4 x 256: 131 us per gradient with 512, 139 with 1,024 or 2,048)
    const int tiles = g.first[l1 + 1];
    const int want = std::max(1, std::min(kGradTiles / tiles, (rows + 255) / 256));
    g.chunk = ((rows + want - 1) / want + 127) / 128 * 128;
    const int splits = (rows + g.chunk - 1) / g.chunk;
    if (splits > 1) part_.reserve(g.n_par * 4 * std::max(1, kGradTiles / tiles));
    g.part = splits > 1 ? part_.as<float>() : grad_ + base;
    hipLaunchKernelGGL(wgrad_kernel, dim3(tiles, splits), dim3(256), 0, st, g);
    check(hipGetLastError(), "surrogate weight gradient");
    const size_t nsum = splits > 1 ? g.n_par : 0;
    hipLaunchKernelGGL(grad_sum_kernel, dim3(static_cast<unsigned>((nsum + 1023) / 1024 + (nsum == 0))), dim3(256), 0, st,
                       nsum, splits, part_.as<float>(), grad_ + base, loss_);
    check(hipGetLastError(), "surrogate gradient sum");
}

// loss of out_ against the pairs (rows idx, or all), gradient into grad_,
// optional Adam step
double SurrogateNet::backward_and_loss(int rows, const int* idx, const double* y0, const double* y1, bool update,
                                       double lr, hipStream_t st) {
    const size_t r = static_cast<size_t>(rows);
    const int held = held_operands(rows);
    const auto G = [&](int l) {   // in turn, from G_depth to G_0
        return g_.as<uint16_t>() + static_cast<size_t>((s_.depth - l) % held) * r * std::max(s_.out_p, s_.hidden);
    };
    int top = s_.depth;           // the layers above are done
    hipLaunchKernelGGL(loss_kernel, dim3(kLossBlocks), dim3(256), 0, st, rows, idx, s_.K + 2, s_.n_out, s_.in_p,
                       s_.out_p, y0, y1, norm_, out_.as<float>(), G(s_.depth), loss_);
    check(hipGetLastError(), "surrogate loss");
    for (int l = s_.depth; l > 0; l--) {
        // G_{l-1} = (G_l W_l) * gelu'(Z_{l-1})  (rows x fan_in)
        EpiArgs e{};
        e.hb = G(l - 1);
        e.zin = pre_.as<float>() + r * static_cast<size_t>(l - 1) * s_.hidden;
        e.ldc = s_.fan_in(l);
        gemm<kBwdGelu>(rows, s_.fan_in(l), s_.fan_out(l), G(l), wb_ + oW_[l], e, st);
        // the operand of layer `top` makes place for that of l - 2
        if (top - (l - 1) + 1 == held && l > 1) {
            weight_gradients(rows, l - 1, top, G, st);
            top = l - 2;
        }
    }
    if (top >= 0) weight_gradients(rows, 0, top, G, st);
    if (update) {
        adam_t_ += 1;
        const float c1 = 1.f - std::pow(0.9f, static_cast<float>(adam_t_));
        const float c2 = 1.f - std::pow(0.999f, static_cast<float>(adam_t_));
        hipLaunchKernelGGL(adam_kernel, dim3(512), dim3(256), 0, st, n_par_, par_, grad_, m1_, m2_, wb_,
                           static_cast<float>(lr), c1, c2);
        check(hipGetLastError(), "surrogate Adam");
    }
    double loss = 0.0;
    check(hipMemcpyAsync(&loss, loss_, sizeof(double), hipMemcpyDeviceToHost, st), "hipMemcpyAsync(loss)");
    check(hipStreamSynchronize(st), "hipStreamSynchronize");
    return loss;
}

void SurrogateNet::fit_normalization(long n, const double* y0, const double* P, const double* y1, long sample) {
    const long S = std::min(n, sample);
    const int N = s_.K + 2;
    std::vector<double> a(static_cast<size_t>(S) * N), b(static_cast<size_t>(S) * N), p(S);
    check(hipMemcpy(a.data(), y0, a.size() * 8, hipMemcpyDeviceToHost), "hipMemcpy");
    check(hipMemcpy(b.data(), y1, b.size() * 8, hipMemcpyDeviceToHost), "hipMemcpy");
    check(hipMemcpy(p.data(), P, p.size() * 8, hipMemcpyDeviceToHost), "hipMemcpy");
    const int ip = s_.in_p, op = s_.out_p;
    std::vector<double> nm(norm_len(), 0.0), s1(ip, 0.0), s2(ip, 0.0), t1(op, 0.0), t2(op, 0.0), sq(op, 0.0);
    // scale of each increment: 1e-3 of its RMS over the sample
    for (long r = 0; r < S; r++)
        for (int j = 0; j < s_.n_out; j++) {
            const double d = b[static_cast<size_t>(r) * N + 1 + j] - a[static_cast<size_t>(r) * N + 1 + j];
            sq[j] += d * d;
        }
    std::vector<double> sc(op, 1.0);
    for (int j = 0; j < s_.n_out; j++) sc[j] = std::max(1e-3 * std::sqrt(sq[j] / S), 1e-300);
    for (long r = 0; r < S; r++) {
        const double* y = &a[static_cast<size_t>(r) * N];
        const double* z = &b[static_cast<size_t>(r) * N];
        for (int j = 0; j < s_.n_in; j++) {
            const double f = (j == 0) ? y[1] : (j == 1) ? std::log(p[r]) : std::log(std::max(y[j], 1e-30));
            s1[j] += f;
            s2[j] += f * f;
        }
        for (int j = 0; j < s_.n_out; j++) {
            const double d = std::asinh((z[1 + j] - y[1 + j]) / sc[j]);
            t1[j] += d;
            t2[j] += d * d;
        }
    }
    for (int j = 0; j < ip; j++) {
        const double mu = s1[j] / S, var = s2[j] / S - mu * mu;
        nm[j] = (j < s_.n_in) ? mu : 0.0;
        nm[ip + j] = (j < s_.n_in && var > 1e-24) ? std::sqrt(var) : 1.0;
    }
    for (int j = 0; j < op; j++) {
        const double mu = t1[j] / S, var = t2[j] / S - mu * mu;
        nm[2 * ip + j] = (j < s_.n_out) ? mu : 0.0;
        nm[2 * ip + op + j] = (j < s_.n_out && var > 1e-24) ? std::sqrt(var) : 1.0;
        nm[2 * ip + 2 * op + j] = sc[j];
    }
    set_normalization(nm.data());
}

double SurrogateNet::train_epoch(long n, const double* y0, const double* P, const double* y1, int batch, double lr,
                                 hipStream_t st) {
    if (batch < 1) throw std::runtime_error("surrogate: batch must be positive");
    reserve_training(batch);
    std::vector<int> perm(n);
    for (long i = 0; i < n; i++) perm[i] = static_cast<int>(i);
    std::mt19937_64 g(rng_++);
    std::shuffle(perm.begin(), perm.end(), g);
    const int N = s_.K + 2;
    double total = 0.0;
    long nb = 0;
    for (long b0 = 0; b0 < n; b0 += batch) {
        const int rows = static_cast<int>(std::min<long>(batch, n - b0));
        check(hipMemcpyAsync(idx_.as<int>(), perm.data() + b0, rows * 4, hipMemcpyHostToDevice, st), "hipMemcpyAsync(idx)");
        hipLaunchKernelGGL(features_kernel, dim3(rows), dim3(64), 0, st, rows, idx_.as<int>(), N, s_.K, y0, P,
                           norm_, s_.in_p, act_.as<uint16_t>());
        check(hipGetLastError(), "surrogate features");
        forward(rows, st);
        total += backward_and_loss(rows, idx_.as<int>(), y0, y1, true, lr, st);
        nb++;
    }
    return nb ? total / nb : 0.0;
}

double SurrogateNet::loss_grad(long n, const double* y0, const double* P, const double* y1, float* grad_host,
                               hipStream_t st) {
    const int rows = static_cast<int>(n);
    reserve_training(rows);
    const int N = s_.K + 2;
    hipLaunchKernelGGL(features_kernel, dim3(rows), dim3(64), 0, st, rows, nullptr, N, s_.K, y0, P, norm_, s_.in_p,
                       act_.as<uint16_t>());
    check(hipGetLastError(), "surrogate features");
    forward(rows, st);
    const double loss = backward_and_loss(rows, nullptr, y0, y1, false, 0.0, st);
    if (grad_host) check(hipMemcpy(grad_host, grad_, n_par_ * 4, hipMemcpyDeviceToHost), "hipMemcpy(grad)");
    return loss;
}

// The fused kernel takes hidden widths of 64, 128, 192 and 256 (weights are
// 16-byte aligned: every width and offset is a multiple of 8 elements).
bool SurrogateNet::fused_shape() const { return s_.hidden % 64 == 0 && s_.hidden <= 256; }

void SurrogateNet::infer_fused(int rows, const double* y0, const double* P, float* out, hipStream_t st) const {
    MlpArgs g{};
    g.rows = rows; g.N = s_.K + 2; g.K = s_.K; g.in_p = s_.in_p; g.out_p = s_.out_p; g.depth = s_.depth;
    g.y = y0; g.P = P; g.norm = norm_; g.W = wb_; g.par = par_; g.out = out;
    for (int l = 0; l <= s_.depth; l++) {
        g.oW[l] = static_cast<int>(oW_[l]);
        g.oB[l] = static_cast<int>(oB_[l]);
    }
    const size_t lds = static_cast<size_t>(kMlpRows) * (std::max(s_.hidden, s_.in_p) + 8) * 2;
    const void* kp = nullptr;
    switch (s_.hidden / 64) {
        case 1: kp = reinterpret_cast<const void*>(&mlp_kernel<1>); break;
        case 2: kp = reinterpret_cast<const void*>(&mlp_kernel<2>); break;
        case 3: kp = reinterpret_cast<const void*>(&mlp_kernel<3>); break;
        default: kp = reinterpret_cast<const void*>(&mlp_kernel<4>);
    }
    void* args[] = {&g};
    check(hipLaunchKernel(kp, dim3((rows + kMlpRows - 1) / kMlpRows), dim3(256), args, lds, st), "surrogate MLP launch");
}

// Workspace of a row: the FP32 output (out_p) and, layer by layer, features (in_p
// BF16) and two hidden activations (BF16, ping-pong).
size_t SurrogateNet::infer_row_bytes() const {
    return static_cast<size_t>(s_.out_p) * 4 +
           (fused_shape() ? 0 : static_cast<size_t>(s_.in_p) * 2 + 4 * static_cast<size_t>(s_.hidden));
}

// y1 of `rows` rows through a workspace for `capacity` of them (every array of it
// starts at a multiple of 16 bytes: widths are multiples of 16).
void SurrogateNet::infer(int rows, const double* y0, const double* P, double* y1, unsigned char* workspace,
                         int capacity, hipStream_t st) const {
    const int N = s_.K + 2;
    const size_t r = static_cast<size_t>(capacity);
    float* const out = reinterpret_cast<float*>(workspace);
    if (fused_shape()) {
        infer_fused(rows, y0, P, out, st);
    } else {
        uint16_t* const feat = reinterpret_cast<uint16_t*>(out + r * s_.out_p);
        uint16_t* const ha = feat + r * s_.in_p;
        uint16_t* const hb = ha + r * s_.hidden;
        hipLaunchKernelGGL(features_kernel, dim3(rows), dim3(64), 0, st, rows, nullptr, N, s_.K, y0, P, norm_, s_.in_p,
                           feat);
        check(hipGetLastError(), "surrogate features");
        const uint16_t* H = feat;
        uint16_t* next = ha;
        for (int l = 0; l <= s_.depth; l++) {
            const int fi = s_.fan_in(l), fo = s_.fan_out(l);
            EpiArgs e{};
            e.bias = par_ + oB_[l];
            e.ldc = fo;
            if (l < s_.depth) {
                e.hb = next;
                gemm<kFwdGelu>(rows, fo, fi, H, wb_ + oW_[l], e, st);
                H = next;
                next = (next == ha) ? hb : ha;
            } else {
                e.zf = out;
                gemm<kFwdLinear>(rows, fo, fi, H, wb_ + oW_[l], e, st);
            }
        }
    }
    launch_apply(rows, N, s_.K, y0, out, norm_, s_.in_p, s_.out_p, comp_, rmw_, E_, y1, st);
}

void SurrogateNet::predict(long n, const double* y0, const double* P, double* y1, hipStream_t st) {
    const int N = s_.K + 2;
    const long chunk = 65536;
    const int cap = static_cast<int>(std::min(chunk, n));
    ws_.reserve(cap * infer_row_bytes());
    for (long c0 = 0; c0 < n; c0 += chunk)
        infer(static_cast<int>(std::min(chunk, n - c0)), y0 + c0 * N, P + c0, y1 + c0 * N, ws_.as<unsigned char>(), cap,
              st);
}

// ---- inference without allocation ------------------------------------------
//
// Workspace of predict_noalloc: one array per device, part of the code object,
// held until the process ends.  Its address on the current device comes from
// hipGetSymbolAddress (the array's name is only a host-side stand-in), once
// per device, and is kept per device.
constexpr size_t kNoAllocBytes = size_t{16} << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

void* scratch_on_current_device() {
    int dev = -1;
    check(hipGetDevice(&dev), "hipGetDevice");
    if (dev < 0 || dev >= kMaxDevices) throw std::runtime_error("surrogate: device index out of range");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        check(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
        if (!p) throw std::runtime_error("surrogate: no address for the inference workspace");
        g_scratch_ptr[dev] = p;
    }
    return g_scratch_ptr[dev];
}
}  // namespace

size_t SurrogateNet::noalloc_workspace_bytes() { return kNoAllocBytes; }

// Rows per pass through the workspace: features (in_p BF16), two hidden
// activations (BF16, ping-pong), the FP32 output (out_p); a multiple of 128
// (the GEMM row tile), so every buffer starts 256-byte aligned.
int SurrogateNet::noalloc_rows() const {
    const size_t per_row = static_cast<size_t>(s_.in_p) * 2 + 4 * static_cast<size_t>(s_.hidden) +
                           static_cast<size_t>(s_.out_p) * 4;
    const size_t rows = kNoAllocBytes / per_row / 128 * 128;
    return static_cast<int>(std::min<size_t>(rows, 1 << 20));
}

void SurrogateNet::predict_noalloc(long n, const double* y0, const double* P, double* y1, hipStream_t st) {
    const int R = noalloc_rows();
    if (R < 128)
        throw std::runtime_error("surrogate: network too wide for the 16 MiB inference workspace (fewer than 128 rows)");
    unsigned char* base = static_cast<unsigned char*>(scratch_on_current_device());
    const int N = s_.K + 2;
    for (long c0 = 0; c0 < n; c0 += R)
        infer(static_cast<int>(std::min<long>(R, n - c0)), y0 + c0 * N, P + c0, y1 + c0 * N, base, R, st);
}

void SurrogateNet::set_elements(const double* comp, const double* rmw, int E) {
    if (E < 1 || E > kMaxE) throw std::runtime_error("surrogate: element projection supports 1 to 8 elements");
    comp_ = comp;
    rmw_ = rmw;
    E_ = E;
}

void SurrogateNet::get_params(float* host) const {
    check(hipMemcpy(host, par_, n_par_ * 4, hipMemcpyDeviceToHost), "hipMemcpy(params)");
}
void SurrogateNet::set_params(const float* host) {
    check(hipMemcpy(par_, host, n_par_ * 4, hipMemcpyHostToDevice), "hipMemcpy(params)");
    sync_bf16(nullptr);
    check(hipDeviceSynchronize(), "surrogate set_params");
}
void SurrogateNet::get_normalization(double* host) const {
    check(hipMemcpy(host, norm_, norm_len() * 8, hipMemcpyDeviceToHost), "hipMemcpy(norm)");
}
void SurrogateNet::set_normalization(const double* host) {
    check(hipMemcpy(norm_, host, norm_len() * 8, hipMemcpyHostToDevice), "hipMemcpy(norm)");
}

}  // namespace cg
