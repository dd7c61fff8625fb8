// hjm_calibration.hip -- batched PCA calibration of the HJM loadings from historical
// forward curves (the step upstream of the path, reference roadmap doc/TODO:16), gfx950.
//
// For each rolling window of `window` consecutive curves (51 tenors each): daily
// differences d_t = f_{t+1} - f_t, their sample covariance annualised by `obs_per_year`,
// its full eigendecomposition, and the loadings sigma_k = sqrt(lambda_k) v_k of the
// leading factors, optionally smoothed by least-squares polynomials in the tenor, and
// the loadings' HJM drift (the cumulative Simpson rule of hjm_hjm_drift).
//
// Two kernels, one wave per window in both:
//   calib_cov_kernel: covariance on the FP64 matrix cores;
//   calib_pca_kernel: Householder tridiagonalisation, all eigenvalues by bisection on Sturm
//     counts, the leading eigenvectors by inverse iteration, then signs, loadings and fits.
#include <math.h>

#include <algorithm>

#include "hjm_host.h"

using namespace hjm;
using namespace hjm_host;

namespace {

constexpr int kN = kTenors;        // 51
constexpr int kMaxFactors = 8;
constexpr int kMaxDegree = 5;

struct CalibParams {
    int64_t ncurves;
    int64_t window;       // curves per window (window - 1 differences)
    int64_t step;         // curves between window starts
    int32_t nwindows;
    int32_t nfactors;
    double obs_per_year;
    double dtau;
    int32_t degree[kMaxFactors];  // < 0: raw PCA loading
};

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef double d2_t __attribute__((ext_vector_type(2)));

// Covariance of window blockIdx.x to cov[window][51][51]: C = D^T D of the centred differences
// D, 4 days per product, tenors in 4 blocks of 16 (10 blocks of the upper triangle, then
// mirrored). Lane l holds tenor 16 b + l % 16 of day t + l / 16, which is the layout of
// either operand, so the differences come straight from the curves and nothing passes
// through LDS. The differences' mean is that of their telescoped sum. Bound by the products (10
// per 4 days, of which 4 are mostly padding: 2101 windows of 500 curves are 68 us at the
// matrix cores' FP64 rate) and the uneven share of windows per SIMD: 178 us, 263 with the
// curves loaded when they are used.
__global__ __launch_bounds__(kWave, 3) void calib_cov_kernel(const CalibParams prm, int64_t first,
                                                        const double* __restrict__ curves,
                                                        double* __restrict__ cov)
{
    constexpr int kBlocks = (kN + 15) / 16;
    const int lane = threadIdx.x, grp = lane >> 4, col = lane & 15;
    const double* base = curves + (first + blockIdx.x) * prm.step * kN;
    const int64_t nd = prm.window - 1;
    int at[kBlocks];
    bool on[kBlocks];
    double mean[kBlocks];
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) {
        on[b] = 16 * b + col < kN;
        at[b] = on[b] ? 16 * b + col : kN - 1;
        mean[b] = (base[nd * kN + at[b]] - base[at[b]]) / (double)nd;
    }
    d4_t acc[kBlocks][kBlocks];
#pragma unroll
    for (int a = 0; a < kBlocks; ++a)
#pragma unroll
        for (int b = a; b < kBlocks; ++b) acc[a][b] = d4_t{0.0, 0.0, 0.0, 0.0};
    // the curves of the next two products are loaded ahead of this one
    constexpr int kAhead = 2;
    double f0[kAhead][kBlocks], f1[kAhead][kBlocks];
    auto load = [&](int slot, int64_t t0) {
        const int64_t t = t0 + grp < nd ? t0 + grp : nd - 1;
#pragma unroll
        for (int b = 0; b < kBlocks; ++b) {
            f0[slot][b] = base[t * kN + at[b]];
            f1[slot][b] = base[(t + 1) * kN + at[b]];
        }
    };
#pragma unroll
    for (int s = 0; s < kAhead; ++s) load(s, 4 * s);
    for (int64_t t0 = 0; t0 < nd; t0 += 4 * kAhead) {
#pragma unroll
        for (int s = 0; s < kAhead; ++s) {
            double x[kBlocks];
            const bool day = t0 + 4 * s + grp < nd;
#pragma unroll
            for (int b = 0; b < kBlocks; ++b)
                x[b] = on[b] && day ? (f1[s][b] - f0[s][b]) - mean[b] : 0.0;
            load(s, t0 + 4 * (s + kAhead));
#pragma unroll
            for (int a = 0; a < kBlocks; ++a)
#pragma unroll
                for (int b = a; b < kBlocks; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[a], x[b], acc[a][b], 0, 0, 0);
        }
    }
    const double scale = prm.obs_per_year / (double)(nd - 1);
    double* C = cov + (int64_t)blockIdx.x * kN * kN;
#pragma unroll
    for (int a = 0; a < kBlocks; ++a)
#pragma unroll
        for (int b = a; b < kBlocks; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = 16 * a + 4 * r + grp, j = 16 * b + col;   // register r of the tile
                if (i < kN && j < kN) {
                    const double c = acc[a][b][r] * scale;
                    C[i * kN + j] = c;
                    if (a < b) C[j * kN + i] = c;
                }
            }
}

// Householder steps [K0, K1) on columns held as a[j] = A[lane][k + j] (j < NB; the columns move
// down one register per step, so that the pivot column is always a[0]). Step k: the reflector
// I - v v^T / h takes column k to (d_k, e_k, 0, ...); A <- A - v w^T - w v^T.
template <int NB, int K0, int K1>
__device__ __forceinline__ void householder(double (&a)[kN], int lane, double* s_v, double* s_w, d2_t* s_de,
                                            double* s_e, double* s_h, double* s_ih)
{
#pragma unroll 1
    for (int k = K0; k < K1; ++k) {
        const double x = lane > k && lane < kN ? a[0] : 0.0;
        const double sigma = wave_sum(lane > k + 1 ? x * x : 0.0);
        const double alpha = __shfl(x, k + 1);
        double e = alpha, v = 0.0, ih = 0.0;
        if (sigma > 0.0) {   // uniform
            const double mu = sqrt(alpha * alpha + sigma);
            e = alpha > 0.0 ? -mu : mu;
            v = lane == k + 1 ? alpha - e : x;
            ih = 1.0 / (mu * (mu + fabs(alpha)));
        }
        if (lane == k) {
            s_de[k][0] = a[0];
            s_e[k] = e;
            s_ih[k] = ih;
        }
        if (lane > k && lane < kN) s_h[k * (kN - 1) - k * (k - 1) / 2 + lane - k - 1] = v;
        s_v[lane] = v;
        __syncthreads();
        double p0 = 0.0, p1 = 0.0;
#pragma unroll
        for (int j = 1; j < NB; ++j) {
            if (j & 1) p0 = fma(a[j], s_v[k + j], p0);
            else p1 = fma(a[j], s_v[k + j], p1);
        }
        const double p = (p0 + p1) * ih;
        const double w = fma(-0.5 * ih * wave_sum(v * p), v, p);
        s_w[lane] = w;
        __syncthreads();
#pragma unroll
        for (int j = 1; j < NB; ++j) a[j - 1] = fma(-w, s_v[k + j], fma(-v, s_w[k + j], a[j]));
        a[NB - 1] = 0.0;
        __syncthreads();
    }
}

// Number of eigenvalues of the tridiagonal {d_j, e_{j-1}^2} below x: sign changes of the leading
// minors' recurrence (3 FP64 instructions a row), rescaled every 8 rows: the matrix's entries are
// scaled to at most 1, so d, e and x are at most 51 or so (a parallel shift's d), and 8 rows
// gain at most 2^64; e^2 has a floor of 2^-118, far below rounding, so that they lose at most
// 2^-480, and a zero minor is followed by one of the opposite sign.
__device__ __forceinline__ int sturm_count(const d2_t* s_de, double x)
{
    // an opaque offset: the entries stay in LDS rather than in 204 registers across the calls
    int at = 0;
    asm volatile("" : "+v"(at));
    s_de += at;
    auto high = [](double v) { return (uint32_t)(__builtin_bit_cast(uint64_t, v) >> 32); };
    double p = s_de[0][0] - x, q = 1.0;
    uint32_t signs = high(p) >> 31;   // the latest minor's sign bit shifted in at the bottom
    int n = (int)signs;
#pragma unroll
    for (int j = 1; j < kN; ++j) {
        const d2_t t = s_de[j];
        const double r = fma(t[0] - x, p, -(t[1] * q));
        q = p;
        p = r;
        signs = __builtin_amdgcn_alignbit(signs, high(r), 31);
        // 25 changes at a time
        if (j % 25 == 0) n += __popc((signs ^ signs >> 1) & 0x1ffffffu);
        if (j % 8 == 0 && j + 1 < kN) {
            const int ex = -__builtin_amdgcn_frexp_exp(fmax(fabs(p), fabs(q)));
            p = ldexp(p, ex);
            q = ldexp(q, ex);
        }
    }
    static_assert((kN - 1) % 25 == 0, "the sign bits are counted 25 at a time");
    return n;
}

// Least-squares polynomial of m <= 6 terms in x = tau / tau_max through y, evaluated to out
// (normal equations, Gauss-Jordan with partial pivoting; degree <= 5 keeps them well
// conditioned on [0, 1]). Every index is a constant once unrolled: the system in registers.
__device__ __forceinline__ void fit_polynomial(const double* y, int m, double* out)
{
    constexpr int M = kMaxDegree + 1;
    double G[M][M + 1] = {};
    for (int j = 0; j < kN; ++j) {
        const double x = (double)j / (double)(kN - 1), v = y[j];
        double pa = 1.0;
#pragma unroll
        for (int a = 0; a < M; ++a) {
            if (a >= m) break;
            double pb = pa;
#pragma unroll
            for (int b = 0; b < M; ++b) {
                if (b < a) continue;
                G[a][b] += pa * pb;
                pb *= x;
            }
            G[a][M] += pa * v;
            pa *= x;
        }
    }
#pragma unroll
    for (int a = 1; a < M; ++a)
#pragma unroll
        for (int b = 0; b < a; ++b) G[a][b] = G[b][a];
#pragma unroll
    for (int c = 0; c < M; ++c) {
        if (c >= m) break;
        int piv = c;
        double best = fabs(G[c][c]);
#pragma unroll
        for (int r = c + 1; r < M; ++r)
            if (r < m && fabs(G[r][c]) > best) {
                best = fabs(G[r][c]);
                piv = r;
            }
#pragma unroll
        for (int r = c + 1; r < M; ++r)
            if (r == piv)
#pragma unroll
                for (int b = 0; b <= M; ++b) {
                    const double t = G[c][b];
                    G[c][b] = G[r][b];
                    G[r][b] = t;
                }
        const double inv = 1.0 / G[c][c];
#pragma unroll
        for (int b = c; b <= M; ++b) G[c][b] *= inv;
#pragma unroll
        for (int r = 0; r < M; ++r) {
            if (r == c || r >= m) continue;
            const double f = G[r][c];
#pragma unroll
            for (int b = c; b <= M; ++b) G[r][b] -= f * G[c][b];
        }
    }
    for (int j = 0; j < kN; ++j) {
        const double x = (double)j / (double)(kN - 1);
        double v = 0.0;
#pragma unroll
        for (int a = M - 1; a >= 0; --a)
            if (a < m) v = v * x + G[a][M];
        out[j] = v;
    }
}

// Eigenvalues and leading eigenvectors of cov[blockIdx.x], one wave: lane = row, the matrix in
// registers. Householder reflectors stay in LDS for the eigenvectors; lane i bisects for the
// i-th largest eigenvalue down to 2^-54 of the largest entry; lanes 0 .. 2 solve for one
// eigenvector each (LU with partial pivoting, three inverse iterations, orthogonalised after
// each so that equal eigenvalues give orthonormal vectors too). Bound by FP64 instructions in
// one or two waves per SIMD, each waiting for its own chain: 17.5 KB of LDS let nine windows
// share a CU (2101 windows on the chip at once). A cyclic Jacobi over a workgroup per window,
// which computes all 51 eigenvectors, took 30 times the operations: 7.8 ms for 2101 windows with
// the covariances, now 0.48 + 0.18 ms (of which the bisection is 0.2, the fit 0.03).
__global__ __launch_bounds__(kWave, 3) void calib_pca_kernel(const CalibParams prm, int64_t first,
                                                        const double* __restrict__ cov,
                                                        double* __restrict__ evals_out,
                                                        double* __restrict__ loadings_out,
                                                        double* __restrict__ raw_out,
                                                        double* __restrict__ drifts_out)
{
    constexpr int F = kFactors;
    // s_vw: v and w of a Householder step (68 each: columns k + j past 50 read zeros), then the
    // eigenvectors
    __shared__ double s_vw[F * kN];
    __shared__ d2_t s_de[kN];          // d_j, e_{j-1}^2
    __shared__ double s_e[kN], s_ih[kN];
    __shared__ double s_h[(kN - 1) * kN / 2];
    __shared__ double s_lu[4][kN][F];  // 1 / U_ii, U_i,i+1, U_i,i+2, multiplier
    const int lane = threadIdx.x;
    const int64_t w = first + blockIdx.x;
    const double* C = cov + (int64_t)blockIdx.x * kN * kN;

    double a[kN];
    double big = 0.0;
#pragma unroll
    for (int j = 0; j < kN; ++j) {
        a[j] = lane < kN ? C[j * kN + lane] : 0.0;
        big = fmax(big, fabs(a[j]));
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) big = fmax(big, __shfl_xor(big, o));
    // a power of two, so that the entries' squares neither overflow nor vanish
    const int ex = big > 0.0 ? __builtin_amdgcn_frexp_exp(big) : 0;
#pragma unroll
    for (int j = 0; j < kN; ++j) a[j] = ldexp(a[j], -ex);
    for (int t = lane; t < F * kN; t += kWave) s_vw[t] = 0.0;
    __syncthreads();

    double *s_v = s_vw, *s_w = s_vw + 68;
    householder<kN, 0, 17>(a, lane, s_v, s_w, s_de, s_e, s_h, s_ih);
    householder<kN - 17, 17, 34>(a, lane, s_v, s_w, s_de, s_e, s_h, s_ih);
    householder<kN - 34, 34, kN - 2>(a, lane, s_v, s_w, s_de, s_e, s_h, s_ih);
    if (lane == kN - 2) {
        s_de[kN - 2][0] = a[0];
        s_e[kN - 2] = a[1];
        s_e[kN - 1] = 0.0;
    }
    if (lane == kN - 1) s_de[kN - 1][0] = a[1];
    __syncthreads();
    if (lane < kN) {
        const double e = lane > 0 ? s_e[lane - 1] : 0.0;
        s_de[lane][1] = fmax(e * e, 0x1p-118);
    }
    // Gershgorin's interval
    double lo = 0.0, hi = 0.0;
    if (lane < kN) {
        const double r = fabs(s_e[lane]) + (lane > 0 ? fabs(s_e[lane - 1]) : 0.0);
        lo = s_de[lane][0] - r;
        hi = s_de[lane][0] + r;
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        lo = fmin(lo, __shfl_xor(lo, o));
        hi = fmax(hi, __shfl_xor(hi, o));
    }
    const double hi0 = fmax(fabs(lo), fabs(hi));
    __syncthreads();
#pragma unroll 1
    for (int it = 0; it < 60; ++it) {
        const double x = 0.5 * (lo + hi);
        if (sturm_count(s_de, x) <= kN - 1 - lane) lo = x;
        else hi = x;
    }
    const double ev = 0.5 * (lo + hi);
    if (lane < kN) evals_out[w * kN + lane] = ldexp(ev, ex);


    // ---- eigenvectors of the tridiagonal: lane f < F solves for z_f, in s_z[f kN ..]; equal
    // eigenvalues are taken apart by a few roundings
    double* s_z = s_vw;
    const double sep = 0x1p-50 * hi0;
    double lam = __shfl(ev, 0);
    for (int f = 1; f < F; ++f) {
        const double below = fmin(__shfl(ev, f), __shfl(lam, f - 1) - sep);
        lam = lane >= f ? below : lam;
    }
    uint64_t swapped = 0;   // rows i and i + 1 exchanged
    constexpr double kTiny = 0x1p-53;
    if (lane < F) {
        double aa = s_de[0][0] - lam, bb = s_e[0];
        for (int i = 0; i < kN; ++i) {
            double c = i < kN - 1 ? s_e[i] : 0.0;
            const double dd = i < kN - 1 ? s_de[i + 1][0] - lam : 0.0, ee = i < kN - 1 ? s_e[i + 1] : 0.0;
            const bool swap = fabs(aa) < fabs(c);
            double pivot = swap ? c : aa;
            if (fabs(pivot) < kTiny) pivot = copysign(kTiny, pivot);
            const double inv = 1.0 / pivot, m = (swap ? aa : c) * inv;
            const double u1 = swap ? dd : bb, u2 = swap ? ee : 0.0;
            s_lu[0][i][lane] = inv;
            s_lu[1][i][lane] = i < kN - 1 ? u1 : 0.0;
            s_lu[2][i][lane] = u2;
            s_lu[3][i][lane] = m;
            if (swap) swapped |= 1ull << i;
            aa = (swap ? bb : dd) - m * u1;
            bb = swap ? -m * ee : ee;
            // any start with a part along each eigenvector
            const uint32_t u = (uint32_t)(i * F + lane + 1) * 2654435761u;
            s_z[lane * kN + i] = 0.5 + (double)(u >> 8) * 0x1p-24;
        }
    }
    double z[F] = {};
#pragma unroll 1
    for (int it = 0; it < 3; ++it) {
        if (lane < F) {
            double* y = s_z + lane * kN;
            double cur = y[0];
#pragma unroll 5
            for (int i = 0; i < kN - 1; ++i) {
                const double next = y[i + 1], m = s_lu[3][i][lane];
                const bool swap = swapped >> i & 1;
                y[i] = swap ? next : cur;
                cur = (swap ? cur : next) - m * (swap ? next : cur);
            }
            double x1 = cur * s_lu[0][kN - 1][lane], x2 = 0.0;
            y[kN - 1] = x1;
#pragma unroll 5
            for (int i = kN - 2; i >= 0; --i) {
                const double x = (y[i] - s_lu[1][i][lane] * x1 - s_lu[2][i][lane] * x2) * s_lu[0][i][lane];
                y[i] = x;
                x2 = x1;
                x1 = x;
            }
        }
        __syncthreads();
#pragma unroll
        for (int f = 0; f < F; ++f) {
            z[f] = lane < kN ? s_z[f * kN + lane] : 0.0;
#pragma unroll
            for (int rep = 0; rep < 2; ++rep) {
                const double n = wave_sum(z[f] * z[f]);
                z[f] *= n > 0.0 ? 1.0 / sqrt(n) : 0.0;
#pragma unroll
                for (int g = 0; g < f; ++g) z[f] = fma(-wave_sum(z[f] * z[g]), z[g], z[f]);
            }
            const double n = wave_sum(z[f] * z[f]);
            z[f] *= n > 0.0 ? 1.0 / sqrt(n) : 0.0;
            if (lane < kN) s_z[f * kN + lane] = z[f];
        }
        __syncthreads();
    }
    // the matrix's: the reflectors in reverse
#pragma unroll 1
    for (int k = kN - 3; k >= 0; --k) {
        const double v = lane > k && lane < kN ? s_h[k * (kN - 1) - k * (k - 1) / 2 + lane - k - 1] : 0.0;
        const double ih = s_ih[k];
        double dot[F];
#pragma unroll
        for (int f = 0; f < F; ++f) dot[f] = wave_sum(v * z[f]);
#pragma unroll
        for (int f = 0; f < F; ++f) z[f] = fma(-dot[f] * ih, v, z[f]);
    }
#pragma unroll
    for (int f = 0; f < F; ++f)
        if (lane < kN) s_z[f * kN + lane] = z[f];
    __syncthreads();

    // ---- signs (sum of components > 0, else the first component above 1e-9 in magnitude
    // positive), loadings and fits
    double* s_out = &s_lu[0][0][0];
    double* raw = s_z + (lane < F ? lane : 0) * kN;
    if (lane < F) {
        double sum = 0.0;
        for (int j = 0; j < kN; ++j) sum += raw[j];
        double sign = 1.0;
        if (fabs(sum) > 1e-9) {
            sign = sum > 0.0 ? 1.0 : -1.0;
        } else {
            for (int j = 0; j < kN; ++j)
                if (fabs(raw[j]) > 1e-9) {
                    sign = raw[j] > 0.0 ? 1.0 : -1.0;
                    break;
                }
        }
        const double top = ldexp(ev, ex), sl = sign * (top > 0.0 ? sqrt(top) : 0.0);
        for (int j = 0; j < kN; ++j) raw[j] = sl * raw[j];
        double* out = s_out + lane * kN;
        const int d = prm.degree[lane];
        if (d < 0) {
            for (int j = 0; j < kN; ++j) out[j] = raw[j];
        } else {
            fit_polynomial(raw, d + 1, out);
        }
    }
    __syncthreads();
    for (int t = lane; t < F * kN; t += kWave) {
        raw_out[w * F * kN + t] = s_z[t];
        loadings_out[w * F * kN + t] = s_out[t];
    }
    // drift: the cumulative Simpson rule of hjm_hjm_drift, lane = tenor, the same operations
    if (lane < kN) {
#pragma clang fp contract(off)
        const double h = prm.dtau;
        double drift = 0.0;
        for (int f = 0; f < F; ++f) {
            const double* y = s_out + f * kN;
            double sum = 0.0;
            if (lane == 1) {
                sum = h / 12.0 * (5.0 * y[0] + 8.0 * y[1] - y[2]);
            } else if (lane > 1) {
                const int even_end = lane % 2 == 0 ? lane : lane - 3;
                for (int i = 0; i < even_end; i += 2) sum += h / 3.0 * (y[i] + 4.0 * y[i + 1] + y[i + 2]);
                if (lane % 2 == 1)
                    sum += 3.0 * h / 8.0 * (y[lane - 3] + 3.0 * y[lane - 2] + 3.0 * y[lane - 1] + y[lane]);
            }
            drift += y[lane] * sum;
        }
        drifts_out[w * kN + lane] = drift;
    }
}

}  // namespace

extern "C" {

int hjm_calibrate_pca(const hjm_calibration* c, hjm_calibration_results* r)
{
    if (!c || !r || !c->curves || !r->eigenvalues || !r->volatilities || !r->drifts)
        return HJM_ERR_NULL;
    if (c->window < 3 || c->nwindows < 1 || c->step < 1 || c->nfactors < 1 ||
        c->nfactors > kMaxFactors || !(c->obs_per_year > 0.0) || !(c->dtau > 0.0))
        return HJM_ERR_ARG;
    if (c->nfactors != kFactors) return HJM_ERR_ARG;  // the path kernels take 3 loadings
    if ((int64_t)(c->nwindows - 1) * c->step + c->window > c->ncurves) return HJM_ERR_ARG;
    CalibParams prm{};
    prm.ncurves = c->ncurves;
    prm.window = c->window;
    prm.step = c->step;
    prm.nwindows = c->nwindows;
    prm.nfactors = c->nfactors;
    prm.obs_per_year = c->obs_per_year;
    prm.dtau = c->dtau;
    for (int k = 0; k < kMaxFactors; ++k) prm.degree[k] = -1;
    if (c->fit_degrees)
        for (int k = 0; k < c->nfactors; ++k) {
            if (c->fit_degrees[k] > kMaxDegree) return HJM_ERR_ARG;
            prm.degree[k] = c->fit_degrees[k];
        }
    for (int64_t i = 0; i < c->ncurves * kN; ++i)
        if (!isfinite(c->curves[i])) return HJM_ERR_ARG;

    DeviceGuard guard;
    HJM_TRY(guard.set(c->device));
    const size_t W = (size_t)c->nwindows, F = (size_t)c->nfactors;
    // windows at a time: bounds the covariances' buffer to 85 MB
    const int64_t batch = std::min<int64_t>(c->nwindows, 4096);
    double *d_curves = nullptr, *d_ev = nullptr, *d_ld = nullptr, *d_raw = nullptr, *d_cov = nullptr,
           *d_drift = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = dev_alloc(&d_curves, (size_t)c->ncurves * kN);
    if (rc == HJM_OK) rc = dev_alloc(&d_ev, W * kN);
    if (rc == HJM_OK) rc = dev_alloc(&d_ld, W * F * kN);
    if (rc == HJM_OK) rc = dev_alloc(&d_raw, W * F * kN);
    if (rc == HJM_OK) rc = dev_alloc(&d_drift, W * kN);
    if (rc == HJM_OK) rc = dev_alloc(&d_cov, (size_t)batch * kN * kN);
    if (rc == HJM_OK && (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess))
        rc = HJM_ERR_DEVICE;
    if (rc == HJM_OK &&
        hipMemcpy(d_curves, c->curves, (size_t)c->ncurves * kN * sizeof(double),
                  hipMemcpyHostToDevice) != hipSuccess)
        rc = HJM_ERR_DEVICE;
    if (rc == HJM_OK) {
        (void)hipEventRecord(e0, nullptr);
        for (int64_t first = 0; first < c->nwindows; first += batch) {
            const dim3 grid((unsigned)std::min<int64_t>(batch, c->nwindows - first));
            calib_cov_kernel<<<grid, kWave, 0, nullptr>>>(prm, first, d_curves, d_cov);
            calib_pca_kernel<<<grid, kWave, 0, nullptr>>>(prm, first, d_cov, d_ev, d_ld, d_raw, d_drift);
        }
        if (hipGetLastError() != hipSuccess) rc = HJM_ERR_LAUNCH;
        (void)hipEventRecord(e1, nullptr);
    }
    if (rc == HJM_OK && hipDeviceSynchronize() != hipSuccess) rc = HJM_ERR_LAUNCH;
    auto fetch = [&](double* to, const double* from, size_t n) {
        if (rc == HJM_OK && hipMemcpy(to, from, n * sizeof(double), hipMemcpyDeviceToHost) != hipSuccess)
            rc = HJM_ERR_DEVICE;
    };
    fetch(r->eigenvalues, d_ev, W * kN);
    fetch(r->volatilities, d_ld, W * F * kN);
    fetch(r->drifts, d_drift, W * kN);
    if (r->raw_loadings) fetch(r->raw_loadings, d_raw, W * F * kN);
    if (rc == HJM_OK && r->timings_ms) {
        float ms = 0.f;
        (void)hipEventElapsedTime(&ms, e0, e1);
        r->timings_ms[0] = ms;
    }
    const bool clean = hipStreamSynchronize(nullptr) == hipSuccess;
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    dev_free(clean, d_curves, d_ev, d_ld, d_raw, d_cov, d_drift);
    return rc;
}

}  // extern "C"
