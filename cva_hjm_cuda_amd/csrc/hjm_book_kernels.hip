// hjm_book_kernels.hip -- a portfolio's coefficient tables and matrix-core fragments, built on
// the device from the swap list, and the clearing of matured exposure rows.
//
// On the host these tables took 4 ms per plan at 1024 swaps in 128 sets x 61 dates (half a
// million coefficients, each split three ways, and 10 MB of uploads), most of a one-call CVA
// with Greeks; here they are a few launches of some microseconds over a 24 KB swap list.
#include "hjm_common.h"
#include "hjm_kernels.h"
#include "hjm_mfma_plan.h"

namespace hjm {

// V_g(t_e) = a_ge - sum_k gamma_gek P_k with, for every live swap (k_s = n_s - e > 0):
// a += sN, gamma_{k_s} += sN (the -sN P_{n} term), gamma_j += sN K dtau for j <= k_s. One
// workgroup per (date, set), thread j the coefficient of period j + 1: the set's swaps in the
// caller's order, one rounding per term (no product is fused into a sum).
__global__ __launch_bounds__(kWave) void book_tables_kernel(BookSwaps b, int nsets, double* __restrict__ coef,
                                                            double* __restrict__ a, int* __restrict__ kmax)
{
#pragma clang fp contract(off)
    const int set = blockIdx.x, e = blockIdx.y, j = threadIdx.x;
    const int64_t row = (int64_t)e * nsets + set;
    double g = 0.0, base = 0.0;
    int top = 0;
    for (int s = b.first[set]; s < b.first[set + 1]; ++s) {
        const int k = b.periods[s] - e;
        if (k <= 0) continue;
        base += b.notional[s];
        if (j == k - 1) g += b.notional[s];
        if (j < k) g += b.coupon[s];
        top = max(top, k);
    }
    if (j < kMaxPeriods) coef[row * kMaxPeriods + j] = g;
    if (j == 0) {
        a[row] = base;
        kmax[row] = top;
    }
}

// three bf16 parts of w, rounded to nearest (ties to even)
__device__ __forceinline__ void bf16_parts(double w, uint16_t (&p)[3])
{
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        uint32_t u = __builtin_bit_cast(uint32_t, (float)w);
        u += 0x7fffu + ((u >> 16) & 1u);
        p[i] = (uint16_t)(u >> 16);
        w -= (double)__builtin_bit_cast(float, u & 0xffff0000u);
    }
}

// value(i) of 8 consecutive K entries as a lane's three fragments
template <class F>
__device__ __forceinline__ void store_parts(uint16_t* frag, int64_t first, int lane, F value)
{
    uint16_t p[kMfmaParts][8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        uint16_t q[3];
        bf16_parts(value(i), q);
#pragma unroll
        for (int k = 0; k < kMfmaParts; ++k) p[k][i] = q[k];
    }
#pragma unroll
    for (int k = 0; k < kMfmaParts; ++k) {
        uint32_t* o = reinterpret_cast<uint32_t*>(frag + ((first + k) * kWave + lane) * 8);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = p[k][2 * i] | ((uint32_t)p[k][2 * i + 1] << 16);
    }
}

// The valuation's tables (hjm_mfma_plan.h): -gamma's fragments of M-tile blockIdx.x at date
// blockIdx.y, its sets' constants and largest live period. One wave.
__global__ __launch_bounds__(kWave) void value_fragments_kernel(const double* __restrict__ coef,
                                                                const double* __restrict__ a,
                                                                const int* __restrict__ kmax, int nsets,
                                                                uint16_t* __restrict__ frag,
                                                                float* __restrict__ apad, int* __restrict__ tilek)
{
    const int m = blockIdx.x, e = blockIdx.y, lane = threadIdx.x, mt = gridDim.x;
    const int64_t tile = (int64_t)e * mt + m;
    const int g = 16 * m + lane % 16;
    const int64_t row = (int64_t)e * nsets + (g < nsets ? g : 0);
    for (int c = 0; c < 2; ++c)
        store_parts(frag, (tile * 2 + c) * kMfmaParts, lane, [&](int i) {
            const int kk = 32 * c + 8 * (lane / 16) + i;
            return (g < nsets && kk < kMaxPeriods) ? -coef[row * kMaxPeriods + kk] : 0.0;
        });
    int top = (lane < 16 && g < nsets) ? kmax[row] : 0;
    if (lane < 16) apad[tile * 16 + lane] = g < nsets ? (float)a[row] : 0.f;
    for (int o = 8; o > 0; o >>= 1) top = max(top, __shfl_xor(top, o, kWave));
    if (lane == 0) tilek[tile] = top;
}

// The adjoint's second product (hjm_mfma_plan.h): -gamma^T of period tile blockIdx.x % 4, K
// chunk blockIdx.x / 4, date blockIdx.y. One wave.
__global__ __launch_bounds__(kWave) void adjoint_fragments_kernel(const double* __restrict__ coef, int nsets,
                                                                  int nch, uint16_t* __restrict__ frag)
{
    const int pm = blockIdx.x % 4, c = blockIdx.x / 4, e = blockIdx.y, lane = threadIdx.x;
    const int kk = 16 * pm + lane % 16;
    store_parts(frag, (((int64_t)e * 4 + pm) * nch + c) * kMfmaParts, lane, [&](int i) {
        const int set = 16 * (2 * c + i / 4) + 4 * (lane / 16) + i % 4;
        return (set < nsets && kk < kMaxPeriods)
                   ? -coef[((int64_t)e * nsets + set) * kMaxPeriods + kk]
                   : 0.0;
    });
}

// Zeros in the exposure rows whose set has no live swap (the valuation never writes them).
template <typename Real>
__global__ __launch_bounds__(kBlock) void clear_matured_kernel(const int* __restrict__ kmax, int64_t paths,
                                                               Real* __restrict__ ex)
{
    if (kmax[blockIdx.y] > 0) return;
    Real* row = ex + (int64_t)blockIdx.y * paths;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < paths; i += (int64_t)gridDim.x * kBlock)
        row[i] = (Real)0;
}

hipError_t launch_book_tables(const BookSwaps& b, int nsets, int ndates, double* coef, double* a, int* kmax,
                              hipStream_t st)
{
    book_tables_kernel<<<dim3((unsigned)nsets, (unsigned)ndates), kWave, 0, st>>>(b, nsets, coef, a, kmax);
    return hipGetLastError();
}

hipError_t launch_value_fragments(const double* coef, const double* a, const int* kmax, int nsets, int ndates,
                                  uint16_t* frag, float* apad, int* tilek, hipStream_t st)
{
    value_fragments_kernel<<<dim3((unsigned)value_mtiles(nsets), (unsigned)ndates), kWave, 0, st>>>(
        coef, a, kmax, nsets, frag, apad, tilek);
    return hipGetLastError();
}

hipError_t launch_adjoint_fragments(const double* coef, int nsets, int ndates, uint16_t* frag, hipStream_t st)
{
    const int nch = (value_mtiles(nsets) + 1) / 2;
    adjoint_fragments_kernel<<<dim3((unsigned)(4 * nch), (unsigned)ndates), kWave, 0, st>>>(coef, nsets, nch,
                                                                                         frag);
    return hipGetLastError();
}

hipError_t launch_clear_matured(const int* kmax, int rows, int64_t paths, void* ex, int elem_bytes,
                                hipStream_t st)
{
    const dim3 grid((unsigned)std::min<int64_t>(64, (paths + kBlock - 1) / kBlock), (unsigned)rows);
    if (elem_bytes == 8)
        clear_matured_kernel<double><<<grid, kBlock, 0, st>>>(kmax, paths, static_cast<double*>(ex));
    else
        clear_matured_kernel<float><<<grid, kBlock, 0, st>>>(kmax, paths, static_cast<float*>(ex));
    return hipGetLastError();
}

}  // namespace hjm
