// hjm_map_kernels.hip -- the FP32 matrix-core maps (the path kernels' block map and the reverse
// sweep's), built on the device.
//
// Every column of a map is the walk of one 51-vector through the steps of a block, so a
// workgroup is one wave with a column, lane = tenor, its neighbours a shuffle away. Bound by
// the 50 steps' chain, about 250 cycles each. On the host (the same operations, bit for bit)
// the two maps took 100 to 300 us of every call that makes its plan; here the block map
// takes 33 us (its fragments are written two bytes at a time) and the sweep's 5.
#include "hjm_common.h"
#include "hjm_kernels.h"
#include "hjm_mfma_plan.h"

namespace hjm {

__device__ __forceinline__ uint16_t bf16_part(double& w)
{
    const uint16_t h = bf16_rne(w);
    w -= bf16_value(h);
    return h;
}

// K index of the block map that multiplies curve row r (mfma_column inverted), and shock
// (step, factor); the drift's constant is the shock (50, 0).
__host__ __device__ constexpr int curve_k(int r)
{
    return 32 * (r / 32) + 8 * (r % 16 / 4) + 4 * (r / 16 % 2) + r % 4;
}
__host__ __device__ constexpr int shock_k(int step, int factor)
{
    const int v = 3 * (step / 4) + factor;
    return 32 * (2 + v / 8) + 8 * (step % 4) + v % 8;
}

// Workgroup b < 51: the curve column of row b; 51 .. 53: factor b - 51's 50 shock columns; 54:
// the drift's. vec: the three loadings times sqrt(dt), then the drift times dt. up: the
// shocks' scale. frag is zero elsewhere. The operations of mfma_block_map_dense, in its order.
template <bool kPf>
__global__ __launch_bounds__(kWave) void block_map_kernel(const BlockMapParams prm, uint16_t* __restrict__ frag)
{
#pragma clang fp contract(off)
    constexpr int n = kTenors, S = kMfmaStride;
    const int j = threadIdx.x, b = blockIdx.x;
    const double c = prm.c, here = j == n - 1 ? 1.0 + c : 1.0 - c, there = j == n - 1 ? -c : c;
    auto apply = [&](double u) {
        const double up = __shfl_down(u, 1), down = __shfl_up(u, 1);
        const double a = here * u, o = there * (j == n - 1 ? down : up);
        return j == n - 1 ? o + a : a + o;
    };
    auto put = [&](int row, int k, double w) {
        if (j >= n || row / 16 >= prm.mtiles) return;
        const int m = row / 16, ch = k / 32;
        const size_t at = (size_t)(row % 16 + 16 * (k % 32 / 8)) * 8 + k % 8;
        auto part = [&](int p) -> uint16_t& { return frag[(size_t)mfma_frag(m, ch, p) * kWave * 8 + at]; };
        if (ch < 2) {
            // an entry far below its row's largest has no part among the leading ones, whose
            // products the matrix cores drop below 2^-24 of the largest beside them
            const bool minor = fabs(w) < (row < n ? kMinorCurve : kMinorSum);
            part(0) = minor ? (uint16_t)0 : bf16_part(w);
            part(1) = bf16_part(w);
            part(2) = bf16_part(w);
        } else {
            const uint16_t h = fp16_rne((float)(w * prm.up));
            part(0) = h;
            part(1) = fp16_rne((float)(w * prm.up - fp16_value(h)));
        }
    };
    if (b < n) {
        double u = j == b ? 1.0 : 0.0, sum = 0.0, first = 0.0;
        for (int s = 0; s < S; ++s) {
            first += u;
            u = apply(u);
            sum += u;
        }
        const int k = curve_k(b);
        put(j, k, u);
        if constexpr (kPf) {
            if (j == 0) put(n, k, first);
        } else {
            put(n + j, k, sum);
        }
        return;
    }
    const int f = b - n;
    double u = j < n ? prm.vec[f][j] : 0.0, acc = 0.0;
    double cu = 0.0, ca = 0.0;   // the drift's column
    for (int q = 0; q < S; ++q) {
        const double left = acc;   // of tenor 0: the short rate's left-point sum
        acc += u;
        const double second = kPf ? left : acc;
        if (f < 3) {
            const int k = shock_k(S - 1 - q, f);
            put(j, k, u);
            if (!kPf || j == 0) put(n + j, k, second);
        } else {
            cu += u;
            ca += second;
        }
        u = apply(u);
    }
    if (f == 3) {
        const int k = shock_k(S, 0);
        put(j, k, cu);
        if (!kPf || j == 0) put(n + j, k, ca);
    }
}

hipError_t launch_block_map(const BlockMapParams& prm, bool pf, uint16_t* frag, hipStream_t st)
{
    const hipError_t e = hipMemsetAsync(frag, 0, block_map_elems(prm.mtiles) * sizeof(uint16_t), st);
    if (e != hipSuccess) return e;
    if (pf) block_map_kernel<true><<<kTenors + 4, kWave, 0, st>>>(prm, frag);
    else block_map_kernel<false><<<kTenors + 4, kWave, 0, st>>>(prm, frag);
    return hipGetLastError();
}

// Workgroup m: K column m of the sweep's map and, below `tables`, row m of ptab (hjm_mfma_plan.h).
__global__ __launch_bounds__(kWave) void sweep_map_kernel(double c, int tables, uint16_t* __restrict__ frag,
                                                        float* __restrict__ ptab)
{
#pragma clang fp contract(off)
    constexpr int n = kTenors, S = kMfmaStride;
    const int j = threadIdx.x, m = blockIdx.x;
    // column m of the powers of T^T with row 49 holding x_49 + x_50: y_j = (1 - c) x_j + c x_{j-1}
    // below it, y_49 = x_49 + c x_48, y_50 = x_50 + c x_49; b: of their sum, from tenor m
    // (tenor 50 adds to row 49 too)
    auto step = [&](double x) {
        const double below = __shfl_up(x, 1);
        double y = j < n - 2 ? (1.0 - c) * x : x;
        if (j > 0) y += c * below;
        return j < n ? y : 0.0;
    };
    double a = j == m ? 1.0 : 0.0, t = j == m || (m == n - 1 && j == n - 2) ? 1.0 : 0.0, b = 0.0;
    for (int q = 0; q < S; ++q) {
        b += t;
        t = step(t);
        a = step(a);
    }
    if (j >= n) return;
    if (m < tables) ptab[m * 64 + j] = (float)b;
    const int ch = m / 32, i = 4 * (m / 16 % 2) + m % 4, l = j % 16 + 16 * (m % 16 / 4);
#pragma unroll
    for (int p = 0; p < kMfmaParts; ++p)
        frag[(((size_t)(j / 16 * 2 + ch) * kMfmaParts + p) * kWave + l) * 8 + i] = bf16_part(a);
}

hipError_t launch_sweep_map(double c, bool pf, uint16_t* frag, float* ptab, hipStream_t st)
{
    hipError_t e = hipMemsetAsync(frag, 0, kSweepMapElems * sizeof(uint16_t), st);
    if (e == hipSuccess) e = hipMemsetAsync(ptab, 0, sweep_table_elems(pf) * sizeof(float), st);
    if (e != hipSuccess) return e;
    sweep_map_kernel<<<kTenors, kWave, 0, st>>>(c, pf ? 1 : kTenors, frag, ptab);
    return hipGetLastError();
}

}  // namespace hjm
