// hjm_adjoint_mfma.hip -- the adjoint's reverse sweep on the matrix cores, gfx950.
//
// Within a block of S = 50 steps the reverse recursion lambda <- T^T lambda + mu is linear in
// the block-end adjoint lambda_e and in mu, so the loading gradients
//   dJ/dsigma_k = sqrt(dt) sum over paths, blocks and steps of lambda(s) phi_k(s),
//   lambda(s) = (T^T)^{S-1-s} lambda_e + sum_{q < S-1-s} (T^T)^q mu,
// need only the products of lambda_e and mu with the block's 150 shocks, summed over blocks
// and paths -- one contraction over the paths,
//   M[row][3 s + k] = sum_{p, b} x_row(p, b) phi_k(s; p, b),   x = (lambda_e, mu),
// to which the host applies the powers of T^T once (FP64, adjoint_gradients). Column 150 is
// the constant 1 (the sums of lambda_e and mu for the drift gradient), column 151 takes the
// adjoint at time 0. Per path and block that replaces 50 steps of 130 FP32 instructions by
// 64 .. 128 rows x 160 columns of matrix products and one 64 x 64 map for the recursion.
//
// A wave owns 32 paths (two N-tiles) at a time and every accumulator of M for them (R x CT
// tiles of 16 x 16, in AGPRs: one wave per SIMD). lambda lives in the accumulator layout
// (lane l: rows 16 m + 4 (l / 16) + r of path l % 16), which is the next recursion's B operand
// as in the path kernels; for the contraction, whose K runs over the paths, the rows pass
// through the wave's LDS to the A layout (row l % 16, paths 4 g + i of either N-tile, g = l /
// 16). The shocks come straight from their [step][factor][path] rows: lane l reads the same 8
// paths of column l % 16, five column tiles ahead. All products are six bf16 split products
// (FP32 accuracy). Bound by the shocks' traffic (12 B per path-step) and the matrix cores at
// about the same time.
#include <algorithm>

#include "hjm_common.h"
#include "hjm_kernels.h"
#include "hjm_mfma_ops.h"
#include "hjm_mfma_plan.h"
#include "hjm_rng.h"

namespace hjm {

typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));   // any dword address

constexpr int kSweepWaves = 4;
constexpr int kSweepBlock = kSweepWaves * kWave;
constexpr int kSweepUnit = 32;                     // paths of a wave at a time
constexpr int kSweepCols = 160;                    // 150 shocks, 1, time 0, padding
constexpr int kSweepMapFrags = 4 * 2 * kMfmaParts; // one 64 x 64 map
constexpr int kRing = 5;                           // column tiles read ahead

template <bool kPf, int R>
constexpr int sweep_lds_floats()
{
    return (kPf ? 1 : 2) * kSweepMapFrags * kWave * 4 + kSweepWaves * kSweepUnit * (16 * R + 4);
}

// six split products for the R row tiles in turn
template <int R>
__device__ __forceinline__ void outer_tile(const Split8 (&xa)[R], const Split8& b, f4_t (&acc)[R])
{
#pragma unroll
    for (int m = 0; m < R; ++m) acc[m] = mfma_bf16(xa[m].h, b.h, acc[m]);
#pragma unroll
    for (int m = 0; m < R; ++m) acc[m] = mfma_bf16(xa[m].h, b.m, acc[m]);
#pragma unroll
    for (int m = 0; m < R; ++m) acc[m] = mfma_bf16(xa[m].m, b.h, acc[m]);
#pragma unroll
    for (int m = 0; m < R; ++m) acc[m] = mfma_bf16(xa[m].h, b.l, acc[m]);
#pragma unroll
    for (int m = 0; m < R; ++m) acc[m] = mfma_bf16(xa[m].l, b.h, acc[m]);
#pragma unroll
    for (int m = 0; m < R; ++m) acc[m] = mfma_bf16(xa[m].m, b.m, acc[m]);
}

// kPf false (reference semantics): R = 4 + the tiles of live mu rows (row 64 + j: mu_j);
// seed_a = gx, seed_b = gA, [slot][path]. kPf true: R = 4, mu (a scalar, on tenor 0) is row 51;
// seed_a = gbar [date][tenor][path], seed_b = beta [date][path]. Columns 16 CT blockIdx.y ..
// are this workgroup's. maps: (T^T)^S in the path kernels' K order, then (reference) sum_{q <
// S} (T^T)^q; for kPf its column of tenor 0 sits in the K slot of row 51.
template <bool kPf, int R, int CT>
__global__ __attribute__((amdgpu_flat_work_group_size(kSweepBlock, kSweepBlock), amdgpu_waves_per_eu(1, 1)))
void adjoint_mfma_kernel(const SweepGrid g, const u4_t* __restrict__ maps, const float* __restrict__ zs,
                         const float* __restrict__ seed_a, const float* __restrict__ seed_b,
                         float* __restrict__ partials)
{
    constexpr int kMu = R - 4, kMaps = kPf ? 1 : 2, kPitch = 16 * R + 4;
    extern __shared__ float lds[];
    u4_t* lds_map = reinterpret_cast<u4_t*>(lds);
    for (int t = threadIdx.x; t < kMaps * kSweepMapFrags * kWave; t += kSweepBlock) lds_map[t] = maps[t];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int grp = lane / 16, col = lane % 16;
    float* xt = lds + kMaps * kSweepMapFrags * kWave * 4 + wave * kSweepUnit * kPitch;
    __syncthreads();

    const int64_t P = g.paths;
    const int t0 = (int)blockIdx.y * CT;
    f4_t acc[CT][R];
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
        for (int m = 0; m < R; ++m) acc[t][m] = f4_t{0.f, 0.f, 0.f, 0.f};

    const int64_t first = ((int64_t)blockIdx.x * kSweepWaves + wave) * g.units;
    for (int64_t unit = first; unit < first + g.units; ++unit) {
        const int64_t base = g.begin + unit * kSweepUnit;   // paths [begin, end) of this launch
        if (base >= g.end) break;
        const bool whole = base + kSweepUnit <= g.end;      // wave-uniform
        const float* zrow = zs + (base - g.begin) + 4 * grp;
        float ring[kRing][8];
        auto load_tile = [&](int b, int t, float (&d)[8]) {
            const int n = 16 * (t0 + t) + col;
            const float* q = zrow + (int64_t)(b * 3 * kMfmaStride + (n < 3 * kMfmaStride ? n : 0)) * g.zld;
            if (whole) {
                const f4u_t lo = *reinterpret_cast<const f4u_t*>(q), hi = *reinterpret_cast<const f4u_t*>(q + 16);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    d[i] = lo[i];
                    d[4 + i] = hi[i];
                }
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int o = i < 4 ? i : 12 + i;
                    d[i] = base + 4 * grp + o < g.end ? q[o] : 0.f;
                }
            }
        };
        int64_t path[2];
        bool live[2];
        float x[2][16], mu[2][kMu > 0 ? 4 * kMu : 1], mus[2] = {0.f, 0.f};
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            path[n] = base + 16 * n + col;
            live[n] = path[n] < g.end;
#pragma unroll
            for (int i = 0; i < 16; ++i) x[n][i] = 0.f;
#pragma unroll
            for (int i = 0; i < 4 * kMu; ++i) mu[n][i] = 0.f;
        }
        // rows of date e: x += gbar (kPf)
        auto add_rows = [&](int e) {
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int row = 16 * (i / 4) + 4 * grp + i % 4;
                    if (row < kTenors)
                        x[n][i] += live[n] ? seed_a[((int64_t)e * kTenors + row) * P + path[n]] : 0.f;
                }
        };
        if constexpr (kPf) add_rows(g.hi + 1);
#pragma unroll
        for (int t = 0; t < kRing; ++t) load_tile(g.hi, t, ring[t]);

        // the rows of x (and mu) in the A layout, split
        auto rows_to_a = [&](Split8 (&xa)[R]) {
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int m = 0; m < R; ++m) {
                    f4_t v;
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = m < 4 ? x[n][4 * (m < 4 ? m : 0) + r] : mu[n][m < 4 ? 0 : 4 * (m - 4) + r];
                    *reinterpret_cast<f4_t*>(xt + (16 * n + col) * kPitch + 16 * m + 4 * grp) = v;
                }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int m = 0; m < R; ++m) {
                float v[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = xt[(4 * grp + (i < 4 ? i : 12 + i)) * kPitch + 16 * m + col];
                xa[m] = split8(v);
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            __builtin_amdgcn_wave_barrier();
        };

        for (int b = g.hi; b >= g.lo; --b) {
            // injections at the end of block b
            if constexpr (kPf) {
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    mus[n] += live[n] ? g.dt * seed_b[(int64_t)(b + 1) * P + path[n]] : 0.f;
                    if (grp == 0) x[n][15] = mus[n];   // row 51
                }
            } else {
                const int slot = b + 1, at = 4 * (slot / 16) + slot % 4;
                const bool mine = grp == (slot % 16) / 4;
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    const bool on = live[n] && mine;
                    const float sx = on ? seed_a[(int64_t)slot * P + path[n]] : 0.f;
                    const float sa = on ? seed_b[(int64_t)slot * P + path[n]] : 0.f;
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (i == at) x[n][i] += sx + sa;
#pragma unroll
                    for (int i = 0; i < 4 * kMu; ++i)
                        if (i == at) mu[n][i] += sa;
                }
            }
            Split8 xa[R];
            rows_to_a(xa);
            // the contraction, one column tile at a time
#pragma unroll
            for (int t = 0; t < CT; ++t) {
                float z[8];
                const int n = 16 * (t0 + t) + col;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    z[i] = ring[t % kRing][i];
                    if (16 * t + 15 + 16 * (10 - CT) >= 3 * kMfmaStride)   // possibly the last tile
                        z[i] = n < 3 * kMfmaStride ? z[i] : (n == 3 * kMfmaStride ? 1.f : 0.f);
                }
                const Split8 bz = split8(z);
                if (t + kRing < CT) load_tile(b, t + kRing, ring[t % kRing]);
                else if (b > g.lo) load_tile(b - 1, t + kRing - CT, ring[t % kRing]);
                outer_tile<R>(xa, bz, acc[t]);
                __builtin_amdgcn_sched_barrier(0);
            }
            // the recursion: x <- (T^T)^S x + (sum_q (T^T)^q) mu
            uint32_t off = (uint32_t)lane;
            asm volatile("" : "+v"(off));
            f4_t big[4][2], small[4][2];
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int n = 0; n < 2; ++n) big[m][n] = small[m][n] = f4_t{0.f, 0.f, 0.f, 0.f};
            auto apply = [&](const u4_t* map, int c, const Split8 (&v)[2]) {
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    if (!kPf && c == 1 && m < 2) continue;   // rows <= 31 take no tenor >= 32
                    const u4_t* a = map + ((m * 2 + c) * kMfmaParts) * kWave + off;
                    const u4_t ah = a[0], am = a[kWave], al = a[2 * kWave];
#pragma unroll
                    for (int n = 0; n < 2; ++n) big[m][n] = mfma_bf16(ah, v[n].h, big[m][n]);
#pragma unroll
                    for (int n = 0; n < 2; ++n) small[m][n] = mfma_bf16(ah, v[n].m, small[m][n]);
#pragma unroll
                    for (int n = 0; n < 2; ++n) small[m][n] = mfma_bf16(am, v[n].h, small[m][n]);
#pragma unroll
                    for (int n = 0; n < 2; ++n) small[m][n] = mfma_bf16(ah, v[n].l, small[m][n]);
#pragma unroll
                    for (int n = 0; n < 2; ++n) small[m][n] = mfma_bf16(al, v[n].h, small[m][n]);
#pragma unroll
                    for (int n = 0; n < 2; ++n) small[m][n] = mfma_bf16(am, v[n].m, small[m][n]);
                }
            };
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                Split8 v[2];
#pragma unroll
                for (int n = 0; n < 2; ++n) v[n] = split8(&x[n][8 * c]);
                apply(lds_map, c, v);
                if constexpr (kMu > 0) {
                    if (8 * c < 4 * kMu) {
#pragma unroll
                        for (int n = 0; n < 2; ++n) {
                            float w[8];
#pragma unroll
                            for (int i = 0; i < 8; ++i) w[i] = 8 * c + i < 4 * kMu ? mu[n][8 * c + i < 4 * kMu ? 8 * c + i : 0] : 0.f;
                            v[n] = split8(w);
                        }
                        apply(lds_map + kSweepMapFrags * kWave, c, v);
                    }
                }
            }
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int m = 0; m < 4; ++m)
#pragma unroll
                    for (int r = 0; r < 4; ++r) x[n][4 * m + r] = big[m][n][r] + small[m][n][r];
            if constexpr (kPf) add_rows(b);
        }
        // time 0: column 151 takes the rows themselves (reference: the seeds of slot 1, whose
        // gA is live in all S steps of the frozen block 0, on tenor 1)
        if constexpr (!kPf) {
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                const bool on = live[n] && grp == 0;
                const float sx = on ? seed_a[P + path[n]] : 0.f, sa = on ? seed_b[P + path[n]] : 0.f;
                x[n][1] += sx + (float)kMfmaStride * sa;
            }
        }
        if (t0 + CT == kSweepCols / 16) {
            Split8 xa[R];
            rows_to_a(xa);
            float one[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) one[i] = col == 151 % 16 ? 1.f : 0.f;
            outer_tile<R>(xa, split8(one), acc[CT - 1]);
        }
    }

    // the workgroup's sum, in wave order, and its rows of partials [16 R][160]
    __syncthreads();
    for (int w = 0; w < kSweepWaves; ++w) {
        if (wave == w) {
#pragma unroll
            for (int t = 0; t < CT; ++t)
#pragma unroll
                for (int m = 0; m < R; ++m)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        float* o = lds + ((t * R + m) * 4 + r) * kWave + lane;
                        *o = w ? *o + acc[t][m][r] : acc[t][m][r];
                    }
        }
        __syncthreads();
    }
    float* out = partials + (int64_t)blockIdx.x * (16 * R * kSweepCols);
    for (int e = threadIdx.x; e < CT * R * 4 * kWave; e += kSweepBlock) {
        const int l = e % kWave, r = e / kWave % 4, m = e / (4 * kWave) % R, t = e / (4 * kWave * R);
        out[(16 * m + 4 * (l / 16) + r) * kSweepCols + 16 * (t0 + t) + l % 16] = lds[e];
    }
}

// out[c] = the FP64 sum of partials[r][c] over the rows r, in a fixed order.
__global__ __launch_bounds__(kBlock) void sweep_sum_kernel(const float* __restrict__ partials, int64_t rows,
                                                           int cols, double* __restrict__ out)
{
    __shared__ double red[kBlock / kWave][kWave];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int c = blockIdx.x * kWave + lane;   // cols is a multiple of 64
    double s = 0.0;
    for (int64_t r = wave; r < rows; r += kBlock / kWave) s += (double)partials[r * cols + c];
    red[wave][lane] = s;
    __syncthreads();
    if (wave == 0) {
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < kBlock / kWave; ++w) t += red[w][lane];
        out[c] = t;
    }
}

// The shocks of blocks [lo, hi] and paths [begin, begin + count) as the path kernels keep
// them: zs[(50 b + t)][factor][count]. Lane = path, the wave-uniform (class, call) of a block
// spread over the workgroup's waves.
__global__ __launch_bounds__(kBlock) void sweep_shocks_kernel(uint32_t seed_lo, uint32_t seed_hi, int64_t path0,
                                                              int64_t begin, int64_t count, int lo,
                                                              int64_t zld, float* __restrict__ zs)
{
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int64_t p = (int64_t)blockIdx.x * kWave + lane;
    const int b = lo + (int)blockIdx.y;
    if (p >= count) return;
    for (int it = wave; it < 40; it += kBlock / kWave) {
        const int cls = it % 4, c = it / 4;
        float z[4];
        stream_call(seed_lo, seed_hi, (uint32_t)(path0 + begin + p), (uint32_t)b, (uint32_t)cls, (uint32_t)c, z);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int j = 4 * c + e, t = 4 * (j / 3) + cls;
            if (t < kMfmaStride) zs[(int64_t)((b * kMfmaStride + t) * 3 + j % 3) * zld + p] = z[e];
        }
    }
}

// mu rows 64 + j of the reference sweep: j up to the last slot
int sweep_row_tiles(bool pf, int ndates) { return pf ? 4 : 4 + ndates / 16 + 1; }

int sweep_units(int64_t paths)
{
    // one wave per SIMD of 256 CUs: more paths, more units per wave
    const int64_t units = (paths + kSweepUnit - 1) / kSweepUnit;
    return (int)std::max<int64_t>(1, (units + 1023) / 1024);
}

int64_t sweep_group(int64_t paths) { return (int64_t)kSweepWaves * sweep_units(paths) * kSweepUnit; }

template <bool kPf, int R, int CT>
static hipError_t sweep_launch(const SweepGrid& g, const u4_t* maps, const float* zs, const float* a,
                               const float* b, float* partials, hipStream_t st)
{
    const size_t lds = std::max<size_t>(sizeof(float) * sweep_lds_floats<kPf, R>(),
                                        sizeof(float) * (size_t)CT * R * 4 * kWave);
    const void* fn = (const void*)adjoint_mfma_kernel<kPf, R, CT>;
    const hipError_t err = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) return err;
    const int64_t per = (int64_t)kSweepWaves * g.units * kSweepUnit;
    const dim3 grid((unsigned)((g.end - g.begin + per - 1) / per), kSweepCols / 16 / CT);
    adjoint_mfma_kernel<kPf, R, CT><<<grid, kSweepBlock, lds, st>>>(g, maps, zs, a, b, partials);
    return hipGetLastError();
}

hipError_t launch_adjoint_mfma(const SweepGrid& g, bool pf, const uint16_t* maps, const float* zs,
                               const float* seed_a, const float* seed_b, float* partials, hipStream_t st)
{
    if (g.begin < 0 || g.end <= g.begin || g.end > g.paths || g.hi < g.lo) return hipErrorInvalidValue;
    const u4_t* m = reinterpret_cast<const u4_t*>(maps);
    if (pf) return sweep_launch<true, 4, 10>(g, m, zs, seed_a, seed_b, partials, st);
    switch (sweep_row_tiles(false, g.hi + 1)) {
    case 5: return sweep_launch<false, 5, 10>(g, m, zs, seed_a, seed_b, partials, st);
    case 6: return sweep_launch<false, 6, 10>(g, m, zs, seed_a, seed_b, partials, st);
    case 7: return sweep_launch<false, 7, 5>(g, m, zs, seed_a, seed_b, partials, st);
    default: return sweep_launch<false, 8, 5>(g, m, zs, seed_a, seed_b, partials, st);
    }
}

hipError_t launch_sweep_sum(const float* partials, int64_t rows, int cols, double* out, hipStream_t st)
{
    sweep_sum_kernel<<<(unsigned)(cols / kWave), kBlock, 0, st>>>(partials, rows, cols, out);
    return hipGetLastError();
}

hipError_t launch_sweep_shocks(uint64_t seed, int64_t path0, const SweepGrid& g, float* zs, hipStream_t st)
{
    const dim3 grid((unsigned)((g.end - g.begin + kWave - 1) / kWave), (unsigned)(g.hi - g.lo + 1));
    sweep_shocks_kernel<<<grid, kBlock, 0, st>>>((uint32_t)seed, (uint32_t)(seed >> 32), path0, g.begin,
                                                 g.end - g.begin, g.lo, g.zld, zs);
    return hipGetLastError();
}

}  // namespace hjm
