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
// A pair of waves owns 32 paths (two N-tiles, one each) at a time; each wave holds half of M's
// column tiles (R x 5 tiles of 16 x 16). lambda lives in the accumulator layout (lane l: rows
// 16 m + 4 (l / 16) + r of path l % 16), which is the next recursion's B operand as in the
// path kernels; for the contraction, whose K runs over the paths, the pair's rows pass
// through LDS to the A layout (row l % 16, paths 4 g + i of either N-tile, g = l / 16). mu
// changes by one entry per block (reference: slot b + 1's; portfolio: tenor 0's), so its rows
// stay in LDS and its part of the recursion is a running vector updated by one column of
// sum_q (T^T)^q. The shocks come straight from their [step][factor][path] rows: lane l reads
// the same 8 paths of column l % 16, tiles ahead of their use. All products are six bf16 split
// products (FP32 accuracy). Bound by the shocks' traffic, 12 B per path-step: a unit's 19 KB
// take longer at HBM rate than its 312 .. 372 products.
#include <algorithm>

#include "hjm_common.h"
#include "hjm_kernels.h"
#include "hjm_mfma_ops.h"
#include "hjm_mfma_plan.h"
#include "hjm_rng.h"

namespace hjm {

typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));   // any dword address

// A load at a wave-uniform base plus the lane's 32-bit byte offset (scalar-base addressing).
template <typename T>
__device__ __forceinline__ T load_at(const float* base, uint32_t off)
{
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + off);
}

constexpr int kSweepPairs = 2;                     // per workgroup
constexpr int kSweepBlock = 2 * kSweepPairs * kWave;
constexpr int kSweepUnit = 32;                     // paths of a pair at a time
constexpr int kSweepCols = 160;                    // 150 shocks, 1, time 0, padding
constexpr int kSweepTiles = 5;                     // column tiles per wave
constexpr int kSweepMapFrags = 4 * 2 * kMfmaParts; // the 64 x 64 map

// floats of LDS: the map, and per pair the rows [path][row] and their split fragments
template <int R>
constexpr int sweep_lds_floats()
{
    return kSweepMapFrags * kWave * 4 + kSweepPairs * (kSweepUnit * (16 * R + 4) + R * kMfmaParts * kWave * 4);
}

// kPf false (reference semantics): rows 49 + j are mu_j, j = 2 .. last slot; seed_a = gx, seed_b
// = gA, [slot][path]. kPf true: R = 4, mu (a scalar, on tenor 0) is row 51; seed_a = gbar
// [date][tenor][path], seed_b = beta [date][path]. map: (T^T)^S in the path kernels' K order;
// ptab[j][64]: column j of sum_{q < S} (T^T)^q (kPf: column 0 only).
template <bool kPf, int R>
__global__ __attribute__((amdgpu_flat_work_group_size(kSweepBlock, kSweepBlock), amdgpu_waves_per_eu(R <= 5 ? 2 : 1, 2)))
void adjoint_mfma_kernel(const SweepGrid g, const u4_t* __restrict__ map, const float* __restrict__ ptab,
                         const float* __restrict__ zs, const float* __restrict__ seed_a,
                         const float* __restrict__ seed_b, float* __restrict__ partials)
{
    constexpr int kPitch = 16 * R + 4, kT = kSweepTiles;
    extern __shared__ float lds[];
    u4_t* lds_map = reinterpret_cast<u4_t*>(lds);
    for (int t = threadIdx.x; t < kSweepMapFrags * kWave; t += kSweepBlock) lds_map[t] = map[t];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int grp = lane / 16, col = lane % 16;
    const int half = __builtin_amdgcn_readfirstlane(wave % 2), pair = __builtin_amdgcn_readfirstlane(wave / 2);
    // the pair's rows [path][row], then their split A fragments [row tile][part][lane]
    float* xt = lds + kSweepMapFrags * kWave * 4 +
                pair * (kSweepUnit * kPitch + R * kMfmaParts * kWave * 4);
    u4_t* xf = reinterpret_cast<u4_t*>(xt + kSweepUnit * kPitch);
    float* mine = xt + (16 * half + col) * kPitch;         // the lane's path

    const int64_t P = g.paths;
    const int t0 = half * kT;
    // byte offsets of the lane's column and paths in a column tile; the very last tile has
    // columns 144 .. 149 and then none (column 144 read instead, replaced after)
    const uint32_t zoff = 4u * ((uint32_t)col * (uint32_t)g.zld + 4u * (uint32_t)grp);
    const uint32_t zlast = half == 1 && col >= 6 ? 16u * (uint32_t)grp : zoff;
    f4_t acc[kT][R];
#pragma unroll
    for (int t = 0; t < kT; ++t)
#pragma unroll
        for (int m = 0; m < R; ++m) acc[t][m] = f4_t{0.f, 0.f, 0.f, 0.f};

    const int64_t first = ((int64_t)blockIdx.x * kSweepPairs + pair) * g.units;
    for (int64_t unit = first; unit < first + g.units; ++unit) {
        // paths [begin, end) of this launch; a pair past the end goes along with zeros (the
        // workgroup's barriers)
        const int64_t base = g.begin + unit * kSweepUnit;
        // (the last unit's reads run into the next row, or past the last into kSweepSlack
        // zeros; the rows of paths past the end are zero, so any finite value will do)
        const float* zrow = zs + (base < g.end ? base - g.begin : 0);
        float za[2][8], zb[2][8];   // tiles 0, 1 (then 4) and 2, 3
        auto load_tile = [&](int b, int t, float (&d)[8]) {
            const float* q = zrow + (int64_t)(b * 3 * kMfmaStride + 16 * (t0 + t)) * g.zld;
            const uint32_t at = t == kT - 1 ? zlast : zoff;
            const f4u_t lo = load_at<f4u_t>(q, at), hi = load_at<f4u_t>(q + 16, at);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                d[i] = lo[i];
                d[4 + i] = hi[i];
            }
        };
        const int64_t path = base + 16 * half + col;
        const bool live = path < g.end;
        const int64_t pc = live ? path : g.begin;
        // x: the rows of lambda; pm: the recursion's mu part (kPf: column 0 of the table times
        // the scalar mus); sa, sx: the next injection
        float x[16], pm[kPf ? 1 : 16], sa = 0.f, sx = 0.f, mus = 0.f;
        // factors, not conditions: no branches around the loads (exact wait counts). Rows 48 .. 50
        // are lane group 0's; the other groups read them too
        const float on = live ? 1.f : 0.f, on48 = grp == 0 ? on : 0.f;
        const uint32_t poff = 4u * (uint32_t)pc, roff = poff + 16u * (uint32_t)grp * (uint32_t)P;
        auto load_rows = [&](int e, float (&d)[16]) {   // kPf: gbar of date e
            const float* q = seed_a + (int64_t)e * kTenors * P;
#pragma unroll
            for (int i = 0; i < 15; ++i)
                d[i] = (i < 12 ? on : on48) * load_at<float>(q + (16 * (i / 4) + i % 4) * P, i < 12 ? roff : poff);
            d[15] = 0.f;
        };
        auto load_seeds = [&](int slot) {
            sa = on * load_at<float>(seed_b + (int64_t)slot * P, poff);
            if constexpr (!kPf) sx = on * load_at<float>(seed_a + (int64_t)slot * P, poff);
        };
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            x[i] = 0.f;
            pm[kPf ? 0 : i] = 0.f;
        }
        if constexpr (kPf) {
            load_rows(g.hi + 1, x);
            x[13] += x[14];   // row 49: x_49 + x_50
        }
        load_seeds(g.hi + 1);
        load_tile(g.hi, 0, za[0]);
        load_tile(g.hi, 1, za[1]);
        load_tile(g.hi, 2, zb[0]);
        load_tile(g.hi, 3, zb[1]);
        __syncthreads();   // the unit before is read (and the map and table are there)
        // rows 48 .. 16 R - 1 start at zero: the mu rows not yet injected, and the padding; by the
        // lane that also writes them
        if (grp == 0) {
#pragma unroll
            for (int q = 0; q < 4 * (R - 3); ++q)
                *reinterpret_cast<f4_t*>(mine + 48 + 4 * q) = f4_t{0.f, 0.f, 0.f, 0.f};
        }

        auto write_rows = [&]() {
#pragma unroll
            for (int m = 0; m < 3; ++m)
                *reinterpret_cast<f4_t*>(mine + 16 * m + 4 * grp) =
                    f4_t{x[4 * m], x[4 * m + 1], x[4 * m + 2], x[4 * m + 3]};
            if (grp == 0) {
#pragma unroll
                for (int r = 0; r < 3; ++r) mine[48 + r] = x[12 + r];
            }
        };
        // the pair's rows in the A layout, split, half of the row tiles by either wave
        auto split_rows = [&]() {
#pragma unroll
            for (int mm = 0; mm < (R + 1) / 2; ++mm) {
                const int m = 2 * mm + half;
                if (R % 2 && m >= R) continue;
                float v[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = xt[(4 * grp + (i < 4 ? i : 12 + i)) * kPitch + 16 * m + col];
                const Split8 s = split8(v);
                xf[(m * kMfmaParts + 0) * kWave + lane] = s.h;
                xf[(m * kMfmaParts + 1) * kWave + lane] = s.m;
                xf[(m * kMfmaParts + 2) * kWave + lane] = s.l;
            }
        };
        // column tiles [t, t + N) += rows x shocks
        auto contract = [&](int t, auto& bz) {
            constexpr int N = sizeof(bz) / sizeof(Split8);
#pragma unroll
            for (int m = 0; m < R; ++m) {
                const u4_t ah = xf[(m * kMfmaParts + 0) * kWave + lane], am = xf[(m * kMfmaParts + 1) * kWave + lane],
                           al = xf[(m * kMfmaParts + 2) * kWave + lane];
#pragma unroll
                for (int n = 0; n < N; ++n) acc[t + n][m] = mfma_bf16(ah, bz[n].h, acc[t + n][m]);
#pragma unroll
                for (int n = 0; n < N; ++n) acc[t + n][m] = mfma_bf16(ah, bz[n].m, acc[t + n][m]);
#pragma unroll
                for (int n = 0; n < N; ++n) acc[t + n][m] = mfma_bf16(am, bz[n].h, acc[t + n][m]);
#pragma unroll
                for (int n = 0; n < N; ++n) acc[t + n][m] = mfma_bf16(ah, bz[n].l, acc[t + n][m]);
#pragma unroll
                for (int n = 0; n < N; ++n) acc[t + n][m] = mfma_bf16(al, bz[n].h, acc[t + n][m]);
#pragma unroll
                for (int n = 0; n < N; ++n) acc[t + n][m] = mfma_bf16(am, bz[n].m, acc[t + n][m]);
            }
        };

        for (int b = g.hi; b >= g.lo; --b) {
            // injection at the end of block b
            if constexpr (kPf) {
                mus += g.dt * sa;
                if (grp == 0) mine[kTenors] = mus;
            } else {
                const int slot = b + 1, at = 4 * (slot / 16) + slot % 4;
                const float v = grp == (slot % 16) / 4 ? sx + sa : 0.f;
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (i == at) x[i] += v;
                if (slot == kTenors - 1) x[13] += v;   // (row 49: x_49 + x_50)
                if (grp == 0) mine[49 + slot] = sa;
                const float* pr = ptab + slot * 64 + 4 * grp;
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const f4_t pv = *reinterpret_cast<const f4_t*>(pr + 16 * m);
#pragma unroll
                    for (int r = 0; r < 4; ++r) pm[4 * m + r] = __builtin_fmaf(pv[r], sa, pm[4 * m + r]);
                }
            }
            write_rows();
            __syncthreads();
            split_rows();
            __syncthreads();
            load_seeds(b);
            // the contraction, two column tiles at a time; a tile's registers take the next
            // block's tile as soon as they are split
            const int bn = b > g.lo ? b - 1 : b;   // (loads without a branch: exact wait counts)
            {
                const Split8 bz[2] = {split8(za[0]), split8(za[1])};
                load_tile(b, 4, za[0]);
                load_tile(bn, 1, za[1]);
                contract(0, bz);
            }
            __builtin_amdgcn_sched_barrier(0);
            {
                const Split8 bz[2] = {split8(zb[0]), split8(zb[1])};
                load_tile(bn, 2, zb[0]);
                load_tile(bn, 3, zb[1]);
                contract(2, bz);
            }
            __builtin_amdgcn_sched_barrier(0);
            float rows[kPf ? 16 : 1];
            {
                // the last wave's last tile holds the constant 1 and padding
                const int n = 16 * (t0 + kT - 1) + col;
                float z[8];
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    z[i] = n < 3 * kMfmaStride ? za[0][i] : (n == 3 * kMfmaStride ? 1.f : 0.f);
                const Split8 bz[1] = {split8(z)};
                load_tile(bn, 0, za[0]);
                if constexpr (kPf) load_rows(b, rows);
                contract(kT - 1, bz);
            }
            __builtin_amdgcn_sched_barrier(0);
            // the recursion: x <- (T^T)^S x + (sum_q (T^T)^q) mu
            uint32_t off = (uint32_t)lane;
            asm volatile("" : "+v"(off));
            f4_t big[4], small[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) big[m] = small[m] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const Split8 v = split8(&x[8 * c]);
                // two row tiles at a time (registers), in turn: no product waits for the one before
#pragma unroll
                for (int m0 = 2 * c; m0 < 4; m0 += 2) {   // rows <= 31 take no tenor >= 32
                    u4_t ah[2], am[2], al[2];
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        const u4_t* a = lds_map + (((m0 + k) * 2 + c) * kMfmaParts) * kWave + off;
                        ah[k] = a[0];
                        am[k] = a[kWave];
                        al[k] = a[2 * kWave];
                    }
#pragma unroll
                    for (int k = 0; k < 2; ++k) big[m0 + k] = mfma_bf16(ah[k], v.h, big[m0 + k]);
#pragma unroll
                    for (int k = 0; k < 2; ++k) small[m0 + k] = mfma_bf16(ah[k], v.m, small[m0 + k]);
#pragma unroll
                    for (int k = 0; k < 2; ++k) small[m0 + k] = mfma_bf16(am[k], v.h, small[m0 + k]);
#pragma unroll
                    for (int k = 0; k < 2; ++k) small[m0 + k] = mfma_bf16(ah[k], v.l, small[m0 + k]);
#pragma unroll
                    for (int k = 0; k < 2; ++k) small[m0 + k] = mfma_bf16(al[k], v.h, small[m0 + k]);
#pragma unroll
                    for (int k = 0; k < 2; ++k) small[m0 + k] = mfma_bf16(am[k], v.m, small[m0 + k]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            f4_t pv[kPf ? 4 : 1];
            if constexpr (kPf) {
                rows[13] += rows[14];
                int at = 4 * grp;
                asm volatile("" : "+v"(at));   // read here each time, not held in registers
#pragma unroll
                for (int m = 0; m < 4; ++m) pv[m] = *reinterpret_cast<const f4_t*>(ptab + at + 16 * m);
            }
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = 4 * m + r;
                    if constexpr (kPf) x[i] = big[m][r] + __builtin_fmaf(pv[m][r], mus, small[m][r]) + rows[i];
                    else x[i] = big[m][r] + (small[m][r] + pm[i]);
                }
        }
        // time 0: column 151 takes the rows themselves (reference: the seeds of slot 1, whose
        // gA is live in all S steps of the frozen block 0, on tenor 1)
        if constexpr (!kPf) x[1] += grp == 0 ? sx + (float)kMfmaStride * sa : 0.f;
        write_rows();
        __syncthreads();
        split_rows();
        __syncthreads();
        if (half == 1) {
            float one[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) one[i] = col == 151 % 16 ? 1.f : 0.f;
            const Split8 bz[1] = {split8(one)};
            contract(kT - 1, bz);
        }
    }

    // the workgroup's sum, in pair order, and its rows of partials [16 R][160]
    __syncthreads();
    constexpr int kHalf = kT * R * 4 * kWave;
    for (int q = 0; q < kSweepPairs; ++q) {
        if (pair == q) {
#pragma unroll
            for (int t = 0; t < kT; ++t)
#pragma unroll
                for (int m = 0; m < R; ++m)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        float* o = lds + half * kHalf + ((t * R + m) * 4 + r) * kWave + lane;
                        *o = q ? *o + acc[t][m][r] : acc[t][m][r];
                    }
        }
        __syncthreads();
    }
    float* out = partials + (int64_t)blockIdx.x * (16 * R * kSweepCols);
    for (int e = threadIdx.x; e < 2 * kHalf; e += kSweepBlock) {
        const int l = e % kWave, r = e / kWave % 4, m = e / (4 * kWave) % R, t = e / (4 * kWave * R);
        out[(16 * m + 4 * (l / 16) + r) * kSweepCols + 16 * t + l % 16] = lds[e];
    }
}

// out[c] = (add ? out[c] : 0) + the FP64 sum of partials[r][c] over the rows r, in a fixed order:
// 16 waves a row each in turn, 8 rows' loads in flight per wave (4096 rows are 160 to 290 MB).
constexpr int kSumWaves = 16;
__global__ __launch_bounds__(kSumWaves * kWave) void sweep_sum_kernel(const float* __restrict__ partials,
                                                                      int64_t rows, int cols, bool add,
                                                                      double* __restrict__ out)
{
    __shared__ double red[kSumWaves][kWave];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int c = blockIdx.x * kWave + lane;   // cols is a multiple of 64
    double s = 0.0;
    constexpr int kAhead = 8;
    int64_t r = wave;
    for (; r + (kAhead - 1) * kSumWaves < rows; r += kAhead * kSumWaves) {
        float x[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) x[i] = partials[(r + i * kSumWaves) * cols + c];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) s += (double)x[i];
    }
    for (; r < rows; r += kSumWaves) s += (double)partials[r * cols + c];
    red[wave][lane] = s;
    __syncthreads();
    if (wave == 0) {
        double t = add ? out[c] : 0.0;
#pragma unroll
        for (int w = 0; w < kSumWaves; ++w) t += red[w][lane];
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

// row tiles: lambda, then mu_j at row 49 + j up to the last slot (the portfolio's at row 51)
int sweep_row_tiles(bool pf, int ndates) { return pf ? 4 : (49 + ndates) / 16 + 1; }

// One unit until the chip holds two waves per SIMD of 256 CUs, then two. Not more: an FP32
// accumulator is truncated, not rounded, at every product, so that sums of one sign drift
// linearly with its chain. Deal Greeks at 1048576 paths x 10y against 64 bits with 32 units:
// d_drift 6.8e-6, d_vol 1.2e-6; with two 1.8e-7 and 2.1e-7 (the VALU sweep 6.3e-7 and 8.6e-7), in
// 4.15 ms against 4.28, and 7.4 against 29 with regenerated shocks, whose bounded portions held
// 14 workgroups of 32 units at a time.
int sweep_units(int64_t paths) { return paths <= 1024 * kSweepUnit ? 1 : 2; }

int64_t sweep_group(int64_t paths) { return (int64_t)kSweepPairs * sweep_units(paths) * kSweepUnit; }

template <bool kPf, int R>
static hipError_t sweep_launch(const SweepGrid& g, const u4_t* map, const float* ptab, const float* zs,
                               const float* a, const float* b, float* partials, hipStream_t st)
{
    const size_t lds = sizeof(float) * std::max<size_t>(sweep_lds_floats<R>(),
                                                        (size_t)2 * kSweepTiles * R * 4 * kWave);
    const void* fn = (const void*)adjoint_mfma_kernel<kPf, R>;
    const hipError_t err = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) return err;
    const int64_t per = (int64_t)kSweepPairs * g.units * kSweepUnit;
    const dim3 grid((unsigned)((g.end - g.begin + per - 1) / per));
    adjoint_mfma_kernel<kPf, R><<<grid, kSweepBlock, lds, st>>>(g, map, ptab, zs, a, b, partials);
    return hipGetLastError();
}

hipError_t launch_adjoint_mfma(const SweepGrid& g, bool pf, const uint16_t* map, const float* ptab,
                               const float* zs, const float* seed_a, const float* seed_b, float* partials,
                               hipStream_t st)
{
    if (g.begin < 0 || g.end <= g.begin || g.end > g.paths || g.hi < g.lo || g.paths > kSweepMaxPaths)
        return hipErrorInvalidValue;
    const u4_t* m = reinterpret_cast<const u4_t*>(map);
    if (pf) return sweep_launch<true, 4>(g, m, ptab, zs, seed_a, seed_b, partials, st);
    switch (sweep_row_tiles(false, g.hi + 1)) {
    case 4: return sweep_launch<false, 4>(g, m, ptab, zs, seed_a, seed_b, partials, st);
    case 5: return sweep_launch<false, 5>(g, m, ptab, zs, seed_a, seed_b, partials, st);
    case 6: return sweep_launch<false, 6>(g, m, ptab, zs, seed_a, seed_b, partials, st);
    default: return sweep_launch<false, 7>(g, m, ptab, zs, seed_a, seed_b, partials, st);
    }
}

hipError_t launch_sweep_sum(const float* partials, int64_t rows, int cols, bool add, double* out,
                            hipStream_t st)
{
    sweep_sum_kernel<<<(unsigned)(cols / kWave), kSumWaves * kWave, 0, st>>>(partials, rows, cols, add, out);
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
