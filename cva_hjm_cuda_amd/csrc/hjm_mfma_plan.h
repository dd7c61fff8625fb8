// hjm_mfma_plan.h -- host construction of the 50-step block maps for the matrix-core
// path kernels (FP32 as bf16 parts, FP64 as they are) and of the valuation's fragments.
//
// One block of S = 50 Euler steps is affine in the curve f, the scaled shocks
// s_{t,k} = sqrt(dt) phi_k(t) and 1:
//   f_out  = T^S f_in + sum_t T^{S-1-t} (m dt + V s_t)
// with T = I + (dt/dtau) Dfwd (backward difference on the last tenor). Two maps:
//   reference semantics (102 rows, 7 M-tiles of 16): rows 51..101 hold the block's
//     discount-integral increments dA = sum_{r=1}^{S} f_r
//       = (sum_{r=1}^{S} T^r) f_in + sum_t (sum_{q=0}^{S-1-t} T^q)(m dt + V s_t);
//   portfolio semantics (52 rows, 4 M-tiles): row 51 holds the short rate's left-point sum
//       sum_{r=0}^{S-1} f_r[0] = (sum_{r=0}^{S-1} T^r f_in)[0]
//                               + sum_t (sum_{q=0}^{S-2-t} T^q (m dt + V s_t))[0].
// The kernel computes W x [f_in; phi; 1] with v_mfma_f32_16x16x32_{bf16,f16}. K has 224 entries
// in 7 chunks of 32; in chunk c lane group g = lane / 16 supplies slots i = 0..7, the
// K index being 32 c + 8 g + i:
//   chunks 0, 1: curve row R = 16 (2c + i/4) + 4 g + i%4 (zero column where R > 50): the
//     previous block's accumulator registers 8c + i of the lane, unchanged;
//   chunks 2..6 (s = c - 2): value v = 8 s + i of lane group g, which generates the steps
//     t = 4 q + g, q = 0..12: v = 3 q + k is factor k of step t (t < 50); at t = 50
//     (g = 2, q = 12) factor 0 is the constant 1 carrying the drift; other slots are zero.
// The curve columns of W (FP64) are split into three bf16 parts W = Wh + Wm + Wl (round to
// nearest); the kernel splits the curve exactly (truncation: xh + xm + xl = x) and accumulates
// the six products Wh xh + Wh xm + Wm xh + Wh xl + Wl xh + Wm xm in FP32, which leaves an
// error of the order of FP32 rounding. The shock columns take two fp16 parts on either side
// (11 bits each, to nearest) and three products Wh xh + Wh xl + Wl xh, half as many: a shock's
// contribution loses at most 2^-21 of itself, 5e-8 rms with either sign. A block's 150 add up to
// a fraction of an ordinary curve, and this stays under the curve's own rounding; where they outweigh
// it, a block's forwards are 1.1e-7 (rms, relative) from FP64 instead of 0.6e-7 with three bf16
// parts throughout, ten years of blocks 1.25e-7 instead of 1.55e-7.
// Fragment (m, c, part)[lane][i] = part of W[16 m + lane % 16][32 c + 8 (lane / 16) + i].
#pragma once
#include <math.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "hjm_common.h"

namespace hjm {

constexpr int kMfmaStride = 50;   // steps per block handled by the matrix-core kernels
constexpr int kMfmaMTiles = 7;    // reference map: 102 output rows -> 7 x 16
constexpr int kMfmaPfMTiles = 4;  // portfolio map: 52 output rows -> 4 x 16
constexpr int kMfmaQuads = 13;    // steps 4 q + g, q = 0..12, per lane group
constexpr int kMfmaChunks = 7;    // 2 curve chunks + 5 shock chunks of 32 K entries
constexpr int kMfmaK = 32 * kMfmaChunks;  // 224
constexpr int kMfmaParts = 3;      // bf16 parts of W's curve columns (and of -gamma)
constexpr int kMfmaShockParts = 2; // fp16 parts of W's shock columns
// fragments (64 lanes x 8 16-bit elements) of one M-tile: curve chunks 0, 1 in three bf16
// parts, shock chunks 2..6 in two fp16 parts
constexpr int kMfmaTileFrags = 2 * kMfmaParts + (kMfmaChunks - 2) * kMfmaShockParts;  // 16
__host__ __device__ constexpr int mfma_frag(int m, int c, int part)
{
    return m * kMfmaTileFrags +
           (c < 2 ? c * kMfmaParts : 2 * kMfmaParts + (c - 2) * kMfmaShockParts) + part;
}
// 16-bit elements of one kernel's fragments
constexpr int kMfmaPfFragElems = kMfmaPfMTiles * kMfmaTileFrags * kWave * 8;
// LDS bytes of the first mt M-tiles' fragments (the reference kernel stages only its live
// tiles)
constexpr int ref_mfma_lds_bytes(int mt) { return mt * kMfmaTileFrags * kWave * 8 * 2; }

enum class MfmaMap { kReference, kPortfolio };

// Live M-tiles of the reference map for a run of ndates dates: the curve's four and the
// integral rows 51 + j up to j = ndates (the last slot recorded).
inline int ref_mfma_tiles(int ndates)
{
    const int last = kTenors + (ndates > 1 ? ndates : 1);
    return last / 16 + 1 < 4 ? 4 : last / 16 + 1;
}

// Structural zeros of the maps' curve columns. T couples tenor j only to j + 1 (and 50 to
// 49), so T^n and the integral rows' sums of powers vanish in columns R < min(j, 49) of
// row j; integral row 51 + j follows tenor j; the portfolio's row 51 (the short rate's
// sum) spans every tenor. The kernels skip a product whose curve inputs all lie below the
// first input of every row of its M-tile.
__host__ __device__ constexpr int map_row_first_input(int row, bool pf)
{
    return row < kTenors ? (row < 49 ? row : 49) : pf ? 0 : (row - kTenors < 49 ? row - kTenors : 49);
}
__host__ __device__ constexpr int tile_first_input(int m, bool pf)
{
    const int rows = pf ? kTenors + 1 : 2 * kTenors;
    int lo = kTenors;
    for (int r = 16 * m; r < 16 * m + 16 && r < rows; ++r)
        lo = map_row_first_input(r, pf) < lo ? map_row_first_input(r, pf) : lo;
    return lo;
}
// FP32 kernels: curve chunk c (rows 32 c .. 32 c + 31) of M-tile m is all zero
__host__ __device__ constexpr bool mfma_chunk_zero(int m, int c, bool pf)
{
    return c < 2 && 32 * c + 31 < tile_first_input(m, pf);
}

// What K index k of the block map multiplies: a curve row, a shock (step, factor), the
// constant 1, or nothing.
struct MfmaColumn {
    enum Kind { kZero, kCurve, kShock, kConst } kind;
    int row;     // kCurve
    int step;    // kShock
    int factor;  // kShock
};

inline MfmaColumn mfma_column(int k)
{
    const int c = k / 32, g = (k % 32) / 8, i = k % 8;
    if (c < 2) {
        const int R = 16 * (2 * c + i / 4) + 4 * g + i % 4;
        if (R < kTenors) return {MfmaColumn::kCurve, R, 0, 0};
        return {MfmaColumn::kZero, 0, 0, 0};
    }
    const int v = 8 * (c - 2) + i;
    if (v >= 3 * kMfmaQuads) return {MfmaColumn::kZero, 0, 0, 0};
    const int q = v / 3, f = v % 3, t = 4 * q + g;
    if (t < kMfmaStride) return {MfmaColumn::kShock, 0, t, f};
    if (t == kMfmaStride && f == 0) return {MfmaColumn::kConst, 0, 0, 0};
    return {MfmaColumn::kZero, 0, 0, 0};
}

// Dense FP64 block map [rows][224]: rows = 102 (reference) or 52 (portfolio).
inline std::vector<double> mfma_block_map_dense(const double* drift, const double* vols, double dt,
                                                double dtau, MfmaMap map)
{
    const bool pf = map == MfmaMap::kPortfolio;
    const int n = kTenors, S = kMfmaStride;
    const int rows = pf ? n + 1 : 2 * n;
    const double c = dt / dtau, sq = sqrt(dt);
    // y = T x for one column of values `step` apart: T has two entries a row
    auto apply = [n, c](const double* x, double* y, int step) {
        for (int j = 0; j < n - 1; ++j)
            for (int m = 0; m < step; ++m)
                y[j * step + m] = (1.0 - c) * x[j * step + m] + c * x[(j + 1) * step + m];
        for (int m = 0; m < step; ++m)
            y[(n - 1) * step + m] = -c * x[(n - 2) * step + m] + (1.0 + c) * x[(n - 1) * step + m];
    };
    // T^S, sum_{q=1}^{S} T^q and row 0 of sum_{q=0}^{S-1} T^q
    std::vector<double> Tp((size_t)n * n, 0.0), next((size_t)n * n), Sum((size_t)n * n, 0.0);
    std::vector<double> first(n, 0.0);
    for (int j = 0; j < n; ++j) Tp[(size_t)j * n + j] = 1.0;
    for (int s = 1; s <= S; ++s) {
        for (int m = 0; m < n; ++m) first[m] += Tp[m];
        apply(Tp.data(), next.data(), n);
        Tp.swap(next);
        for (size_t i = 0; i < Sum.size(); ++i) Sum[i] += Tp[i];
    }
    std::vector<double> W((size_t)rows * kMfmaK, 0.0);
    int shock_k[kMfmaStride][3] = {}, const_k = 0;
    for (int k = 0; k < kMfmaK; ++k) {
        const MfmaColumn col = mfma_column(k);
        if (col.kind == MfmaColumn::kShock) shock_k[col.step][col.factor] = k;
        if (col.kind == MfmaColumn::kConst) const_k = k;
        if (col.kind != MfmaColumn::kCurve) continue;
        for (int j = 0; j < n; ++j) W[(size_t)j * kMfmaK + k] = Tp[(size_t)j * n + col.row];
        if (pf) W[(size_t)n * kMfmaK + k] = first[col.row];
        else
            for (int j = 0; j < n; ++j) W[(size_t)(n + j) * kMfmaK + k] = Sum[(size_t)j * n + col.row];
    }
    // A vector v added at step t reaches the block's end as T^{S-1-t} v and its integral as
    // sum_{q <= S-1-t} T^q v (the left-point sum: q <= S-2-t, tenor 0): walked from the last
    // step back, u = T^q v and its running sum.
    auto walk = [&](const double* v, auto put) {
        std::vector<double> u(v, v + n), acc(n, 0.0), t(n);
        for (int q = 0; q < S; ++q) {
            const double left = acc[0];
            for (int j = 0; j < n; ++j) acc[j] += u[j];
            put(S - 1 - q, u.data(), acc.data(), left);
            apply(u.data(), t.data(), 1);
            u.swap(t);
        }
    };
    std::vector<double> v(n);
    for (int f = 0; f < 3; ++f) {
        for (int i = 0; i < n; ++i) v[i] = sq * vols[f * n + i];
        walk(v.data(), [&](int t, const double* u, const double* acc, double left) {
            const int k = shock_k[t][f];
            for (int j = 0; j < n; ++j) W[(size_t)j * kMfmaK + k] = u[j];
            if (pf) W[(size_t)n * kMfmaK + k] = left;
            else
                for (int j = 0; j < n; ++j) W[(size_t)(n + j) * kMfmaK + k] = acc[j];
        });
    }
    for (int i = 0; i < n; ++i) v[i] = drift[i] * dt;
    walk(v.data(), [&](int, const double* u, const double* acc, double left) {
        for (int j = 0; j < n; ++j) W[(size_t)j * kMfmaK + const_k] += u[j];
        if (pf) W[(size_t)n * kMfmaK + const_k] += left;
        else
            for (int j = 0; j < n; ++j) W[(size_t)(n + j) * kMfmaK + const_k] += acc[j];
    });
    return W;
}

// bf16 bits of x rounded to nearest (ties to even); x finite.
__host__ __device__ inline uint16_t bf16_rne(double x)
{
    const float f = (float)x;
    uint32_t u;
    memcpy(&u, &f, 4);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__host__ __device__ inline double bf16_value(uint16_t b)
{
    const uint32_t u = (uint32_t)b << 16;
    float f;
    memcpy(&f, &u, 4);
    return (double)f;
}

// fp16 bits of x rounded to nearest (ties to even); |x| < 65504
__host__ __device__ inline uint16_t fp16_rne(float x)
{
    uint32_t u;
    memcpy(&u, &x, 4);
    const uint32_t sign = (u >> 16) & 0x8000u;
    u &= 0x7fffffffu;
    if (u < 0x38800000u) {   // below 2^-14: subnormal, quantum 2^-24
        const float m = nearbyintf(ldexpf(x < 0.f ? -x : x, 24));
        return (uint16_t)(sign | (uint32_t)m);
    }
    u += 0xfffu + ((u >> 13) & 1u);
    return (uint16_t)(sign | ((u >> 13) - (112u << 10)));
}

__host__ __device__ inline double fp16_value(uint16_t h)
{
    const uint32_t e = (h >> 10) & 31u, m = h & 1023u;
    if (!e) return ((h & 0x8000u) ? -0x1p-24 : 0x1p-24) * m;
    const uint32_t u = ((uint32_t)(h & 0x8000u) << 16) | ((e + 112u) << 23) | (m << 13);
    float f;
    memcpy(&f, &u, 4);
    return (double)f;
}

// The block map's fragments (block_map_kernel) in the path kernel's A-operand order: row 16 m +
// lane % 16 and column 32 c + 8 (lane / 16) + i of fragment mfma_frag(m, c, part); the curve
// columns as three bf16 parts, the shock columns (and the drift constant's) times 2^k as two
// fp16 parts rounded to nearest.
struct BlockMapParams {
    double c, up;            // dt / dtau, 2^k
    double vec[4][kTenors];  // loadings times sqrt(dt), drift times dt
    int mtiles;              // the M-tiles built (the reference kernel's live ones)
    int scale;               // k
};

// k is the power of two that brings the largest shock entry (the drift's and the integral rows'
// among them) to [2^12, 2^13); without it the entries, 1e-4 .. 1e-2, would leave their low parts
// to fp16's subnormals. An entry down to 2^-14 of the largest keeps 22 bits in its two parts, a
// smaller one an absolute 2^-37 of the largest. The kernels hold the curve and the integrals times
// 2^k too, so both kinds of products share the final sum; k is bounded by the curve's size
// (max |spot| 2^k < 2^40, so that 25 years of integrals stay far from FP32's end; shocks that
// this leaves below 2^12 are under 2^-27 of the curve), and 0 without shocks.
inline BlockMapParams block_map_params(const double* spot, const double* drift, const double* vols, double dt,
                                       double dtau, int mtiles, MfmaMap map = MfmaMap::kReference)
{
    const bool pf = map == MfmaMap::kPortfolio;
    constexpr int n = kTenors;
    BlockMapParams p{};
    p.c = dt / dtau;
    p.mtiles = mtiles;
    const double sq = sqrt(dt), c = p.c;
    for (int j = 0; j < n; ++j) {
        for (int f = 0; f < 3; ++f) p.vec[f][j] = sq * vols[f * n + j];
        p.vec[3][j] = drift[j] * dt;
    }
    // the largest entry of the shock columns and the drift's (mfma_block_map_dense's walks)
    double tops[n] = {0.0}, left_top = 0.0, curve = 0.0;
    auto raise = [&tops](const double* x) {
        for (int j = 0; j < n; ++j) tops[j] = fabs(x[j]) > tops[j] ? fabs(x[j]) : tops[j];
    };
    for (int f = 0; f < 4; ++f) {
        double u[n], t[n], acc[n] = {0.0}, cu[n] = {0.0}, ca[n] = {0.0}, cleft = 0.0;
        memcpy(u, p.vec[f], sizeof u);
        for (int q = 0; q < kMfmaStride; ++q) {
            const double left = acc[0];
            for (int j = 0; j < n; ++j) acc[j] += u[j];
            if (f < 3) {
                raise(u);
                if (!pf) raise(acc);
                left_top = fabs(left) > left_top ? fabs(left) : left_top;
            } else {
                for (int j = 0; j < n; ++j) {
                    cu[j] += u[j];
                    ca[j] += acc[j];
                }
                cleft += left;
            }
            for (int j = 0; j < n - 1; ++j) t[j] = (1.0 - c) * u[j] + c * u[j + 1];
            t[n - 1] = -c * u[n - 2] + (1.0 + c) * u[n - 1];
            memcpy(u, t, sizeof u);
        }
        if (f == 3) {
            raise(cu);
            if (!pf) raise(ca);
            left_top = fabs(cleft) > left_top ? fabs(cleft) : left_top;
        }
    }
    double top = pf ? left_top : 0.0;
    for (int j = 0; j < n; ++j) {
        top = std::max(top, tops[j]);
        curve = std::max(curve, fabs(spot[j]));
    }
    if (top > 0.0) {
        p.scale = std::max(-120, std::min(120, 12 - ilogb(top)));
        if (curve > 0.0) p.scale = std::min(p.scale, 39 - ilogb(curve));
    }
    p.up = ldexp(1.0, p.scale);
    return p;
}

// Curve columns: an entry below 2^-16 of its row's largest takes only the second and third part
// (16 bits, 2^-32 of the largest). As a leading part its product would lie so far below the
// others that the matrix cores drop it: with dt = 0.01f instead of 0.01 the last tenors' map has
// entries of 2e-8 beside 1, which carry what the others lack to a row sum of 1, and without them
// the last forwards drift, quadratically in time (mean error of EE over 10 curves against FP64:
// 20y 1.8e-6, 25y 4.3e-6; with them 3.3e-7 and 3.5e-7). Lines from 2^-12 to 2^-20 measure the
// same; at 2^-8 the products among the small ones are large enough that their truncation
// shows (10y 3.3e-7 -> 4.5e-7). With dt / dtau = 1 / 50 the largest entries are 0.37 to 2 in
// the curve's rows and 31 in the sums'.
constexpr double kMinorCurve = 0x1p-17, kMinorSum = 0x1p-11;

inline size_t block_map_elems(int mtiles) { return (size_t)mtiles * kMfmaTileFrags * kWave * 8; }

// The FP64 block map for v_mfma_f64_16x16x4f64 (ref_paths_mfma64_kernel). One instruction
// takes K = 4 entries, one per lane group g = lane / 16, from one register of every lane;
// its accumulator holds row 4 i + g of the 16-row tile in register i of lane group g (not
// 4 g + i as in the FP32 16x16 forms). The kernel issues kMfma64K = 52 instructions per
// M-tile and block:
//   j = 0..12 (curve): register i = j % 4 of the previous block's accumulator tile j / 4,
//     i.e. curve row R = 16 (j / 4) + 4 i + g (zero column where R > 50; tile 3 holds
//     rows 48..50 in register 0 only, hence 13 and not 16);
//   j = 13..51 (shocks): value v = j - 13 of lane group g, factor v % 3 of step
//     4 (v / 3) + g -- the FP32 kernel's shocks, in its order; at step 50 factor 0 is the
//     constant 1 carrying the drift, other entries past step 49 are zero.
// Fragment [m][j][lane] = W[16 m + lane % 16][column (j, lane / 16)], FP64; the reference
// map (ref_paths_mfma64_kernel, up to 7 M-tiles) or the portfolio map (pf_paths_mfma64_kernel,
// 4 M-tiles; the short rate's sum, row 51, is register 0 of lane group 3 of tile 3).
constexpr int kMfma64Curve = 13;
constexpr int kMfma64K = kMfma64Curve + 3 * kMfmaQuads;  // 52
constexpr int kMfma64TileBytes = kMfma64K * kWave * 8;   // 26624
constexpr int kMfma64LdsTiles = 5;  // M-tiles staged in LDS (133 KB); later tiles from HBM
// curve instruction j < 13 of M-tile m is all zero (its rows 16 (j / 4) + 4 (j % 4) + g lie
// below the tile's first input; tiles 0..3 agree for both maps)
__host__ __device__ constexpr bool mfma64_column_zero(int m, int j)
{
    return j < kMfma64Curve && 16 * (j / 4) + 4 * (j % 4) + 3 < tile_first_input(m, false);
}

inline MfmaColumn mfma64_column(int j, int g)
{
    if (j < kMfma64Curve) {
        const int R = 16 * (j / 4) + 4 * (j % 4) + g;
        if (R < kTenors) return {MfmaColumn::kCurve, R, 0, 0};
        return {MfmaColumn::kZero, 0, 0, 0};
    }
    const int v = j - kMfma64Curve, q = v / 3, f = v % 3, t = 4 * q + g;
    if (t < kMfmaStride) return {MfmaColumn::kShock, 0, t, f};
    if (t == kMfmaStride && f == 0) return {MfmaColumn::kConst, 0, 0, 0};
    return {MfmaColumn::kZero, 0, 0, 0};
}

inline void build_mfma64_block_map(const double* drift, const double* vols, double dt, double dtau,
                                   int mtiles, std::vector<double>& frag,
                                   MfmaMap map = MfmaMap::kReference)
{
    const int rows = map == MfmaMap::kPortfolio ? kTenors + 1 : 2 * kTenors;
    const std::vector<double> W = mfma_block_map_dense(drift, vols, dt, dtau, map);
    // the dense map's column of each curve row, shock (step, factor) and the constant
    int curve_k[kTenors] = {}, shock_k[kMfmaStride][3] = {}, const_k = -1;
    for (int k = 0; k < kMfmaK; ++k) {
        const MfmaColumn c = mfma_column(k);
        if (c.kind == MfmaColumn::kCurve) curve_k[c.row] = k;
        else if (c.kind == MfmaColumn::kShock) shock_k[c.step][c.factor] = k;
        else if (c.kind == MfmaColumn::kConst) const_k = k;
    }
    frag.assign((size_t)mtiles * kMfma64K * kWave, 0.0);
    for (int m = 0; m < mtiles; ++m)
        for (int j = 0; j < kMfma64K; ++j)
            for (int l = 0; l < kWave; ++l) {
                const int row = 16 * m + l % 16;
                const MfmaColumn c = mfma64_column(j, l / 16);
                int k = -1;
                if (c.kind == MfmaColumn::kCurve) k = curve_k[c.row];
                else if (c.kind == MfmaColumn::kShock) k = shock_k[c.step][c.factor];
                else if (c.kind == MfmaColumn::kConst) k = const_k;
                if (row < rows && k >= 0)
                    frag[((size_t)m * kMfma64K + j) * kWave + l] = W[(size_t)row * kMfmaK + k];
            }
}

// Matrix-core valuation of netting sets (pf_value_mfma_kernel): per date, M-tiles of 16
// sets x 2 chunks of 32 periods x 3 bf16 parts of -gamma, in the A-operand order
// [date][m][chunk][part][lane][i] = part of -gamma[date][16 m + lane % 16][32 chunk +
// 8 (lane / 16) + i] (0 past the last set or period); apad[date][16 m + j] = a of set
// 16 m + j (0 past the last set); tilek[date][m] = the largest kmax of the tile's sets.
constexpr int kValueFragsPerTile = 2 * kMfmaParts;  // u4 fragments per lane and M-tile

inline int value_mtiles(int nsets) { return (nsets + 15) / 16; }
constexpr int kMaxPfMTiles = (HJM_MAX_SETS + 15) / 16;

// The portfolio adjoint's second product dP = (-Gamma)^T u on the matrix cores
// (pf_adjoint_seed_mfma_kernel): per date, 4 period tiles x ceil(mtiles / 2) K chunks of 32
// sets x 3 bf16 parts, [date][pm][c][part][lane][i] = part of -gamma[date][set][16 pm +
// lane % 16] with set = 16 (2c + i/4) + 4 (lane/16) + i%4, the order in which the first
// product's accumulators hold u (0 past the last set or period). Built on the device
// (hjm_book_kernels.hip), as are the valuation's.

// Tables of the matrix-core reverse sweep (hjm_adjoint_mfma.hip): the 64 x 64 map (T^T)^S as
// [m][c][part][lane][8] bf16 parts of row 16 m + lane % 16 and the curve column of K slot (c,
// lane / 16, i); and ptab[j][64], column j of sum_{q < S} (T^T)^q (portfolio: j = 0 only).
constexpr size_t kSweepMapElems = (size_t)8 * kMfmaParts * kWave * 8;
inline size_t sweep_table_elems(bool pf) { return (size_t)(pf ? 1 : kTenors) * 64; }

}  // namespace hjm
