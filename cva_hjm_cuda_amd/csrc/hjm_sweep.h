// hjm_sweep.h -- buffers and launches of the matrix-core reverse sweep (host side, shared by
// the reference and portfolio Greeks).
#pragma once
#include "hjm_host.h"
#include "hjm_kernels.h"
#include "hjm_mfma_plan.h"

namespace hjm_host {

// Shocks regenerated for the sweep pass through a buffer of at most this many bytes, a whole
// number of workgroups' paths at a time (the sums do not depend on it: every workgroup writes
// its own partial).
constexpr size_t kSweepChunkBytes = (size_t)1 << 30;
// Partials of at most this many workgroups (40 to 72 KB each) are held at a time; each such
// segment is summed into the FP64 result before the next.
constexpr int64_t kSweepSegment = 4096;

struct SweepBuffers {
    uint16_t* map = nullptr;
    float* ptab = nullptr;
    float* partials = nullptr;
    double* out = nullptr;
    float* chunk = nullptr;
    int64_t chunk_paths = 0;
    int rows = 0;             // 16 x row tiles

    // Allocates for g.paths paths and builds the maps; stored: the forward keeps the shocks.
    // What could be had of the memory is given back if the rest cannot (the VALU sweep's
    // buffers are allocated then).
    int take(SweepGrid& g, bool pf, double c, int nsteps, bool stored, hipStream_t st)
    {
        const int rc = allocate(g, pf, nsteps, stored);
        if (rc != HJM_OK) {
            free(true);
            return rc;
        }
        HJM_HIP(launch_sweep_map(c, pf, map, ptab, st), HJM_ERR_LAUNCH);
        return HJM_OK;
    }

    int allocate(SweepGrid& g, bool pf, int nsteps, bool stored)
    {
        if (g.paths > kSweepMaxPaths) return HJM_ERR_UNSUPPORTED;
        g.units = sweep_units(g.paths);
        const int64_t group = sweep_group(g.paths), groups = (g.paths + group - 1) / group;
        rows = 16 * sweep_row_tiles(pf, g.hi + 1);
        HJM_TRY(dev_alloc(&map, kSweepMapElems));
        HJM_TRY(dev_alloc(&ptab, sweep_table_elems(pf)));
        HJM_TRY(dev_alloc(&partials, (size_t)std::min(groups, kSweepSegment) * rows * 160));
        HJM_TRY(dev_alloc(&out, (size_t)rows * 160));
        if (!stored) {
            const size_t per = (size_t)group * nsteps * 3 * sizeof(float);
            int64_t n = std::min<int64_t>(std::min(groups, kSweepSegment),
                                          std::max<int64_t>(1, (int64_t)(kSweepChunkBytes / per)));
            while (n > 1 && dev_alloc(&chunk, (size_t)n * per / sizeof(float) + kSweepSlack) != HJM_OK) n /= 2;
            if (!chunk) HJM_TRY(dev_alloc(&chunk, (size_t)n * per / sizeof(float) + kSweepSlack));
            chunk_paths = n * group;
        }
        return HJM_OK;
    }

    // zs[n]: a buffer of n shocks with its slack cleared.
    static int clear_slack(float* zs, size_t n, hipStream_t st)
    {
        HJM_HIP(hipMemsetAsync(zs + n, 0, kSweepSlack * sizeof(float), st), HJM_ERR_DEVICE);
        return HJM_OK;
    }

    // The sweep and its sums, copied to the (pinned) host array sums[rows * 160].
    int run(SweepGrid g, bool pf, float* zs, int nsteps, uint64_t seed, int64_t path0, const float* seed_a,
            const float* seed_b, double* sums, hipStream_t st)
    {
        const int64_t group = sweep_group(g.paths), groups = (g.paths + group - 1) / group;
        const int cols = rows * 160;
        const int64_t segment = kSweepSegment * group, step = zs ? segment : chunk_paths;
        if (zs) HJM_TRY(clear_slack(zs, (size_t)g.paths * nsteps * 3, st));
        for (int64_t first = 0; first < groups; first += kSweepSegment) {
            const int64_t end = std::min(g.paths, first * group + segment);
            for (int64_t p = first * group; p < end; p += step) {
                g.begin = p;
                g.end = std::min(end, p + step);
                g.zld = zs ? g.paths : g.end - g.begin;
                if (!zs) {
                    HJM_TRY(clear_slack(chunk, (size_t)g.zld * nsteps * 3, st));
                    HJM_HIP(launch_sweep_shocks(seed, path0, g, chunk, st), HJM_ERR_LAUNCH);
                }
                HJM_HIP(launch_adjoint_mfma(g, pf, map, ptab, zs ? zs + p : chunk, seed_a, seed_b,
                                            partials + (size_t)(p / group - first) * cols, st),
                        HJM_ERR_LAUNCH);
            }
            HJM_HIP(launch_sweep_sum(partials, std::min(groups - first, kSweepSegment), cols, first > 0, out, st),
                    HJM_ERR_LAUNCH);
        }
        HJM_HIP(hipMemcpyAsync(sums, out, sizeof(double) * cols, hipMemcpyDeviceToHost, st), HJM_ERR_DEVICE);
        return HJM_OK;
    }

    void free(bool idle) { dev_free(idle, map, ptab, partials, out, chunk); }
};

}  // namespace hjm_host
