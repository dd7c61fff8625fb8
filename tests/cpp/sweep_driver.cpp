// The portions and segments of the matrix-core reverse sweep (hjm_sweep.h) over the stand-in
// runtime of fake_hip/: the launches are recorded instead of made. One check per argument name.
#include <stdio.h>
#include <string.h>

#include <vector>

#include "hjm_sweep.h"

using namespace hjm_host;

static int failures = 0;
#define CHECK(x)                                                  \
    do {                                                          \
        if (!(x)) {                                               \
            printf("%s:%d: %s\n", __func__, __LINE__, #x);        \
            ++failures;                                           \
        }                                                         \
    } while (0)

struct Launch {
    SweepGrid g;
    const float* zs;
    float* partials;
};
static std::vector<Launch> launches;
static std::vector<int64_t> summed;   // rows
static bool first_sum_adds;

namespace hjm {
int sweep_units(int64_t paths) { return paths <= 32768 ? 1 : 2; }
int64_t sweep_group(int64_t paths) { return 64 * sweep_units(paths); }
int sweep_row_tiles(bool, int) { return 4; }
hipError_t launch_sweep_map(double, bool, uint16_t*, float*, hipStream_t) { return hipSuccess; }
hipError_t launch_sweep_shocks(uint64_t, int64_t, const SweepGrid&, float*, hipStream_t) { return hipSuccess; }
hipError_t launch_adjoint_mfma(const SweepGrid& g, bool, const uint16_t*, const float*, const float* zs,
                               const float*, const float*, float* partials, hipStream_t)
{
    launches.push_back({g, zs, partials});
    return hipSuccess;
}
hipError_t launch_sweep_sum(const float*, int64_t rows, int, bool add, double*, hipStream_t)
{
    if (summed.empty()) first_sum_adds = add;
    else CHECK(add);
    summed.push_back(rows);
    return hipSuccess;
}
}  // namespace hjm

// Every path once, in whole workgroups, each partial within the segment's buffer and summed once;
// stored shocks are read from the portion's first column, within the array and its slack.
static void portions_cover_every_path_once()
{
    const int nsteps = 250;
    for (int64_t paths : {int64_t(1), int64_t(63), int64_t(65), int64_t(32768), int64_t(32769), int64_t(600001),
                          int64_t(1048576), int64_t(1100003)}) {
        for (bool stored : {true, false}) {
            launches.clear();
            summed.clear();
            SweepGrid g{};
            g.hi = 4;
            g.lo = 0;
            g.paths = paths;
            SweepBuffers b;
            CHECK(b.take(g, true, 0.02, nsteps, stored, nullptr) == HJM_OK);
            const int64_t group = sweep_group(paths), groups = (paths + group - 1) / group;
            float* zs = nullptr;
            if (stored) CHECK(dev_alloc(&zs, (size_t)paths * nsteps * 3 + kSweepSlack) == HJM_OK);
            CHECK(b.run(g, true, zs, nsteps, 1, 0, nullptr, nullptr, nullptr, nullptr) == HJM_OK);
            int64_t at = 0;
            for (const Launch& l : launches) {
                CHECK(l.g.begin == at && l.g.end > at && l.g.end <= paths && l.g.begin % group == 0);
                const int64_t n = (l.g.end - l.g.begin + group - 1) / group;
                const int64_t row = (l.partials - b.partials) / (b.rows * 160);
                CHECK(row == at / group % kSweepSegment && row + n <= std::min(groups, kSweepSegment));
                CHECK(l.g.zld == (stored ? paths : l.g.end - l.g.begin));
                CHECK(l.zs == (stored ? zs + at : b.chunk));
                if (!stored) CHECK((size_t)(l.g.end - l.g.begin) * nsteps * 12 <= kSweepChunkBytes);
                at = l.g.end;
            }
            int64_t rows = 0;
            for (int64_t r : summed) rows += r;
            CHECK(at == paths && rows == groups && !first_sum_adds);
            dev_free(true, zs);
            b.free(true);
        }
    }
}

// Without memory for the regenerated shocks the sweep's other buffers are given back.
static void memory_that_does_not_suffice()
{
    SweepGrid g{};
    g.hi = 4;
    g.paths = 32768;
    SweepBuffers b;
    fake::budget = (size_t)21 << 20;   // the partials' 20 MB and little more
    CHECK(b.take(g, true, 0.02, 3000, false, nullptr) == HJM_ERR_ALLOC);
    char* p = nullptr;
    CHECK(dev_alloc(&p, (size_t)20 << 20) == HJM_OK);
}

int main(int argc, char** argv)
{
    const struct {
        const char* name;
        void (*run)();
    } checks[] = {{"portions_cover_every_path_once", portions_cover_every_path_once},
                  {"memory_that_does_not_suffice", memory_that_does_not_suffice}};
    for (const auto& c : checks)
        if (argc == 2 && !strcmp(argv[1], c.name)) {
            c.run();
            return failures ? 1 : 0;
        }
    printf("no such check\n");
    return 2;
}
