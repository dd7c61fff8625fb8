// The cache of device memory and plan contexts (hjm_pool.hip) against the stand-in runtime of
// fake_hip/: one check per argument name; prints what failed and exits with 1.
#include <stdio.h>
#include <string.h>

#include "hjm_host.h"

using namespace hjm_host;

static int failures = 0;
#define CHECK(x)                                                  \
    do {                                                          \
        if (!(x)) {                                               \
            printf("%s:%d: %s\n", __func__, __LINE__, #x);        \
            ++failures;                                           \
        }                                                         \
    } while (0)

// A freed block is handed out again; one that a stream in error used is not, and goes back to
// the device at once, not by way of the cache.
static void blocks_of_a_failed_stream()
{
    ContextHolder h;
    CHECK(h.take(0, 64) == HJM_OK);
    double *a = nullptr, *b = nullptr;
    CHECK(dev_alloc(&a, 1000) == HJM_OK);
    double* const first = a;
    dev_free(h.quiesce(), a);
    CHECK(a == nullptr && dev_alloc(&a, 1000) == HJM_OK && a == first && fake::mallocs == 1);
    CHECK(dev_alloc(&b, 3000) == HJM_OK && fake::mallocs == 2);
    h.c->stream->bad = true;
    dev_free(h.quiesce(), a, b);
    h.give();
    CHECK(fake::device.empty() && fake::frees == 2 && fake::bad_frees == 0);
    CHECK(dev_alloc(&a, 1000) == HJM_OK && fake::mallocs == 3);
    // the stream itself is not kept either
    CHECK(h.take(0, 64) == HJM_OK && !h.c->stream->bad);
}

int main(int argc, char** argv)
{
    const struct {
        const char* name;
        void (*run)();
    } checks[] = {{"blocks_of_a_failed_stream", blocks_of_a_failed_stream}};
    for (const auto& c : checks)
        if (argc == 2 && !strcmp(argv[1], c.name)) {
            c.run();
            return failures ? 1 : 0;
        }
    printf("no such check\n");
    return 2;
}
