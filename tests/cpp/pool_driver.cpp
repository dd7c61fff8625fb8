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
    CHECK(a == nullptr && dev_alloc(&a, 1000) == HJM_OK && a == first);
    CHECK(dev_alloc(&b, 3000) == HJM_OK && b != first);
    h.c->stream->bad = true;
    dev_free(h.quiesce(), a, b);
    h.give();
    CHECK(fake::device.empty() && fake::bad_frees == 0);
    const int mallocs = fake::mallocs;
    CHECK(dev_alloc(&a, 1000) == HJM_OK && fake::mallocs == mallocs + 1);
    // the stream itself is not kept either
    CHECK(h.take(0, 64) == HJM_OK && !h.c->stream->bad);
}

// A pinned buffer that cannot be had is an allocation failure, as a device block is, and is
// reported only after the idle contexts' buffers were given back.
static void pinned_buffers_that_cannot_be_had()
{
    ContextHolder a, b, c, d;
    CHECK(a.take(0, 1 << 20) == HJM_OK && b.take(0, 1 << 20) == HJM_OK);
    a.give();
    b.give();
    fake::pinned_budget = 5 << 19;   // two and a half such buffers
    CHECK(c.take(0, 2 << 20) == HJM_OK);   // one context's buffer grows, the other's goes
    CHECK(d.take(0, 1 << 20) == HJM_ERR_ALLOC);
    CHECK(d.c == nullptr && fake::streams.size() == 1 && fake::pinned.size() == 1 && fake::bad_frees == 0);
}

// What fits the card is not refused for being rounded up: one block too large to be kept, several
// that could be, and a card with less than a rounding left.
static void memory_close_to_the_cards()
{
    const size_t gb = (size_t)1 << 30;
    char *a = nullptr, *b[10] = {}, *c = nullptr;
    fake::budget = 20 * gb - gb / 20;
    CHECK(dev_alloc(&a, 20 * gb - gb / 10) == HJM_OK);
    dev_free(true, a);
    CHECK(fake::device.empty());
    fake::budget = 43 * gb + 10 * ((size_t)2 << 20);
    for (auto& p : b) CHECK(dev_alloc(&p, 43 * (gb / 10)) == HJM_OK);
    // blocks kept are not handed to requests far smaller
    const int before = fake::mallocs;
    for (auto& p : b) dev_free(true, p);
    CHECK(dev_alloc(&c, 4 * gb) == HJM_OK && fake::mallocs > before);
    dev_free(true, c);
    pool_release_all();
    CHECK(fake::device.empty());
    fake::budget = 1000001;   // rounded: 1048576
    CHECK(dev_alloc(&c, 1000001) == HJM_OK);
}

// After hipDeviceReset nothing from before it is handed out, waited for or freed, also where the
// runtime has given its address to somebody else by then.
static void a_device_reset()
{
    ContextHolder kept, held;
    double *a = nullptr, *b = nullptr, *c = nullptr;
    CHECK(kept.take(0, 64) == HJM_OK && held.take(0, 64) == HJM_OK);
    CHECK(dev_alloc(&a, 1000) == HJM_OK && dev_alloc(&b, 1000) == HJM_OK && dev_alloc(&c, 5000) == HJM_OK);
    double* const old = a;
    dev_free(kept.quiesce(), a);
    kept.give();
    fake::reset();
    void* theirs = nullptr;   // another user of the device, at the cached block's address
    while (theirs != old) CHECK(hipMalloc(&theirs, 8192) == hipSuccess);
    ContextHolder after;
    CHECK(after.take(0, 64) == HJM_OK && fake::streams.count(after.c->stream) == 1);
    CHECK(dev_alloc(&a, 1000) == HJM_OK && a != old);
    // a plan from before the reset goes
    const bool clean = held.quiesce();
    CHECK(clean);
    dev_free(clean, c);
    held.give();
    CHECK(fake::bad_frees == 0);
    double* d = nullptr;
    CHECK(dev_alloc(&d, 5000) == HJM_OK && fake::device.count((uintptr_t)d) == 1);
    dev_free(after.quiesce(), a, d);
    after.give();
    hjm_release_cached_memory();
    CHECK(fake::bad_frees == 0 && fake::streams.empty() && fake::pinned.empty());
    for (const auto& x : fake::device) CHECK(x.second.bytes == 8192);   // theirs
}

int main(int argc, char** argv)
{
    const struct {
        const char* name;
        void (*run)();
    } checks[] = {{"blocks_of_a_failed_stream", blocks_of_a_failed_stream},
                  {"a_device_reset", a_device_reset},
                  {"memory_close_to_the_cards", memory_close_to_the_cards},
                  {"pinned_buffers_that_cannot_be_had", pinned_buffers_that_cannot_be_had}};
    for (const auto& c : checks)
        if (argc == 2 && !strcmp(argv[1], c.name)) {
            c.run();
            return failures ? 1 : 0;
        }
    printf("no such check\n");
    return 2;
}
