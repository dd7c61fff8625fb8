// hjm_pool.hip -- the device-memory and plan-context cache of hjm_pool.h (host code).
#include "hjm_pool.h"

#include <algorithm>
#include <deque>
#include <mutex>
#include <new>
#include <unordered_map>
#include <vector>

#include "hjm_cva.h"

namespace hjm_host {
namespace {

struct Block {
    void* p;
    size_t bytes;
    int device;
};

struct Pool {
    std::mutex m;
    std::unordered_map<void*, Block> live;  // handed out
    std::deque<Block> idle;                 // oldest first, all devices
    std::vector<PlanContext*> contexts;     // idle
};

// never destroyed: the HIP runtime may be gone when static destructors run
Pool& pool()
{
    static Pool* p = new Pool();
    return *p;
}

// Sizes in steps of 1/8 of their power of two, at least 512 bytes and at most 2 MB: repeated
// calls of nearby sizes share blocks. What is too large to be kept is not rounded.
size_t rounded(size_t bytes)
{
    if (bytes > kPoolBytes) return bytes;
    size_t step = 512;
    while (step * 16 < bytes && step < ((size_t)2 << 20)) step *= 2;
    return (bytes + step - 1) / step * step;
}

// A kept block serves a request of `want` bytes if it is larger by no more than 1/8, or 16 MB:
// what a plan holds beyond its needs does not decide whether it fits the card.
bool serves(size_t bytes, size_t want)
{
    return bytes >= want && bytes - want <= std::min(want / 8, (size_t)16 << 20);
}

void device_free(const Block& b)
{
    int prev = -1;
    (void)hipGetDevice(&prev);
    if (prev != b.device) (void)hipSetDevice(b.device);
    (void)hipFree(b.p);
    if (prev >= 0 && prev != b.device) (void)hipSetDevice(prev);
}

void context_destroy(PlanContext* c)
{
    int prev = -1;
    (void)hipGetDevice(&prev);
    if (prev != c->device) (void)hipSetDevice(c->device);
    if (c->host) (void)hipHostFree(c->host);
    for (auto& e : c->ev)
        if (e) (void)hipEventDestroy(e);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    if (prev >= 0 && prev != c->device) (void)hipSetDevice(prev);
    delete c;
}

}  // namespace

hipError_t pool_alloc(void** out, size_t bytes)
{
    *out = nullptr;
    int device = -1;
    hipError_t err = hipGetDevice(&device);
    if (err != hipSuccess) return err;
    size_t want = rounded(bytes);
    Pool& q = pool();
    try {
        {
            std::lock_guard<std::mutex> lock(q.m);
            auto best = q.idle.end();
            for (auto it = q.idle.begin(); it != q.idle.end(); ++it)
                if (it->device == device && serves(it->bytes, want) &&
                    (best == q.idle.end() || it->bytes < best->bytes))
                    best = it;
            if (best != q.idle.end()) {
                const Block b = *best;
                q.live.emplace(b.p, b);
                q.idle.erase(best);
                *out = b.p;
                return hipSuccess;
            }
        }
        void* p = nullptr;
        err = hipMalloc(&p, want);
        if (err != hipSuccess) {
            (void)hipGetLastError();
            pool_release_all();
            err = hipMalloc(&p, want = bytes);
            if (err != hipSuccess) {
                (void)hipGetLastError();
                return err;
            }
        }
        try {
            std::lock_guard<std::mutex> lock(q.m);
            q.live.emplace(p, Block{p, want, device});
        } catch (...) {
            (void)hipFree(p);
            return hipErrorOutOfMemory;
        }
        *out = p;
        return hipSuccess;
    } catch (...) {
        return hipErrorOutOfMemory;
    }
}

void pool_free(void* p, bool idle)
{
    if (!p) return;
    Pool& q = pool();
    std::vector<Block> drop;
    Block b{p, 0, 0};
    try {
        std::lock_guard<std::mutex> lock(q.m);
        const auto it = q.live.find(p);
        if (it != q.live.end()) {
            b = it->second;
            q.live.erase(it);
            if (idle && b.bytes <= kPoolBytes) {
                size_t held = b.bytes;
                for (const Block& x : q.idle) held += x.device == b.device ? x.bytes : 0;
                for (auto x = q.idle.begin(); held > kPoolBytes && x != q.idle.end();) {
                    if (x->device != b.device) {
                        ++x;
                        continue;
                    }
                    drop.push_back(*x);
                    held -= x->bytes;
                    x = q.idle.erase(x);
                }
                q.idle.push_back(b);
                b.p = nullptr;
            }
        }
    } catch (...) {
        // bookkeeping memory ran out: the block itself goes back to the device below
    }
    if (b.p) {
        if (b.bytes) device_free(b);
        else (void)hipFree(p);
    }
    for (const Block& x : drop) device_free(x);
}

void pool_release_all()
{
    Pool& q = pool();
    std::deque<Block> idle;
    std::vector<PlanContext*> contexts;
    {
        std::lock_guard<std::mutex> lock(q.m);
        idle.swap(q.idle);
        contexts.swap(q.contexts);
    }
    for (const Block& b : idle) device_free(b);
    for (PlanContext* c : contexts) context_destroy(c);
}

int context_acquire(int device, size_t host_bytes, PlanContext** out)
{
    *out = nullptr;
    Pool& q = pool();
    PlanContext* c = nullptr;
    {
        std::lock_guard<std::mutex> lock(q.m);
        for (size_t i = q.contexts.size(); i-- > 0;)
            if (q.contexts[i]->device == device) {
                c = q.contexts[i];
                q.contexts.erase(q.contexts.begin() + (std::ptrdiff_t)i);
                break;
            }
    }
    if (!c) {
        c = new (std::nothrow) PlanContext();
        if (!c) return HJM_ERR_ALLOC;
        c->device = device;
        bool ok = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) == hipSuccess;
        for (auto& e : c->ev) ok = ok && hipEventCreate(&e) == hipSuccess;
        if (!ok) {
            (void)hipGetLastError();
            context_destroy(c);
            return HJM_ERR_DEVICE;
        }
    }
    if (c->host_bytes < host_bytes) {
        if (c->host) (void)hipHostFree(c->host);
        c->host = nullptr;
        c->host_bytes = 0;
        auto take = [&] {
            if (hipHostMalloc(&c->host, host_bytes, hipHostMallocDefault) == hipSuccess) return true;
            (void)hipGetLastError();
            c->host = nullptr;
            return false;
        };
        if (!take()) {
            pool_release_all();   // the idle contexts' buffers
            if (!take()) {
                context_destroy(c);
                return HJM_ERR_ALLOC;
            }
        }
        c->host_bytes = host_bytes;
    }
    *out = c;
    return HJM_OK;
}

void context_release(PlanContext* c)
{
    if (!c) return;
    const bool idle = hipStreamSynchronize(c->stream) == hipSuccess;
    if (idle) {
        Pool& q = pool();
        try {
            std::lock_guard<std::mutex> lock(q.m);
            int n = 0;
            for (const PlanContext* x : q.contexts) n += x->device == c->device ? 1 : 0;
            if (n < kPoolContexts) {
                q.contexts.push_back(c);
                return;
            }
        } catch (...) {
        }
    }
    context_destroy(c);
}

}  // namespace hjm_host

extern "C" void hjm_release_cached_memory(void) { hjm_host::pool_release_all(); }
