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
    unsigned long long id;   // the runtime's number of the allocation; 0: unknown
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

// The number of the allocation that p belongs to (an address comes back, its number does not);
// 0 if it belongs to none.
unsigned long long buffer_id(void* p)
{
    unsigned long long id = 0;
    if (hipPointerGetAttribute(&id, HIP_POINTER_ATTRIBUTE_BUFFER_ID, (hipDeviceptr_t)p) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return id;
}

// a device reset has ended it
bool gone(const Block& b) { return b.id != 0 && buffer_id(b.p) != b.id; }
bool gone(const PlanContext& c) { return c.mark_id != 0 && buffer_id(c.mark) != c.mark_id; }

void device_free(const Block& b)
{
    if (gone(b)) return;
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
    if (c->host && buffer_id(c->host) == c->host_id) (void)hipHostFree(c->host);
    if (!gone(*c)) {
        for (auto& e : c->ev)
            if (e) (void)hipEventDestroy(e);
        if (c->stream) (void)hipStreamDestroy(c->stream);
        if (c->mark) (void)hipFree(c->mark);
    }
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
            for (;;) {
                auto best = q.idle.end();
                for (auto it = q.idle.begin(); it != q.idle.end(); ++it)
                    if (it->device == device && serves(it->bytes, want) &&
                        (best == q.idle.end() || it->bytes < best->bytes))
                        best = it;
                if (best == q.idle.end()) break;
                const Block b = *best;
                const bool usable = !gone(b);
                if (usable) q.live.insert_or_assign(b.p, b);
                q.idle.erase(best);
                if (!usable) continue;
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
            // (an entry of that address is of a plan that a device reset has outlived)
            q.live.insert_or_assign(p, Block{p, want, device, buffer_id(p)});
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
    Block b{p, 0, 0, 0};
    try {
        std::lock_guard<std::mutex> lock(q.m);
        const auto it = q.live.find(p);
        if (it != q.live.end()) {
            b = it->second;
            q.live.erase(it);
            if (idle && b.bytes <= kPoolBytes && b.id != 0 && !gone(b)) {
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
    for (bool found = true; found && !c;) {
        {
            std::lock_guard<std::mutex> lock(q.m);
            found = false;
            for (size_t i = q.contexts.size(); i-- > 0;)
                if (q.contexts[i]->device == device) {
                    c = q.contexts[i];
                    q.contexts.erase(q.contexts.begin() + (std::ptrdiff_t)i);
                    found = true;
                    break;
                }
        }
        if (c && gone(*c)) {
            context_destroy(c);
            c = nullptr;
        }
    }
    if (!c) {
        c = new (std::nothrow) PlanContext();
        if (!c) return HJM_ERR_ALLOC;
        c->device = device;
        bool ok = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) == hipSuccess;
        for (auto& e : c->ev) ok = ok && hipEventCreate(&e) == hipSuccess;
        ok = ok && hipMalloc(&c->mark, 512) == hipSuccess;
        c->mark_id = ok ? buffer_id(c->mark) : 0;
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
        c->host_id = buffer_id(c->host);
    }
    *out = c;
    return HJM_OK;
}

bool context_quiesce(PlanContext* c) { return gone(*c) || hipStreamSynchronize(c->stream) == hipSuccess; }

void context_release(PlanContext* c)
{
    if (!c) return;
    const bool idle = context_quiesce(c);
    if (idle && c->mark_id != 0 && !gone(*c)) {
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
