// hjm_pool.h -- device memory, streams and events kept between plans.
//
// hipMalloc and hipFree of large blocks map and unmap (and clear) their pages, at about
// 33 GB/s on an MI355X: a one-call CVA with Greeks at 65536 paths x 10y spent 23 of its 24 ms
// there, the full book's at 65536 paths x 30y 175 of 182 ms. Freed blocks therefore go to a
// per-device cache and are handed out again to requests they fit. The cache
//   * holds at most kPoolBytes per device (the oldest blocks are returned to the device
//     beyond that; larger blocks never enter), gives everything back when an allocation
//     fails (which is then tried again) and on hjm_release_cached_memory;
//   * takes a block only when no work on it is outstanding: whoever frees one has
//     synchronised the stream that used it (hipFree used to wait for the device), and says so
//     if that failed: such a block goes back to the device and to no other plan;
//   * survives hipDeviceReset: the runtime numbers its allocations, and a block (or a context, by
//     its mark) whose number is no longer the one it was given is forgotten, not handed out and
//     not freed (60 ns a look);
//   * is behind one mutex: any thread may allocate and free on any device.
// Blocks come back with their old contents, as undefined as hipMalloc's.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace hjm_host {

constexpr size_t kPoolBytes = (size_t)8 << 30;  // cached (unused) bytes per device
constexpr int kPoolContexts = 8;                // idle plan contexts per device

// Memory of the current device; hipErrorOutOfMemory (or the runtime's error) on failure.
hipError_t pool_alloc(void** p, size_t bytes);
// idle: the work that used the block is known to be done, so it may be kept.
void pool_free(void* p, bool idle);
void pool_release_all();

// A plan's stream (non-blocking, default priority), timing events and pinned host buffer.
struct PlanContext {
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev[7] = {};
    void* host = nullptr;      // pinned, host_bytes long
    size_t host_bytes = 0;
    void* mark = nullptr;      // a small block: gone with the stream if the device was reset
    unsigned long long mark_id = 0, host_id = 0;
};
// A context of the current device (an idle one if there is); HJM_ERR_ALLOC if its pinned
// buffer cannot be had, after the cache was given back, HJM_ERR_DEVICE if its stream cannot.
int context_acquire(int device, size_t host_bytes, PlanContext** out);
// Waits for the context's stream (true as well if a device reset has ended it).
bool context_quiesce(PlanContext* c);
// Waits for the context's stream, then keeps the context for the next plan.
void context_release(PlanContext* c);

}  // namespace hjm_host
