// Large copies between the device and pageable host memory, staged through
// pinned slots of the context by several host threads.  The runtime's own
// pageable copy moves a chunk and then lets one thread copy it, 10-15 GB/s
// whatever the link does; here every thread owns some of the slots, so one
// slot is on the link while the others are copied.  51 MB to the host: 5.3 ms
// by the runtime, 3.0 with two threads, 1.7 with four, 1.9 with eight (from
// the host: 1.5 ms throughout).
#include "igr_ctx.hpp"

#include <cstring>

namespace igr_dev {

Staging::~Staging() {
    for (hipEvent_t e : done)
        if (e) (void)hipEventDestroy(e);
    if (mem) (void)hipHostFree(mem);
}

// Whether the slots are there.  The events belong to the context's device,
// whichever the caller has current.
bool Staging::open(int device) {
    if (mem || failed) return mem != nullptr;
    int cur = -1;
    HIP_OK(hipGetDevice(&cur));
    if (cur != device) HIP_OK(hipSetDevice(device));
    char* m = nullptr;
    bool ok = hipHostMalloc(reinterpret_cast<void**>(&m), (size_t)SLOTS * SLOT_BYTES, 0) == hipSuccess;
    for (hipEvent_t& e : done) ok = ok && (e || hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess);
    if (cur != device) (void)hipSetDevice(cur);
    failed = !ok;
    if (failed) {
        (void)hipGetLastError();
        if (m) (void)hipHostFree(m);
        return false;
    }
    mem = m;
    return true;
}

// Chunk k goes through slot k % SLOTS; thread t owns the slots t, t + T, ..,
// so nothing but the stream is shared between threads.
template <class F>
static void over_chunks(int device, int64_t bytes, F&& chunk) {
    const int64_t chunks = (bytes + Staging::SLOT_BYTES - 1) / Staging::SLOT_BYTES;
    int T = std::max(1, std::min(std::min(host_threads(), Staging::THREADS), (int)std::min<int64_t>(Staging::SLOTS, chunks)));
    while (Staging::SLOTS % T) T--;
    igr::parallel_ranges(T, T, [&](int64_t a, int64_t b, int) {
        int cur = -1;   // a thread of its own has device 0; the caller keeps the one it has
        HIP_OK(hipGetDevice(&cur));
        if (cur != device) HIP_OK(hipSetDevice(device));
        for (int64_t t = a; t < b; t++)
            for (int64_t k = t; k < chunks; k += T) {
                const int64_t at = k * Staging::SLOT_BYTES;
                chunk((int)(k % Staging::SLOTS), at, std::min<int64_t>(Staging::SLOT_BYTES, bytes - at));
            }
        if (cur != device) (void)hipSetDevice(cur);
    });
}

// The slots for a copy of this size, held while the lock lives; none for a small
// copy and without pinned memory.
static std::unique_lock<std::mutex> use_slots(igr_ctx* c, int64_t bytes) {
    Staging& g = c->staging;
    if (bytes < Staging::MIN_BYTES) return {};
    std::unique_lock<std::mutex> lk(g.mu);
    if (!g.open(c->device)) return {};
    return lk;
}

void copy_to_host(igr_ctx* c, void* dst, const void* src, int64_t bytes, hipStream_t s) {
    Staging& g = c->staging;
    const auto slots = use_slots(c, bytes);
    if (!slots) {
        HIP_OK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s));
        HIP_OK(hipStreamSynchronize(s));
        return;
    }
    const auto start = [&](int slot, int64_t at) {
        HIP_OK(hipMemcpyAsync(g.slot(slot), static_cast<const char*>(src) + at,
                              std::min<int64_t>(Staging::SLOT_BYTES, bytes - at), hipMemcpyDeviceToHost, s));
        HIP_OK(hipEventRecord(g.done[slot], s));
    };
    for (int k = 0; k < Staging::SLOTS && k * Staging::SLOT_BYTES < bytes; k++) {
        HIP_OK(hipEventSynchronize(g.done[k]));   // an earlier upload from the slot
        start(k, k * Staging::SLOT_BYTES);
    }
    over_chunks(c->device, bytes, [&](int slot, int64_t at, int64_t len) {
        HIP_OK(hipEventSynchronize(g.done[slot]));
        std::memcpy(static_cast<char*>(dst) + at, g.slot(slot), len);
        const int64_t next = at + (int64_t)Staging::SLOTS * Staging::SLOT_BYTES;
        if (next < bytes) start(slot, next);
    });
}

void copy_to_device(igr_ctx* c, void* dst, const void* src, int64_t bytes, hipStream_t s) {
    Staging& g = c->staging;
    const auto slots = use_slots(c, bytes);
    if (!slots) {
        if (bytes) HIP_OK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s));
        return;
    }
    over_chunks(c->device, bytes, [&](int slot, int64_t at, int64_t len) {
        HIP_OK(hipEventSynchronize(g.done[slot]));
        std::memcpy(g.slot(slot), static_cast<const char*>(src) + at, len);
        HIP_OK(hipMemcpyAsync(static_cast<char*>(dst) + at, g.slot(slot), len, hipMemcpyHostToDevice, s));
        HIP_OK(hipEventRecord(g.done[slot], s));
    });
}

} // namespace igr_dev
