// msm_copy.cpp -- pinned-ring copies (msm_copy.h).
#include "msm_copy.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>

namespace msm {

namespace {

struct Ring {
    std::mutex mu;            // everything below, and one transfer at a time
    int users = 0;
    bool refused = false;     // the memory could not be pinned
    char* base = nullptr;
    hipEvent_t ev[kCopySlots] = {};
};

constexpr int kMaxDevices = 64;

Ring* ring_of(int device) {
    static Ring rings[kMaxDevices];
    return device >= 0 && device < kMaxDevices ? &rings[device] : nullptr;
}

void drop(Ring& r) {
    for (hipEvent_t& e : r.ev) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    if (r.base) (void)hipHostFree(r.base);
    r.base = nullptr;
}

// Whether there is a ring (r.mu held): the first copy that asks pins it.
bool pinned(Ring& r) {
    if (r.base) return true;
    if (r.users == 0 || r.refused) return false;
    hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&r.base), kCopySlots * kCopySlotBytes);
    if (e != hipSuccess) r.base = nullptr;
    for (int k = 0; k < kCopySlots && e == hipSuccess; ++k)
        e = hipEventCreateWithFlags(&r.ev[k], hipEventDisableTiming);
    if (e == hipSuccess) return true;
    drop(r);
    r.refused = true;
    (void)hipGetLastError();
    return false;
}

// Runs work(slot) on the calling thread (slot 0) and up to extra others; a thread that cannot be
// had is one fewer.
template <typename F>
void on_threads(int extra, F&& work) {
    std::thread th[kCopySlots];
    int n = 0;
    for (; n < extra; ++n) {
        try {
            th[n] = std::thread(work, n + 1);
        } catch (...) {
            break;
        }
    }
    work(0);
    for (int k = 0; k < n; ++k) th[k].join();
}

}  // namespace

void copy_ring_acquire(int device) {
    Ring* r = ring_of(device);
    if (!r) return;
    std::lock_guard<std::mutex> g(r->mu);
    ++r->users;
}

void copy_ring_release(int device) {
    Ring* r = ring_of(device);
    if (!r) return;
    std::lock_guard<std::mutex> g(r->mu);
    if (r->users == 0 || --r->users > 0) return;
    drop(*r);
    r->refused = false;
}

hipError_t copy_to_host(int device, const void* base, size_t total, const CopyPart* parts,
                        int nparts, hipStream_t stream) {
    // the stream's earlier work ends before the ring is taken, for other streams to use it meanwhile
    const hipError_t idle = hipStreamSynchronize(stream);
    if (idle != hipSuccess || total == 0) return idle;
    const bool one_slot = nparts > 1 && total <= kOneSlot;
    Ring* r = one_slot || total > kRingFrom ? ring_of(device) : nullptr;
    std::unique_lock<std::mutex> g;
    if (r) g = std::unique_lock<std::mutex>(r->mu);
    if (!r || !pinned(*r)) {
        if (r) g.unlock();
        hipError_t e = hipSuccess;
        for (int k = 0; k < nparts && e == hipSuccess; ++k)
            e = hipMemcpyAsync(parts[k].host, static_cast<const char*>(base) + parts[k].offset,
                               parts[k].bytes, hipMemcpyDeviceToHost, stream);
        const hipError_t done = hipStreamSynchronize(stream);
        return e != hipSuccess ? e : done;
    }
    // an equal share a slot, in chunks of at most the slot; or all of it through the first
    const size_t share = ((total + kCopySlots - 1) / kCopySlots + 4095) & ~size_t(4095);
    const size_t chunk = one_slot ? total : std::min(kCopySlotBytes, share);
    std::atomic<size_t> next{0};
    std::atomic<int> err{hipSuccess};
    on_threads(one_slot ? 0 : kCopySlots - 1, [&](int slot) {
        if (slot > 0 && hipSetDevice(device) != hipSuccess) return;
        char* pin = r->base + slot * kCopySlotBytes;
        for (;;) {
            const size_t a = next.fetch_add(chunk);
            if (a >= total || err.load() != hipSuccess) return;
            const size_t b = std::min(a + chunk, total);
            hipError_t e = hipMemcpyAsync(pin, static_cast<const char*>(base) + a, b - a,
                                          hipMemcpyDeviceToHost, stream);
            if (e == hipSuccess) e = hipEventRecord(r->ev[slot], stream);
            if (e == hipSuccess) e = hipEventSynchronize(r->ev[slot]);
            if (e != hipSuccess) {
                err.store(e);
                return;
            }
            for (int k = 0; k < nparts; ++k) {
                const size_t lo = std::max(a, parts[k].offset),
                             hi = std::min(b, parts[k].offset + parts[k].bytes);
                if (lo < hi)
                    std::memcpy(static_cast<char*>(parts[k].host) + (lo - parts[k].offset),
                                pin + (lo - a), hi - lo);
            }
        }
    });
    return static_cast<hipError_t>(err.load());
}

}  // namespace msm
