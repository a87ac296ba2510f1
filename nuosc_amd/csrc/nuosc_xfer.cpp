// nuosc_xfer.cpp -- the pinned slots and the threads of nuosc_xfer.h.
#include "nuosc_xfer.h"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <exception>
#include <functional>
#include <map>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace nuosc {
namespace {

struct Slot {
    void* p = nullptr;
    // releases to the system: what a kernel wrote to the slot is in host memory once
    // the event is over, also where pinned memory is not coherent by default
    hipEvent_t done = nullptr;
};
constexpr int kMaxSlots = 2 * kXferThreads;   // per device: 64 MiB of pinned memory

struct DeviceSlots {
    std::vector<Slot> idle;
    int made = 0;
};
std::mutex g_mu;
std::condition_variable g_cv;
std::map<int, DeviceSlots> g_slots;
int g_handles = 0;

void free_slot(Slot& s) {
    if (s.done) (void)hipEventDestroy(s.done);
    if (s.p) (void)hipHostFree(s.p);
    s = Slot{};
}
// (an event belongs to the device that is current when it is made, and can be
// recorded on that device's streams only: the caller may have another one current)
bool make_slot(int device, Slot& s) {
    int current = device;
    (void)hipGetDevice(&current);
    if (current != device) (void)hipSetDevice(device);
    const bool ok = hipHostMalloc(&s.p, kSlotBytes, hipHostMallocPortable) == hipSuccess &&
                    hipEventCreateWithFlags(&s.done, hipEventDisableTiming | hipEventReleaseToSystem) == hipSuccess;
    if (!ok) {
        free_slot(s);
        (void)hipGetLastError();   // (else the next launch check reports it: fewer slots will do)
    }
    if (current != device) (void)hipSetDevice(current);
    return ok;
}

// Adds up to want slots to got, which has room for them (at least one: waits
// while every slot of the device is in use); none if none can be made.
void take_slots(int device, int want, std::vector<Slot>& got) {
    std::unique_lock<std::mutex> lk(g_mu);
    DeviceSlots& d = g_slots[device];
    d.idle.reserve(kMaxSlots);   // (returning a slot allocates nothing)
    while (true) {
        while ((int)got.size() < want && !d.idle.empty()) {
            got.push_back(d.idle.back());
            d.idle.pop_back();
        }
        while ((int)got.size() < want && d.made < kMaxSlots) {
            Slot s;
            if (!make_slot(device, s)) break;
            ++d.made;
            got.push_back(s);
        }
        if (!got.empty() || d.made == 0) return;
        g_cv.wait(lk, [&] { return !d.idle.empty(); });
    }
}
void give_slots(int device, std::vector<Slot>& slots) {
    {
        std::lock_guard<std::mutex> g(g_mu);
        DeviceSlots& d = g_slots[device];
        for (const Slot& s : slots) d.idle.push_back(s);
    }
    g_cv.notify_all();
}

}  // namespace

void xfer_retain() {
    std::lock_guard<std::mutex> g(g_mu);
    ++g_handles;
}
void xfer_release() {
    std::lock_guard<std::mutex> g(g_mu);
    if (--g_handles > 0) return;
    for (auto& kv : g_slots) {   // no handle is left, so none is in use
        for (Slot& s : kv.second.idle) free_slot(s);
        kv.second.idle.clear();
        kv.second.made = 0;
    }
}

hipError_t xfer_run(int device, hipStream_t s, long long nchunks, int nthreads, bool down,
                    const std::function<hipError_t(long long, void*)>& enqueue,
                    const std::function<void(long long, void*)>& host) {
    if (nchunks <= 0) return hipSuccess;
    const int want = (int)std::min<long long>(nchunks, nthreads);
    std::vector<Slot> slots;
    std::vector<std::thread> threads;
    try {
        slots.reserve(want);
        threads.reserve(want);
        take_slots(device, want, slots);
    } catch (const std::bad_alloc&) {
    }
    if (slots.empty()) {
        (void)hipStreamSynchronize(s);   // what the caller queued may read its own memory
        return hipErrorOutOfMemory;
    }
    std::atomic<long long> next{0};
    std::atomic<int> error{hipSuccess};
    auto work = [&](const Slot& slot, bool own_thread) {
        if (own_thread) (void)hipSetDevice(device);   // the device is per host thread
        for (long long c; error.load() == hipSuccess && (c = next.fetch_add(1)) < nchunks;) {
            if (!down) host(c, slot.p);
            hipError_t e = enqueue(c, slot.p);
            if (e == hipSuccess) e = hipEventRecord(slot.done, s);
            if (e == hipSuccess) e = hipEventSynchronize(slot.done);
            if (e != hipSuccess) {
                error.store(e);
                break;
            }
            if (down) host(c, slot.p);
        }
    };
    for (size_t k = 1; k < slots.size(); ++k) {
        try {
            threads.emplace_back(work, std::cref(slots[k]), true);
        } catch (const std::exception&) {   // no thread to be had: the others do its share
            break;
        }
    }
    work(slots[0], false);
    for (std::thread& t : threads) t.join();
    if (error.load() != hipSuccess) (void)hipStreamSynchronize(s);   // nothing queued may still use a slot
    give_slots(device, slots);
    return (hipError_t)error.load();
}

}  // namespace nuosc
