// tws_transfer.hip -- copies between the caller's host arrays and the device.
//
// The caller's arrays are pageable, and the runtime copies such memory through
// pinned memory of its own on the calling thread, which one core's copying
// bounds well below the link.  Large copies are cut into chunks here that a few
// threads copy through pinned slots, so the link moves one chunk while others are
// copied.
// MI355X, us a pass before -> after: 1331 x 1024, 32.7 MB up, 100 steps, 38.2 MB
// down, 3740 -> 3000; 1000 x 700 textures, 22.4 MB up, 30 steps, 25.2 MB down, 3600
// (2360 on another box) -> 2050.

#include "tws_transfer.hpp"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>

namespace tws {

namespace {

// Few and large chunks: a chunk's copy and event cost the host some 40 us.  us a
// pass of the 1331 x 1024 roundtrip by threads, slots of each and MiB a chunk:
// 4, 2, 1/2 4310; 4, 2, 1 3360; 8, 2, 1 3580; 4, 2, 2 3070; 4, 1, 4 2990; 4, 2, 4 2990.
constexpr size_t kChunk = 4 << 20;
constexpr int kThreads = 4;  // a slot each
// Copies below this stay with the runtime: starting the threads and their few
// large chunks costs more.  ms by MiB, runtime and threads: up 16 0.51, 0.55; 24
// 0.76, 0.75; 32 1.15, 0.96; 128 4.9, 3.4; down 4 0.24, 0.27; 6 0.37, 0.31; 16 1.02,
// 0.57; 32 3.6, 1.6; 128 13.2, 4.2.
constexpr size_t kStagedUp = 24 << 20, kStagedDown = 5 << 20;
constexpr int kMaxIdle = 2;  // stagings kept while no copy uses them

struct Staging {
    char* pinned = nullptr;
    hipEvent_t done[kThreads] = {};
    int device = -1;
    Staging* next = nullptr;

    ~Staging() {
        for (hipEvent_t e : done)
            if (e) (void)hipEventDestroy(e);
        if (pinned) (void)hipHostFree(pinned);
    }
};

std::mutex g_mu;
Staging* g_idle = nullptr;
int g_users = 0;

Staging* lease(int device) {
    {
        std::lock_guard<std::mutex> lk(g_mu);
        for (Staging** p = &g_idle; *p; p = &(*p)->next)
            if ((*p)->device == device) {
                Staging* st = *p;
                *p = st->next;
                return st;
            }
    }
    Staging* st = new (std::nothrow) Staging();
    if (!st) return nullptr;
    st->device = device;
    bool ok = hipHostMalloc(&st->pinned, kChunk * kThreads, hipHostMallocDefault) == hipSuccess;
    for (hipEvent_t& e : st->done)
        ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    if (ok) return st;
    (void)hipGetLastError();
    delete st;
    return nullptr;
}

void give_back(Staging* st) {
    {
        std::lock_guard<std::mutex> lk(g_mu);
        int idle = 0;
        for (Staging* p = g_idle; p; p = p->next) ++idle;
        if (g_users > 0 && idle < kMaxIdle) {
            st->next = g_idle;
            g_idle = st;
            return;
        }
    }
    delete st;
}

// Thread t's chunks t, t + kThreads, ...; returns with its slot free.
template <bool UP>
hipError_t copy_chunks(Staging& st, int t, char* device, char* host, size_t bytes, hipStream_t s) {
    hipError_t e = hipSetDevice(st.device);
    char* const slot = st.pinned + (size_t)t * kChunk;
    for (size_t at = (size_t)t * kChunk; at < bytes && e == hipSuccess;
         at += (size_t)kThreads * kChunk) {
        const size_t n = std::min(kChunk, bytes - at);
        if (UP) std::memcpy(slot, host + at, n);
        e = UP ? hipMemcpyAsync(device + at, slot, n, hipMemcpyHostToDevice, s)
               : hipMemcpyAsync(slot, device + at, n, hipMemcpyDeviceToHost, s);
        if (e != hipSuccess) break;
        e = hipEventRecord(st.done[t], s);
        // the copy may be in flight even where the event failed
        const hipError_t w = e == hipSuccess ? hipEventSynchronize(st.done[t])
                                             : hipStreamSynchronize(s);
        if (e == hipSuccess) e = w;
        if (!UP && e == hipSuccess) std::memcpy(host + at, slot, n);
    }
    return e;
}

template <bool UP>
hipError_t copy(char* device, char* host, size_t bytes, hipStream_t s) {
    const auto direct = [&]() {
        return UP ? hipMemcpyAsync(device, host, bytes, hipMemcpyHostToDevice, s)
                  : hipMemcpyAsync(host, device, bytes, hipMemcpyDeviceToHost, s);
    };
    if (bytes < (UP ? kStagedUp : kStagedDown)) return direct();
    // memory that is pinned already needs no copy on the way
    hipPointerAttribute_t attr{};
    if (hipPointerGetAttributes(&attr, host) != hipSuccess) (void)hipGetLastError();
    else if (attr.type != hipMemoryTypeUnregistered) return direct();
    int device_id = -1;
    if (hipGetDevice(&device_id) != hipSuccess) return direct();
    Staging* const st = lease(device_id);
    if (!st) return direct();
    hipError_t result[kThreads] = {};
    std::thread threads[kThreads];
    auto run = [&](int t) { result[t] = copy_chunks<UP>(*st, t, device, host, bytes, s); };
    for (int t = 1; t < kThreads; ++t) {
        try {
            threads[t] = std::thread(run, t);
        } catch (...) {  // no thread to be had: this one copies its part below
        }
    }
    run(0);
    for (int t = 1; t < kThreads; ++t) {
        if (threads[t].joinable()) threads[t].join();
        else run(t);
    }
    give_back(st);
    for (hipError_t e : result)
        if (e != hipSuccess) return e;
    return hipSuccess;
}

}  // namespace

hipError_t copy_to_device(void* device, const void* host, size_t bytes, hipStream_t s) {
    return copy<true>(static_cast<char*>(device), const_cast<char*>(static_cast<const char*>(host)),
                      bytes, s);
}

hipError_t copy_to_host(void* host, const void* device, size_t bytes, hipStream_t s) {
    return copy<false>(const_cast<char*>(static_cast<const char*>(device)), static_cast<char*>(host),
                       bytes, s);
}

TransferUser::TransferUser() {
    std::lock_guard<std::mutex> lk(g_mu);
    ++g_users;
}

TransferUser::~TransferUser() {
    Staging* list = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        if (--g_users == 0) {
            list = g_idle;
            g_idle = nullptr;
        }
    }
    while (list) {
        Staging* const st = list;
        list = st->next;
        delete st;
    }
}

}  // namespace tws
