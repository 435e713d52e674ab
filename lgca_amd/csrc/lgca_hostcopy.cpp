// lgca_hostcopy.cpp -- large results to ordinary host memory.
//
// A copy to pageable memory goes through the runtime's staging buffer on one
// host thread, which moves 17 GB/s while the link carries 56.  So large copies
// are cut into chunks that kThreads threads take in turn: each has a pinned
// slot and a stream of its own, waits for its chunk and copies it on while the
// others' chunks are on the link.  116 MB: 7.1 ms by the runtime, 2.6 ms so
// (8.4 MB: 0.50 and 0.26).  Three threads fill the link as well as eight, chunks
// of 4 MB are no faster than 2, of 512 KB a third slower (18 us of set-up each).
#include "lgca_hostcopy.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>

namespace lgca {

namespace {

// Below this, starting the threads (26 us each) costs what the chunks gain.
constexpr size_t kStagedBytes = (size_t)6 << 20;

}  // namespace

bool pageable(const void* p)
{
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

bool HostCopier::prepare()
{
    if (slots_) return true;
    bool ok = hipHostMalloc((void**)&slots_, kThreads * kSlotBytes, hipHostMallocDefault) == hipSuccess;
    for (hipStream_t& s : streams_) ok = ok && hipStreamCreateWithFlags(&s, hipStreamNonBlocking) == hipSuccess;
    if (ok) ok = hipEventCreateWithFlags(&event_, hipEventDisableTiming) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
        release();
    }
    return ok;
}

void HostCopier::release()
{
    for (hipStream_t& s : streams_) {
        if (s) (void)hipStreamDestroy(s);
        s = nullptr;
    }
    if (event_) (void)hipEventDestroy(event_);
    event_ = nullptr;
    if (slots_) (void)hipHostFree(slots_);
    slots_ = nullptr;
}

hipError_t HostCopier::staged(const HostCopy* list, int n, size_t total, hipStream_t s)
{
    // at least two chunks a thread
    const size_t chunk = std::min(kSlotBytes, std::max(total / (2 * kThreads), kSlotBytes / 4));
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    if ((e = hipEventRecord(event_, s)) != hipSuccess) return e;
    for (hipStream_t c : streams_)
        if ((e = hipStreamWaitEvent(c, event_, 0)) != hipSuccess) return e;
    std::atomic<size_t> next{0};
    std::atomic<int> error{hipSuccess};
    auto work = [&](int t) {
        hipError_t w = hipSetDevice(device);
        char* slot = slots_ + (size_t)t * kSlotBytes;
        while (w == hipSuccess && error.load(std::memory_order_relaxed) == hipSuccess) {
            size_t i = next.fetch_add(1, std::memory_order_relaxed);
            int k = 0;
            for (; k < n; ++k) {
                const size_t chunks = (list[k].bytes + chunk - 1) / chunk;
                if (i < chunks) break;
                i -= chunks;
            }
            if (k == n) return;
            const size_t at = i * chunk, bytes = std::min(chunk, list[k].bytes - at);
            w = hipMemcpyAsync(slot, (const char*)list[k].src + at, bytes, hipMemcpyDeviceToHost, streams_[t]);
            if (w == hipSuccess) w = hipStreamSynchronize(streams_[t]);
            if (w == hipSuccess) std::memcpy((char*)list[k].dst + at, slot, bytes);
        }
        int none = hipSuccess;
        if (w != hipSuccess) error.compare_exchange_strong(none, (int)w);
    };
    std::thread more[kThreads - 1];
    try {
        for (int t = 1; t < kThreads; ++t) more[t - 1] = std::thread(work, t);
    } catch (const std::system_error&) {
        // no further thread: those there are, and this one, do the work
    }
    work(0);
    for (std::thread& t : more)
        if (t.joinable()) t.join();
    return (hipError_t)error.load();
}

hipError_t HostCopier::run(const HostCopy* list, int n, hipStream_t s)
{
    size_t total = 0;
    for (int k = 0; k < n; ++k) total += list[k].bytes;
    if (total >= kStagedBytes) {
        bool all = true;
        for (int k = 0; k < n; ++k) all = all && pageable(list[k].dst);
        if (all && prepare()) return staged(list, n, total, s);
    }
    hipError_t e = hipSuccess;
    for (int k = 0; k < n && e == hipSuccess; ++k)
        e = hipMemcpyAsync(list[k].dst, list[k].src, list[k].bytes, hipMemcpyDeviceToHost, s);
    const hipError_t f = hipStreamSynchronize(s);
    return e != hipSuccess ? e : f;
}

}  // namespace lgca
