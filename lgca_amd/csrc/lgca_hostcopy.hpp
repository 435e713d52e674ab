// lgca_hostcopy.hpp -- large results to ordinary host memory.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>

namespace lgca {

struct HostCopy {
    void* dst;        // host
    const void* src;  // device
    size_t bytes;
};

// Whether a host copy goes through a staging buffer: pinned, managed and device
// memory is copied to directly.
bool pageable(const void* p);

// Copies through pinned slots of its own, made on the first large copy and
// given back by release() (or the destructor).  Not for several threads at
// once: its owner's lock covers it.
class HostCopier {
public:
    HostCopier() = default;
    HostCopier(const HostCopier&) = delete;
    HostCopier& operator=(const HostCopier&) = delete;
    ~HostCopier() { release(); }

    // Copies list[0..n), made by the work on `s`; returns when they are done.
    hipError_t run(const HostCopy* list, int n, hipStream_t s);
    void release();

private:
    static constexpr int kThreads = 4;
    static constexpr size_t kSlotBytes = (size_t)2 << 20;

    bool prepare();
    hipError_t staged(const HostCopy* list, int n, size_t total, hipStream_t s);

    char* slots_ = nullptr;
    hipStream_t streams_[kThreads] = {};
    hipEvent_t event_ = nullptr;
};

}  // namespace lgca
