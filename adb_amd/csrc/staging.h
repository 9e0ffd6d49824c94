// staging.h - pinned host memory for the single-contact entry points.
//
// Such a call is all latency, and six device allocations, their frees and five
// copies were most of it.  The kernel reads its few inputs from pinned host
// memory and writes its results there, so a call is a launch and a wait: a
// point-triangle Hessian 150 -> 33 us (of which its kernel is also shorter, see
// contact.hip), a collision time 47 -> 16 us.  One page per calling thread, freed
// when the thread ends.
#pragma once
#include <hip/hip_runtime.h>

namespace adb {

struct HostStaging {
    static constexpr size_t N = 512;          // doubles
    double* p = nullptr;
    // null when the allocation fails (no device)
    double* get() {
        if (!p && hipHostMalloc((void**)&p, N * sizeof(double), hipHostMallocMapped | hipHostMallocPortable) != hipSuccess) p = nullptr;
        return p;
    }
    ~HostStaging() { if (p) (void)hipHostFree(p); }
};
inline HostStaging& host_staging() {
    static thread_local HostStaging s;
    return s;
}

} // namespace adb
