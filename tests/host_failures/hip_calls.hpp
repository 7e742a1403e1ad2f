// A device without a GPU: the HIP calls that the library's host code makes, defined by the test
// program and so taken before the runtime's.  Memory is the host's, copies happen at once,
// kernels do not run; calls can be made to fail.
#pragma once
#include "context.hpp"

#include <cstdio>
#include <cstdlib>
#include <map>

namespace fake {
inline int launches = 0;         // since the start
inline int in_flight = 0;        // launches since the last synchronisation
inline int fail_launch = -1;     // number of the launch that fails
inline bool fail_pinned = false; // pinned allocations fail
inline hipError_t last = hipSuccess;
inline std::map<void*, unsigned> pinned;   // flags of the pinned allocations
}  // namespace fake

extern "C" {
hipError_t hipMalloc(void** p, size_t n) { *p = std::calloc(n ? n : 1, 1); return hipSuccess; }
hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) {
    *p = nullptr;
    if (fake::fail_pinned) return hipErrorOutOfMemory;
    *p = std::calloc(n ? n : 1, 1);
    fake::pinned[*p] = flags;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { std::free(p); fake::pinned.erase(p); return hipSuccess; }
// a launch's shape on its way to hipLaunchKernel
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
    if (fake::launches++ == fake::fail_launch) return fake::last = hipErrorLaunchFailure;
    ++fake::in_flight;
    return hipSuccess;
}
hipError_t hipGetLastError() { const hipError_t e = fake::last; fake::last = hipSuccess; return e; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { fake::in_flight = 0; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return fake::in_flight ? hipErrorNotReady : hipSuccess; }
}

namespace cipc {
// the library's scans go through rocPRIM, which asks for a device
void exclusive_scan_int(Context&, const int*, int*, int) {}
}  // namespace cipc

#define EXPECT(c) do { if (!(c)) { std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c); return 1; } } while (0)
