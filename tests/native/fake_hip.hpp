// A HIP runtime for host tests of the engine: memory is malloc's, streams and
// events do nothing, copies happen at once.  A countdown makes an allocation fail.
// Kernels that a test meets are defined there; the others stay unresolved.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>

namespace fake {
inline long allocations = 0;    // so far
inline long fail_alloc = -1;    // allocations until one fails; -1: none does
inline bool alloc_fails()
{
     ++allocations;
     return fail_alloc >= 0 && fail_alloc-- == 0;
}
inline hipError_t alloc(void** p, size_t n)
{
     if (alloc_fails()) return hipErrorOutOfMemory;
     *p = std::malloc(n ? n : 1);
     return hipSuccess;
}
inline int handle;  // what streams and events point to
}  // namespace fake

extern "C" {
hipError_t hipGetDeviceCount(int* n)
{
     *n = 1;
     return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "injected error"; }
hipError_t hipMalloc(void** p, size_t n) { return fake::alloc(p, n); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return fake::alloc(p, n); }
hipError_t hipFree(void* p)
{
     std::free(p);
     return hipSuccess;
}
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
     std::memcpy(d, s, n);
     return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
     *s = reinterpret_cast<hipStream_t>(&fake::handle);
     return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
     *e = reinterpret_cast<hipEvent_t>(&fake::handle);
     return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
     *ms = 0;
     return hipSuccess;
}
}
