// Host stand-ins for the HIP declarations that channel_flow_amd/csrc/hostcopy.hip
// uses, for its CPU test: device memory is host memory and every copy is done when
// it is asked for.
#pragma once
#include <cstdlib>
#include <cstring>

#define __device__
#define __host__
#define __forceinline__ inline

struct double2 { double x, y; };
struct float2 { float x, y; };

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
using hipStream_t = void*;
using hipEvent_t = void*;
constexpr unsigned hipStreamNonBlocking = 1, hipEventDisableTiming = 2, hipHostMallocDefault = 0;

inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline int streams_made = 0;
inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return ++streams_made, *s = std::malloc(1), hipSuccess; }
inline hipError_t hipStreamDestroy(hipStream_t s) { return std::free(s), hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = std::malloc(1), hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { return std::free(e), hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, std::size_t n, unsigned) { return *p = std::malloc(n), hipSuccess; }
inline hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
inline hipError_t hipMemcpyAsync(void* to, const void* from, std::size_t n, hipMemcpyKind, hipStream_t) {
  return std::memcpy(to, from, n), hipSuccess;
}
