// Host stand-ins for the HIP declarations that channel_flow_amd/csrc/hostcopy.hip
// uses, for its CPU test: device memory is host memory, every copy is done when it is
// asked for, and streams and events belong to the device that was current when they
// were made (an event is refused by another device's stream).
#pragma once
#include <cstdlib>
#include <cstring>

#define __device__
#define __host__
#define __forceinline__ inline

struct double2 { double x, y; };
struct float2 { float x, y; };

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorInvalidHandle = 400, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
using hipStream_t = int*;  // the device
using hipEvent_t = int*;
constexpr unsigned hipStreamNonBlocking = 1, hipEventDisableTiming = 2, hipHostMallocDefault = 0;

inline hipError_t hipGetLastError() { return hipSuccess; }
inline thread_local int current_device = 0;
inline hipError_t hipGetDevice(int* d) { return *d = current_device, hipSuccess; }
inline hipError_t hipSetDevice(int d) { return current_device = d, hipSuccess; }
inline int* of_device() {
  int* p = static_cast<int*>(std::malloc(sizeof(int)));
  *p = current_device;
  return p;
}
inline int streams_made = 0;
inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return ++streams_made, *s = of_device(), hipSuccess; }
inline hipError_t hipStreamDestroy(hipStream_t s) { return std::free(s), hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = of_device(), hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { return std::free(e), hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return *e == *s ? hipSuccess : hipErrorInvalidHandle; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, std::size_t n, unsigned) { return *p = std::malloc(n), hipSuccess; }
inline hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
inline hipError_t hipMemcpyAsync(void* to, const void* from, std::size_t n, hipMemcpyKind, hipStream_t) {
  return std::memcpy(to, from, n), hipSuccess;
}
