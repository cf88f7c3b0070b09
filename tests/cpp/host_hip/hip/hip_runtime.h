// Host stand-in for the few HIP calls of akx_host.hpp and akx_download.hpp: the
// "device" is host memory and the test decides which calls fail.
#pragma once
#include <atomic>
#include <chrono>
#include <cstdlib>
#include <thread>

typedef int hipError_t;
typedef void *hipStream_t;
typedef int *hipEvent_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum { hipEventDisableTiming = 2, hipHostMallocCoherent = 0x40000000, hipMemcpyDeviceToHost = 2 };

namespace fake {
inline std::atomic<int> stream_waits{0};
inline std::atomic<int> records_to_fail{0}; // hipEventRecord calls of helpers that fail
inline std::atomic<int> event_waits{0};     // that have returned
inline std::atomic<int> slow_waits{0};      // ms of the test's thread's next one
inline thread_local bool helper = true;     // the test's own thread sets false
} // namespace fake

inline const char *hipGetErrorString(hipError_t) { return "a test's error"; }
inline hipError_t hipMalloc(void *p, size_t n) { return (*(void **)p = std::malloc(n)) ? 0 : 2; }
inline hipError_t hipFree(void *p) { return std::free(p), 0; }
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return (*p = std::malloc(n)) ? 0 : 2; }
inline hipError_t hipHostFree(void *p) { return std::free(p), 0; }
inline hipError_t hipSetDevice(int) { return 0; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = new int, 0; }
inline hipError_t hipEventDestroy(hipEvent_t e) { return delete e, 0; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) {
  return fake::helper && fake::records_to_fail.fetch_sub(1) > 0 ? hipErrorUnknown : hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t) {
  if (!fake::helper && fake::slow_waits.load()) // the stream has earlier work
    std::this_thread::sleep_for(std::chrono::milliseconds(fake::slow_waits.exchange(0)));
  return fake::event_waits.fetch_add(1), 0;
}
inline hipError_t hipStreamSynchronize(hipStream_t) { return fake::stream_waits.fetch_add(1), 0; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, int, hipStream_t);
