// The part of the HIP runtime that channel_amd/csrc/host_copy.hip uses, on the
// CPU: device memory is host memory, a stream does its work at once, a launch is a
// loop over its threads.  Counts what is asked for, and can run out of pinned memory.
#pragma once
#include <atomic>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>

#define __global__
#define __launch_bounds__(n)

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
enum hipMemoryType { hipMemoryTypeUnregistered, hipMemoryTypeHost };
enum hipStreamCaptureMode { hipStreamCaptureModeRelaxed };
struct hipPointerAttribute_t {
  hipMemoryType type;
};
typedef void *hipStream_t;
typedef int *hipEvent_t;
struct dim3 {
  unsigned x;
  dim3(unsigned x = 1) : x(x) {}
};
struct uint4 {
  unsigned x, y, z, w;
};
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

namespace fake {
inline std::atomic<int> launches{0}, plain{0}, pinned{0}, pin_calls{0}, events{0}, pin_limit{1 << 30}, waits{0};
inline std::atomic<const void *> pinned_host{nullptr};
inline thread_local dim3 block, thread, blocks;
}  // namespace fake
#define blockIdx fake::block
#define threadIdx fake::thread
#define gridDim fake::blocks

template <class F, class... A>
void hipLaunchKernelGGL(F f, dim3 g, dim3 b, int, hipStream_t, A... a) {
  fake::launches++;
  fake::blocks = g;
  for (fake::block.x = 0; fake::block.x < g.x; fake::block.x++)
    for (fake::thread.x = 0; fake::thread.x < b.x; fake::thread.x++) f(a...);
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return fake::waits++, hipSuccess; }
inline hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  fake::plain++;
  std::memcpy(d, s, n);
  return hipSuccess;
}
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  fake::pin_calls++;
  if (fake::pinned.fetch_add(1) >= fake::pin_limit) {
    fake::pinned--;
    return hipErrorOutOfMemory;
  }
  *p = std::malloc(n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void *p) { return fake::pinned--, std::free(p), hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return fake::events++, *e = new int(0), hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { return fake::events--, delete e, hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { return ++*e, hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
  a->type = p == fake::pinned_host ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return hipSuccess;
}
