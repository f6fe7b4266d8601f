// host_copy.hip -- see host_copy.hpp.
//
// The runtime's own copy to a pageable buffer moves 10 GB/s: one thread empties a
// small staging buffer and takes the page faults of the fresh destination while
// the bus waits.  Eight threads with two slots each keep the bus busy: to the host
// 41 GB/s (1.35 GB, 129 -> 33 ms; 115 MB, 11.2 -> 2.9 ms), to the device 47 instead
// of 29 (46 -> 29 ms; 115 MB, 3.9 -> 2.6 ms).  A kernel moves the chunks: copy
// engines reached that rate in some processes and 18 GB/s in others.  Chunks of 1 MiB
// reach 40 GB/s either way, of 4 MiB 50 to the device and the same to the host, and
// take 1.5 ms more to pin.
#include "host_copy.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>
#include <vector>

namespace chan {

void HostStage::free() {
  for (auto &e : ev)
    if (e) (void)hipEventDestroy(e);
  for (char *b : buf)
    if (b) (void)hipHostFree(b);
  *this = HostStage();
}

namespace {

constexpr int MOVE_BLOCKS = 64;
// Where staging begins.  To the host it wins from the first size that is worth its
// threads (0.1 ms): 9 MB take 0.5 ms, 0.7 directly.  To the device the runtime
// pins the caller's pages and moves 29 GB/s, so there is less to win: 115 MB 2.6 ms,
// directly 3.9; 12 MB the same 0.5.
constexpr size_t TO_HOST_MIN = 8u << 20, TO_DEVICE_MIN = 96u << 20;

// An owner's first transfers go directly until what they lose by it (0.07 ms/MB to the
// host, 0.012 to the device, a sixth) is what pinning the slots costs (2 to 3 ms), so that
// a short-lived owner does not pay for slots it will not use: a first 15 MB to the host took
// 2.0 ms with the pinning, 1.4 without, a first 110 MB to the device (a closure forward
// of 599040 rows in all) 4.1 to 8.4 ms, 5.4 without.
bool staging_pays(HostStage &s, size_t bytes, bool to_host) {
  if (s.ev[0]) return true;
  s.direct += to_host ? bytes : bytes / 6;
  return s.direct > STAGE_SLOTS * STAGE_CHUNK;
}

// Makes slot i, in the thread that uses it: pinning all at once takes twice the time.
hipError_t make_slot(HostStage &s, int i) {
  if (s.ev[i]) return hipSuccess;
  // an allocation here must not end a capture that the caller has elsewhere
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  const bool relaxed = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
  hipError_t e = s.buf[i] ? hipSuccess : hipHostMalloc((void **)&s.buf[i], STAGE_CHUNK, hipHostMallocDefault);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&s.ev[i], hipEventDisableTiming);
  if (relaxed) (void)hipThreadExchangeStreamCaptureMode(&mode);
  return e;
}

// One chunk between device memory and a slot, a multiple of 4 bytes from 16-byte
// aligned addresses.
__global__ __launch_bounds__(256) void k_move(const uint4 *__restrict__ a, uint4 *__restrict__ b, unsigned words) {
  const unsigned t = blockIdx.x * 256 + threadIdx.x, n = words / 4;
  for (unsigned i = t; i < n; i += gridDim.x * 256) b[i] = a[i];
  if (t < words % 4) reinterpret_cast<unsigned *>(b + n)[t] = reinterpret_cast<const unsigned *>(a + n)[t];
}
hipError_t move(const void *a, void *b, size_t bytes, hipStream_t st) {
  hipLaunchKernelGGL(k_move, dim3(MOVE_BLOCKS), dim3(256), 0, st, static_cast<const uint4 *>(a), static_cast<uint4 *>(b),
                     (unsigned)(bytes / 4));
  return hipGetLastError();
}

// memory that the runtime does not know, i.e. neither pinned nor on a device
bool pageable(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

// Thread k of nt moves the chunks k, k + nt, ..., alternating between its slots.
template <bool TO_HOST>
hipError_t worker(HostStage &s, int dev, int k, int nt, char *host, char *device, size_t bytes, hipStream_t st) {
  hipError_t e = hipSetDevice(dev);
  const size_t n = (bytes + STAGE_CHUNK - 1) / STAGE_CHUNK;
  auto len = [&](size_t c) { return std::min(STAGE_CHUNK, bytes - c * STAGE_CHUNK); };
  auto slot = [&](size_t c) { return 2 * k + (int)(c / nt % 2); };
  auto stage = [&](size_t c) { return s.buf[slot(c)]; };
  if constexpr (TO_HOST) {
    auto start = [&](size_t c) {
      if (c >= n || e != hipSuccess) return;
      e = make_slot(s, slot(c));
      if (e == hipSuccess) e = move(device + c * STAGE_CHUNK, stage(c), len(c), st);
      if (e == hipSuccess) e = hipEventRecord(s.ev[slot(c)], st);
    };
    start(k);
    start((size_t)k + nt);
    for (size_t c = k; c < n && e == hipSuccess; c += nt) {
      e = hipEventSynchronize(s.ev[slot(c)]);
      if (e != hipSuccess) break;
      std::memcpy(host + c * STAGE_CHUNK, stage(c), len(c));
      start(c + 2 * (size_t)nt);
    }
  } else {
    for (size_t c = k; c < n && e == hipSuccess; c += nt) {
      e = c < 2 * (size_t)nt + k ? make_slot(s, slot(c)) : hipEventSynchronize(s.ev[slot(c)]);
      if (e != hipSuccess) break;
      std::memcpy(stage(c), host + c * STAGE_CHUNK, len(c));
      e = move(stage(c), device + c * STAGE_CHUNK, len(c), st);
      if (e == hipSuccess) e = hipEventRecord(s.ev[slot(c)], st);
    }
  }
  return e;
}

template <bool TO_HOST>
hipError_t staged(HostStage &s, char *host, char *device, size_t bytes, hipStream_t st) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const size_t n = (bytes + STAGE_CHUNK - 1) / STAGE_CHUNK;
  const int nt = (int)std::min<size_t>(STAGE_THREADS, n);
  std::atomic<int> first{(int)hipSuccess};
  auto job = [&](int k) {
    const hipError_t r = worker<TO_HOST>(s, dev, k, nt, host, device, bytes, st);
    int none = (int)hipSuccess;
    if (r != hipSuccess) first.compare_exchange_strong(none, (int)r);
  };
  std::vector<std::thread> threads;
  int started = 1;  // thread 0 is the caller
  try {
    threads.reserve(nt - 1);
    for (; started < nt; started++) threads.emplace_back(job, started);
  } catch (...) {  // no more threads: their chunks are the caller's
  }
  job(0);
  for (int k = started; k < nt; k++) job(k);
  for (auto &t : threads) t.join();
  const hipError_t end = hipStreamSynchronize(st);
  return first != (int)hipSuccess ? (hipError_t)first.load() : end;
}

template <bool TO_HOST>
hipError_t copy(HostStage &s, void *host, void *device, size_t bytes, hipStream_t st) {
  if (!s.off && bytes >= (TO_HOST ? TO_HOST_MIN : TO_DEVICE_MIN) && pageable(host) && staging_pays(s, bytes, TO_HOST)) {
    if (staged<TO_HOST>(s, static_cast<char *>(host), static_cast<char *>(device), bytes, st) == hipSuccess)
      return hipSuccess;
    // no pinned memory left, or a fault that the plain copy meets again: this owner
    // gives back what it has and does not try once more
    (void)hipGetLastError();
    s.free();
    s.off = true;
  }
  // to the device the caller's next wait serves as well: a wait of its own here took 7
  // of 42 us from a small closure forward
  if (!TO_HOST) return hipMemcpyAsync(device, host, bytes, hipMemcpyHostToDevice, st);
  const hipError_t e = hipMemcpyAsync(host, device, bytes, hipMemcpyDeviceToHost, st);
  return e != hipSuccess ? e : hipStreamSynchronize(st);
}

}  // namespace

hipError_t copy_to_host(HostStage &s, void *dst, const void *src, size_t bytes, hipStream_t st) {
  return copy<true>(s, dst, const_cast<void *>(src), bytes, st);
}
hipError_t copy_to_device(HostStage &s, void *dst, const void *src, size_t bytes, hipStream_t st) {
  return copy<false>(s, const_cast<void *>(src), dst, bytes, st);
}

}  // namespace chan
