// host_copy.hpp -- transfers between device memory and pageable host buffers
// (fields, the closure's rows).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace chan {

// Pinned staging of one owner (a context or a model).  A slot is made by the first
// transfer that reaches it and kept until the owner goes: at most
// STAGE_SLOTS * STAGE_CHUNK bytes.  One transfer at a time, as the owner's calls are.
constexpr size_t STAGE_CHUNK = 2u << 20;
constexpr int STAGE_THREADS = 8, STAGE_SLOTS = 2 * STAGE_THREADS;
struct HostStage {
  char *buf[STAGE_SLOTS] = {};
  hipEvent_t ev[STAGE_SLOTS] = {};
  size_t direct = 0;  // bytes that went without it, those to the device at a sixth
  bool off = false;   // making or using the slots has failed
  void free();
};

// Copies `bytes` (a multiple of 4, device side aligned to 16) on the stream.  To the
// host it returns when they have arrived; to the device the stream may still be
// copying, and the caller waits for it before it returns to its own.  Large pageable buffers go through the stage in
// chunks, each of a few host threads filling or emptying its two slots while the
// others' are on the bus; smaller ones and pinned memory are copied directly.
hipError_t copy_to_host(HostStage &s, void *dst, const void *src, size_t bytes, hipStream_t st);
hipError_t copy_to_device(HostStage &s, void *dst, const void *src, size_t bytes, hipStream_t st);

}  // namespace chan
