// Staged transfers between device memory and a caller's pageable arrays.
//
// The runtime copies pageable memory through one staging buffer, transfer and host copy in turn: 18 GB/s
// here, and a host pass more wherever the caller's layout is not the device's.  Instead two slots
// of pinned memory alternate: a kernel writes a chunk, already in the caller's layout, over the bus
// into one slot while the host copies the other slot out, so that the host copy (32 GB/s into fresh pages)
// bounds it, no device memory is needed, and no host pass is spent on the layout.  Where pinned memory is
// refused, the chunks go through a slot on the device and the runtime's pageable copy.  Measured:
// 262144 particles' records (23 MB) 6.8 -> 1.05 ms, the potentials of two levels of 131072 nodes (6.3 MB)
// 1.17 -> 0.39 ms, 524k of a mesh's nodes by index 4.1 -> 1.4 ms.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <new>

#include "../../../include/mithra_gpu.h"

namespace mithra {

struct HostStage {
  char* base;       // two slots, pinned; kept by the owner for its next transfer
  size_t slot;      // bytes of one
  hipEvent_t ev[2];
  void* dev;        // a slot on the device, for transfers without pinned memory
  size_t dev_slot;
  bool used;        // a transfer has been made
};

// Chunks of a transfer of `total` bytes: four of them for overlap, but not so small that their launches
// show nor so large that the pinned memory does.
constexpr size_t kSlotLow = 512 << 10, kSlotHigh = 2 << 20;

constexpr long kAnyChunks = 1l << 62;

// An owner's first transfer goes without pinned memory up to this many bytes: allocating and freeing that takes
// more than a pageable copy of as much, and many owners are read once.  A fresh domain's first ten nodes by
// index, us: 50 through pinned slots, 41 so; a small network's first prediction (3 x 512 rows of 5): 74, 60.
constexpr size_t kOnce = 64 << 10;

inline void stage_free(HostStage* h) {
  if (h->base) (void)hipHostFree(h->base);
  for (auto& e : h->ev)
    if (e) (void)hipEventDestroy(e);
  if (h->dev) (void)hipFree(h->dev);
  *h = HostStage{};
}

// Whether this is the owner's first transfer, and one of `most` bytes or less.
inline bool stage_first(HostStage* h, size_t bytes, size_t most) {
  const bool first = !h->used;
  h->used = true;
  return first && bytes <= most;
}

// Room for two slots of `slot` bytes; E_NOMEM where the pinned memory is refused (the stage then has none).
// Nothing may be in flight on the stage's slots (the transfers leave none).
inline int stage_room(HostStage* h, size_t slot) {
  for (auto& e : h->ev)
    if (!e) {
      const hipError_t rc = hipEventCreateWithFlags(&e, hipEventDisableTiming);
      if (rc != hipSuccess) return MITHRA_E_HIP - (int)rc;
    }
  if (slot <= h->slot) return MITHRA_OK;
  if (h->base) (void)hipHostFree(h->base);
  h->base = nullptr;
  h->slot = 0;
  void* p = nullptr;
  if (hipHostMalloc(&p, 2 * slot, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();  // answered here: no later launch is to report it
    return MITHRA_E_NOMEM;
  }
  h->base = (char*)p;
  h->slot = slot;
  return MITHRA_OK;
}

// The transfer without pinned memory: chunk by chunk through a slot on the device, which the owner keeps, and a
// pageable one.
template <class List, class Put, class Take>
int stage_pageable(HostStage* h, hipStream_t s, long n, size_t unit, long chunks, size_t listed, List list, Put put,
                   Take take) {
  const size_t want = std::max(std::min(kSlotLow, (size_t)n * unit), (size_t)((n + chunks - 1) / chunks) * unit);
  if (h->dev_slot < want) {
    void* p = nullptr;
    size_t slot = want;
    while (slot > h->dev_slot && hipMalloc(&p, slot) != hipSuccess) {  // down to what it has, or a page
      (void)hipGetLastError();
      p = nullptr;
      slot = slot / 2 < std::max<size_t>(4096, unit) ? 0 : slot / 2;
    }
    if (p) {
      if (h->dev) (void)hipFree(h->dev);
      h->dev = p;
      h->dev_slot = slot;
    }
  }
  if (h->dev_slot < unit) return MITHRA_E_NOMEM;
  void* const dev = h->dev;
  const size_t slot = h->dev_slot;
  const long per = (long)(slot / unit);
  char* host = new (std::nothrow) char[std::min(slot, (size_t)n * unit)];
  hipError_t e = host ? hipSuccess : hipErrorOutOfMemory;
  for (long first = 0; first < n && e == hipSuccess; first += per) {
    const long m = std::min(per, n - first);
    if (listed) {
      list(first, m, host);
      e = hipMemcpyAsync(dev, host, listed * m, hipMemcpyHostToDevice, s);
    }
    if (e == hipSuccess) e = put(first, m, (char*)dev);
    if (e == hipSuccess) e = hipMemcpyAsync(host, dev, unit * m, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e == hipSuccess) take(first, m, (const char*)host);
  }
  const hipError_t done = hipStreamSynchronize(s);
  if (e == hipSuccess) e = done;
  delete[] host;
  return e == hipSuccess ? MITHRA_OK : e == hipErrorOutOfMemory ? MITHRA_E_NOMEM : MITHRA_E_HIP - (int)e;
}

// n items of `unit` bytes to the host: list(first, count, slot) fills the `listed` bytes an item at the
// slot's beginning that the kernel reads, put(first, count, slot) enqueues on `s` what writes a chunk into the slot,
// take(first, count, slot) copies it out on the host.  No more than `most` chunks, where the memory for
// larger ones can be had.  The stream is idle on return.
template <class List, class Put, class Take>
int stage_listed(HostStage* h, hipStream_t s, long n, size_t unit, long most, size_t listed, List list, Put put,
                 Take take) {
  if (n <= 0) {
    const hipError_t idle = hipStreamSynchronize(s);
    return idle == hipSuccess ? MITHRA_OK : MITHRA_E_HIP - (int)idle;
  }
  if (stage_first(h, (size_t)n * unit, kOnce)) {
    const int rc = stage_pageable(h, s, n, unit, most, listed, list, put, take);
    if (rc != MITHRA_E_NOMEM) return rc;
  }
  const size_t want = std::min(std::max((size_t)n * unit / 4, kSlotLow), kSlotHigh);
  const long per = std::min<long>(n, std::max<long>((n + most - 1) / most, (long)(want / unit)));
  const size_t bytes = ((size_t)per * unit + 255) / 256 * 256;
  if (const int rc = stage_room(h, bytes))
    return rc == MITHRA_E_NOMEM ? stage_pageable(h, s, n, unit, most, listed, list, put, take) : rc;
  const long chunks = (n + per - 1) / per;
  hipError_t e = hipSuccess;
  for (long c = 0; c <= chunks && e == hipSuccess; ++c) {
    if (c < chunks) {
      const long first = c * per, m = std::min(per, n - first);
      char* slot = h->base + (c & 1) * h->slot;
      if (listed) list(first, m, slot);
      e = put(first, m, slot);
      if (e == hipSuccess) e = hipEventRecord(h->ev[c & 1], s);
    }
    if (c > 0 && e == hipSuccess) {
      const long first = (c - 1) * per;
      e = hipEventSynchronize(h->ev[(c - 1) & 1]);
      if (e == hipSuccess) take(first, std::min(per, n - first), (const char*)h->base + ((c - 1) & 1) * h->slot);
    }
  }
  const hipError_t done = hipStreamSynchronize(s);
  if (e == hipSuccess) e = done;
  return e == hipSuccess ? MITHRA_OK : MITHRA_E_HIP - (int)e;
}

// The same without a list.
template <class Put, class Take>
int stage_chunks(HostStage* h, hipStream_t s, long n, size_t unit, Put put, Take take, long most = kAnyChunks) {
  return stage_listed(h, s, n, unit, most, 0, [](long, long, char*) {}, put, take);
}

}  // namespace mithra
