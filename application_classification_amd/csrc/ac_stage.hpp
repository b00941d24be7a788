// Copies between a caller's host memory and the device.
#pragma once

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstring>

#include "ac_host.hpp"

namespace ac {

// Pinned host memory through which results and inputs cross PCIe: slots used in turn, so that the copy engine fills (or
// drains) one while a thread drains (or fills) another.  A copy straight to or from pageable memory runs at 10 GB/s (67 MB
// of MU: 6.4 ms).  The link takes 57 GB/s; one thread writes a fresh host array, page faults included, at 12 GB/s (5.2
// ms), so results of 16 MB and more are written by four threads, each with slots of its own (2.4 ms; eight threads 3.3
// ms, and at 5-13 MB two or four gain nothing over one).
// Memory that HIP knows (page-locked, managed or the device's) is copied directly, at the link's rate: 50 MB of MU into
// page-locked memory 0.89 ms, through the slots 1.64 ms.
// Held by a context to its end: the small buffer from its first small input on, the slots from its first large transfer.
struct HostStage {
  static constexpr int kThreads = 4, kSlots = 2 * kThreads;
  static constexpr size_t kSlot = 1 << 20;
  static constexpr size_t kDirect = 2 << 20;   // below, a direct copy is as fast (1.5 MB: 93 against 97 us)
  static constexpr size_t kSmall = 256 << 10;  // inputs up to this (a pattern) are not waited for: one buffer, pinned
  // Pinned memory with an event for each slot; a copy into or out of a busy slot may be in flight.
  template <int N>
  struct Slots {
    char* p = nullptr;
    size_t slot = 0;
    hipEvent_t ev[N] = {};
    bool busy[N] = {};
    Slots() = default;
    Slots(const Slots&) = delete;
    Slots& operator=(const Slots&) = delete;
    ~Slots() {
      for (auto& e : ev)
        if (e) (void)hipEventDestroy(e);
      if (p) (void)hipHostFree(p);
    }
    // False where no pinned memory is to be had: the caller copies directly.
    bool ready(size_t size) {
      if (p) return true;
      bool ok = true;
      for (auto& e : ev)
        if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) e = nullptr, ok = false;
      slot = size;
      if (ok && hipHostMalloc((void**)&p, N * size, hipHostMallocDefault) == hipSuccess) return true;
      (void)hipGetLastError();
      p = nullptr;
      return false;
    }
    char* at(int s) { return p + s * slot; }
    hipError_t wait(int s) {
      if (!busy[s]) return hipSuccess;
      busy[s] = false;
      return hipEventSynchronize(ev[s]);
    }
    // The copy and its event.
    hipError_t copy(int s, void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t st) {
      hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, st);
      if (e == hipSuccess) e = hipEventRecord(ev[s], st);
      if (e == hipSuccess) busy[s] = true;
      return e;
    }
    hipError_t send(int s, void* dst, const void* src, size_t bytes, hipStream_t st) {
      const hipError_t e = wait(s);
      if (e != hipSuccess) return e;
      std::memcpy(at(s), src, bytes);
      return copy(s, dst, at(s), bytes, hipMemcpyHostToDevice, st);
    }
  };
  Slots<kSlots> large;
  Slots<1> small;

  static bool pageable(const void* p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
    (void)hipGetLastError();  // unknown to HIP
    return true;
  }
  static hipError_t direct(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t st) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, st);
    return e == hipSuccess ? hipStreamSynchronize(st) : e;
  }

  // Device to host, complete when it returns.
  hipError_t to_host(void* dst, const void* src, size_t bytes, hipStream_t st, int device) {
    if (bytes < kDirect || !pageable(dst) || !large.ready(kSlot)) return direct(dst, src, bytes, hipMemcpyDeviceToHost, st);
    const int nt = bytes < (16u << 20) ? 1 : kThreads;
    const size_t chunk = nt == 1 ? kSlot / 2 : kSlot;  // (one thread: a shorter pipeline to fill)
    const size_t n = (bytes + chunk - 1) / chunk;
    hipError_t err[kThreads] = {};
    // Item t takes chunks t, t + nt, ... through slots t, t + nt, ..., on whichever thread it falls to.
    parallel_items(nt, [&](int64_t t) {
      hipError_t e = hipSetDevice(device);
      const size_t per = (size_t)(kSlots / nt);
      auto slot = [&](size_t j) { return (int)t + (int)(j % per) * nt; };  // of the item's j-th chunk, t + j nt
      auto len = [&](size_t i) { return std::min(chunk, bytes - i * chunk); };
      auto start = [&](size_t j) {
        const size_t i = (size_t)t + j * nt;
        if (i >= n || e != hipSuccess) return;
        e = large.wait(slot(j));
        if (e == hipSuccess)
          e = large.copy(slot(j), large.at(slot(j)), static_cast<const char*>(src) + i * chunk, len(i),
                         hipMemcpyDeviceToHost, st);
      };
      for (size_t j = 0; j < per; ++j) start(j);
      for (size_t j = 0;; ++j) {
        const size_t i = (size_t)t + j * nt;
        if (i >= n || e != hipSuccess) break;
        e = large.wait(slot(j));
        if (e != hipSuccess) break;
        std::memcpy(static_cast<char*>(dst) + i * chunk, large.at(slot(j)), len(i));
        start(j + per);
      }
      err[t] = e;
    }, nt);
    for (int t = 0; t < nt; ++t)
      if (err[t] != hipSuccess) return err[t];
    return hipSuccess;
  }

  // Host to device: the source is read when it returns, the copy is ordered on the stream.
  hipError_t to_device(void* dst, const void* src, size_t bytes, hipStream_t st) {
    if (pageable(src)) {
      if (bytes <= kSmall && small.ready(kSmall)) return small.send(0, dst, src, bytes, st);
      if (bytes >= kDirect && large.ready(kSlot)) {
        hipError_t e = hipSuccess;
        for (size_t o = 0, i = 0; o < bytes && e == hipSuccess; o += kSlot, ++i)
          e = large.send((int)(i % kSlots), static_cast<char*>(dst) + o, static_cast<const char*>(src) + o,
                         std::min(kSlot, bytes - o), st);
        return e;
      }
    }
    return direct(dst, src, bytes, hipMemcpyHostToDevice, st);
  }
};

}  // namespace ac
