// Copies from the device into ordinary host memory.
//
// The runtime's copy into pageable memory passes through one staging buffer
// and one host thread, which also takes the page faults of a new array:
// 8 GB/s for 50 MB of particles, 12 GB/s for 400 MB.  Here the device fills
// pinned slots in turn, and a thread to each slot empties it into the caller's
// array.  A piece is the part of the array in one 2 MB page: threads that
// share a page of a new array wait while one of them has it cleared (a 128^3
// Fourier realisation with 50 MB of particles: slots of 2 MB cut into eight
// pieces 3.5 ms, whole pages a thread 2.1 ms, 12 or 16 threads the same).  The
// slots are the context's and go with it; the threads last for one call.
#pragma once
#include "copy_crew.h"
#include "gic_common.h"

namespace gic {

// n words from device memory into a pinned slot.  (The runtime's copy call
// takes 30 us and more of host time for each slot, a launch 5.)
template <typename W> __global__ void k_to_slot(const W *__restrict__ src, W *__restrict__ dst, size_t n) {
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x)
    dst[i] = src[i];
}

class HostCopier {
 public:
  HostCopier() = default;
  HostCopier(const HostCopier &) = delete;
  HostCopier &operator=(const HostCopier &) = delete;
  ~HostCopier() {
    for (auto &e : ready_)
      if (e) (void)hipEventDestroy(e);
    if (slots_) (void)hipHostFree(slots_);
  }
  // copies the parts (arrays of floats or doubles that work on st before
  // writes); returns when done
  void run(const std::vector<CopyPart> &parts, hipStream_t st) {
    size_t total = 0;
    bool pageable = true;
    for (auto &p : parts) {
      total += p.bytes;
      pageable = pageable && is_pageable(p.dst);
    }
    // below a few slots there is little to overlap: 4.3 MB of particles 280 us
    // straight, 336 through the slots, 7.2 MB 434 and 425, 9.6 MB 559 and 455
    if (!pageable || total <= DIRECT) {
      for (auto &p : parts)
        if (p.bytes) GIC_HIP(hipMemcpyAsync(p.dst, p.src, p.bytes, hipMemcpyDeviceToHost, st));
      GIC_HIP(hipStreamSynchronize(st));
      return;
    }
    const std::vector<CopyPart> pieces = copy_pieces(parts, SLOT);
    if (!slots_) {
      for (auto &e : ready_)
        if (!e) GIC_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
      GIC_HIP(hipHostMalloc(&slots_, COPY_THREADS * SLOT, hipHostMallocDefault));
    }
    CopyCrew<> crew(pieces, (const char *)slots_, SLOT);
    auto send = [&](size_t k, const CopyPart &c) {
      char *slot = (char *)slots_ + k * SLOT;
      if (c.bytes % 16 == 0 && reinterpret_cast<uintptr_t>(c.src) % 16 == 0)
        hipLaunchKernelGGL(k_to_slot<uint4>, dim3(256), dim3(256), 0, st, (const uint4 *)c.src, (uint4 *)slot,
                           c.bytes / 16);
      else   // whole floats or doubles
        hipLaunchKernelGGL(k_to_slot<uint32_t>, dim3(256), dim3(256), 0, st, (const uint32_t *)c.src, (uint32_t *)slot,
                           c.bytes / 4);
      GIC_HIP(hipGetLastError());
      GIC_HIP(hipEventRecord(ready_[k], st));
    };
    try {
      copy_through(pieces, crew, send, [&](size_t k) { wait(ready_[k]); });
    } catch (...) {
      (void)hipStreamSynchronize(st);   // nothing may still write to the slots
      throw;                            // ~CopyCrew ends the threads
    }
  }

 private:
  static constexpr size_t SLOT = size_t(2) << 20;   // a large page of the host
  static constexpr size_t DIRECT = 7 * SLOT / 2;
  void *slots_ = nullptr;
  hipEvent_t ready_[COPY_THREADS] = {};

  // (a blocking wait wakes up 50 us late, as long as a slot takes to fill)
  static void wait(hipEvent_t e) {
    for (;;) {
      const hipError_t r = hipEventQuery(e);
      if (r == hipSuccess) return;
      if (r != hipErrorNotReady) GIC_HIP(r);
      (void)hipGetLastError();
      std::this_thread::yield();
    }
  }
  // memory that HIP knows (pinned, managed, the device's) takes the direct copy
  static bool is_pageable(const void *p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
      (void)hipGetLastError();
      return true;
    }
    return a.type == hipMemoryTypeUnregistered;
  }
};

}  // namespace gic
