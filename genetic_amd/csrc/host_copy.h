// Copies from the device into ordinary host memory.
//
// The runtime's copy into pageable memory passes through one staging buffer
// and one host thread, which also takes the page faults of a new array:
// 8 GB/s for 50 MB of particles, 12 GB/s for 400 MB.  Here the device fills
// pinned slots in turn, and a thread to each slot empties it into the caller's
// array.  A chunk is the part of the array in one 2 MB page: threads that
// share a page of a new array wait while one of them has it cleared (a 128^3
// Fourier realisation with 50 MB of particles: slots of 2 MB cut into eight
// pieces 3.5 ms, whole pages a thread 2.1 ms, 12 or 16 threads the same).  The
// slots are the context's and go with it; the
// threads last for one call.
#pragma once
#include "gic_common.h"
#include <sched.h>
#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <system_error>
#include <thread>
#include <vector>

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
  struct Part {
    void *dst;
    const void *src;
    size_t bytes;
  };
  // copies the parts (arrays of floats or doubles that work on st before
  // writes); returns when done
  void run(const std::vector<Part> &parts, hipStream_t st) {
    size_t total = 0;
    bool pageable = true;
    for (auto &p : parts) {
      total += p.bytes;
      pageable = pageable && is_pageable(p.dst);
    }
    // below a few slots there is little to overlap (4 MB: 0.5 ms either way)
    if (!pageable || total <= 2 * SLOT) {
      for (auto &p : parts)
        if (p.bytes) GIC_HIP(hipMemcpyAsync(p.dst, p.src, p.bytes, hipMemcpyDeviceToHost, st));
      GIC_HIP(hipStreamSynchronize(st));
      return;
    }
    std::vector<Part> chunks;
    for (auto &p : parts)
      for (size_t o = 0; o < p.bytes;) {
        const size_t page = SLOT - (reinterpret_cast<uintptr_t>(p.dst) + o) % SLOT, b = std::min(page, p.bytes - o);
        chunks.push_back({(char *)p.dst + o, (const char *)p.src + o, b});
        o += b;
      }
    if (!slots_) {
      for (auto &e : ready_)
        if (!e) GIC_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
      GIC_HIP(hipHostMalloc(&slots_, THREADS * SLOT, hipHostMallocDefault));
    }
    Crew crew(chunks, (const char *)slots_);
    const size_t n = chunks.size(), ns = size_t(crew.size());
    size_t sent = 0;
    auto send = [&] {
      const size_t k = sent % ns;
      const Part &c = chunks[sent];
      char *slot = (char *)slots_ + k * SLOT;
      if (c.bytes % 16 == 0 && reinterpret_cast<uintptr_t>(c.src) % 16 == 0)
        hipLaunchKernelGGL(k_to_slot<uint4>, dim3(256), dim3(256), 0, st, (const uint4 *)c.src, (uint4 *)slot,
                           c.bytes / 16);
      else   // whole floats or doubles
        hipLaunchKernelGGL(k_to_slot<uint32_t>, dim3(256), dim3(256), 0, st, (const uint32_t *)c.src, (uint32_t *)slot,
                           c.bytes / 4);
      GIC_HIP(hipGetLastError());
      GIC_HIP(hipEventRecord(ready_[k], st));
      ++sent;
    };
    try {
      for (size_t i = 0; i < n; ++i) {
        if (sent == i && i >= ns) crew.wait_emptied(i - ns);
        while (sent < n && (sent < ns || crew.emptied(sent - ns))) send();
        wait(ready_[i % ns]);
        crew.filled(i);
      }
      for (size_t i = n > ns ? n - ns : 0; i < n; ++i) crew.wait_emptied(i);
    } catch (...) {
      (void)hipStreamSynchronize(st);   // nothing may still write to the slots
      throw;                            // ~Crew ends the threads
    }
  }

 private:
  static constexpr size_t SLOT = size_t(2) << 20;   // a large page of the host
  static constexpr int THREADS = 8;
  void *slots_ = nullptr;
  hipEvent_t ready_[THREADS] = {};

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

  // The threads: thread t of n copies the chunks t, t + n, ... as they come
  // into slot t.  They poll, as the caller does, for the milliseconds that a
  // copy takes.
  class Crew {
   public:
    Crew(const std::vector<Part> &chunks, const char *slots) : chunks_(chunks), slots_(slots) {
      cpu_set_t set;
      if (sched_getaffinity(0, sizeof set, &set) == 0) n_ = std::max(1, std::min(n_, CPU_COUNT(&set)));
      for (auto &d : done_) d.store(0);
      for (int t = 0; t < n_; ++t) {
        try {
          threads_.emplace_back([this, t] { work(size_t(t)); });
        } catch (const std::system_error &) {
          own_ |= 1u << t;   // without its thread the caller copies the slot's chunks (filled)
        }
      }
    }
    ~Crew() {
      stop_.store(true);
      for (auto &t : threads_) t.join();
    }
    int size() const { return n_; }
    // chunk i, the next one, is in its slot
    void filled(size_t i) {
      filled_.store(i + 1, std::memory_order_release);
      if (own_ >> (i % size_t(n_)) & 1u) copy(i);
    }
    bool emptied(size_t i) const { return done_[i % size_t(n_)].load(std::memory_order_acquire) > i; }
    void wait_emptied(size_t i) const {
      while (!emptied(i)) std::this_thread::yield();
    }

   private:
    void copy(size_t i) {
      const size_t t = i % size_t(n_);
      std::memcpy(chunks_[i].dst, slots_ + t * SLOT, chunks_[i].bytes);
      done_[t].store(i + 1, std::memory_order_release);
    }
    void work(size_t t) {
      for (size_t i = t; i < chunks_.size(); i += size_t(n_)) {
        while (filled_.load(std::memory_order_acquire) <= i) {
          if (stop_.load()) return;
          std::this_thread::yield();
        }
        copy(i);
      }
    }
    const std::vector<Part> &chunks_;
    const char *slots_;
    int n_ = THREADS;
    unsigned own_ = 0;
    std::atomic<size_t> filled_{0}, done_[THREADS];
    std::atomic<bool> stop_{false};
    std::vector<std::thread> threads_;
  };
};

}  // namespace gic
