// The host's part of copies through pinned slots (host_copy.h): how arrays are
// cut into pieces, the threads that empty the slots, and the order of the
// work.  Plain C++, so that it can be tested without a device.
#pragma once
#include <sched.h>
#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <thread>
#include <vector>

namespace gic {

struct CopyPart {
  void *dst;
  const void *src;
  size_t bytes;
};

// The parts in pieces of at most slot bytes, each the part of its array in one
// page of slot bytes.  A piece starts a multiple of 16 bytes after its array
// does, whatever the destination's alignment (its last 15 bytes at most reach
// into the next page then): the slots are filled in words.
inline std::vector<CopyPart> copy_pieces(const std::vector<CopyPart> &parts, size_t slot) {
  std::vector<CopyPart> out;
  for (auto &p : parts)
    for (size_t o = 0; o < p.bytes;) {
      const size_t page = slot - (reinterpret_cast<uintptr_t>(p.dst) + o) % slot;
      const size_t b = std::min(page < 16 ? slot : page / 16 * 16, p.bytes - o);
      out.push_back({(char *)p.dst + o, (const char *)p.src + o, b});
      o += b;
    }
  return out;
}

// The threads: thread t of n copies the pieces t, t + n, ... as they come
// into slot t.  They poll, as the caller does, for the milliseconds that a
// copy takes.
constexpr int COPY_THREADS = 8;
template <class Thread = std::thread> class CopyCrew {
 public:
  CopyCrew(const std::vector<CopyPart> &pieces, const char *slots, size_t slot)
      : pieces_(pieces), slots_(slots), slot_(slot) {
    cpu_set_t set;
    if (sched_getaffinity(0, sizeof set, &set) == 0) n_ = std::max(1, std::min(n_, CPU_COUNT(&set)));
    for (auto &d : done_) d.store(0);
    threads_.reserve(size_t(n_));   // (once threads run, nothing here may throw)
    for (int t = 0; t < n_; ++t) {
      try {
        threads_.emplace_back([this, t] { work(size_t(t)); });
      } catch (...) {
        own_ |= 1u << t;   // without its thread the caller copies the slot's pieces (filled)
      }
    }
  }
  CopyCrew(const CopyCrew &) = delete;
  CopyCrew &operator=(const CopyCrew &) = delete;
  ~CopyCrew() {
    stop_.store(true);
    for (auto &t : threads_) t.join();
  }
  int size() const { return n_; }
  // piece i, the next one, is in its slot
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
    std::memcpy(pieces_[i].dst, slots_ + t * slot_, pieces_[i].bytes);
    done_[t].store(i + 1, std::memory_order_release);
  }
  void work(size_t t) {
    for (size_t i = t; i < pieces_.size(); i += size_t(n_)) {
      while (filled_.load(std::memory_order_acquire) <= i) {
        if (stop_.load()) return;
        std::this_thread::yield();
      }
      copy(i);
    }
  }
  const std::vector<CopyPart> &pieces_;
  const char *slots_;
  const size_t slot_;
  int n_ = COPY_THREADS;
  unsigned own_ = 0;
  std::atomic<size_t> filled_{0}, done_[COPY_THREADS];
  std::atomic<bool> stop_{false};
  std::vector<Thread> threads_;
};

// All pieces: send(k, piece) starts filling slot k, wait(k) returns when it is
// full; a slot is filled again only after its thread has emptied it.
template <class Crew, class Send, class Wait>
void copy_through(const std::vector<CopyPart> &pieces, Crew &crew, Send send, Wait wait) {
  const size_t n = pieces.size(), ns = size_t(crew.size());
  size_t sent = 0;
  for (size_t i = 0; i < n; ++i) {
    if (sent == i && i >= ns) crew.wait_emptied(i - ns);
    for (; sent < n && (sent < ns || crew.emptied(sent - ns)); ++sent) send(sent % ns, pieces[sent]);
    wait(i % ns);
    crew.filled(i);
  }
  for (size_t i = n > ns ? n - ns : 0; i < n; ++i) crew.wait_emptied(i);
}

}  // namespace gic
