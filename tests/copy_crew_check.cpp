// Arrays copied through slots as host_copy.h does it, the device's part played
// by whole words of memory: sizes and destination alignments from standard
// input, "bytes align ..." a line.  Built with the host's sanitizers by
// test_cpu_host_copy.py.
#include "../genetic_amd/csrc/copy_crew.h"
#include <cstdio>
#include <cstdlib>
#include <new>

using namespace gic;

constexpr size_t SLOT = 1 << 16;

// a thread that may not be had
static int refuse = 0;
struct Scarce : std::thread {
  template <class F> explicit Scarce(F f) : std::thread(start(std::move(f))) {}
  template <class F> static std::thread start(F f) {
    if (refuse & 1) {
      refuse >>= 1;
      throw std::bad_alloc();
    }
    refuse >>= 1;
    return std::thread(std::move(f));
  }
};

template <class Crew> static void copy(const std::vector<CopyPart> &parts) {
  const std::vector<CopyPart> pieces = copy_pieces(parts, SLOT);
  std::vector<uint64_t> slots(COPY_THREADS * SLOT / 8);
  Crew crew(pieces, (const char *)slots.data(), SLOT);
  copy_through(pieces, crew,
               [&](size_t k, const CopyPart &c) {
                 // (words of 16 or 4 bytes, as the kernel takes them)
                 const size_t w = c.bytes % 16 == 0 ? 16 : 4;
                 memcpy((char *)slots.data() + k * SLOT, c.src, c.bytes / w * w);
               },
               [](size_t) {});
}

int main() {
  char line[4096];
  while (std::fgets(line, sizeof line, stdin)) {
    std::vector<CopyPart> parts;
    std::vector<std::vector<char>> src, dst;
    char *s = line, *e;
    int mode = int(std::strtol(s, &s, 10));
    for (;;) {
      const size_t bytes = std::strtoul(s, &e, 10);
      if (e == s) break;
      const size_t align = std::strtoul(e, &s, 10);
      src.emplace_back(bytes);
      dst.emplace_back(bytes + 2 * SLOT, char(0x5a));
      for (size_t i = 0; i < bytes; ++i) src.back()[i] = char(i * 131 + i / 251);
      char *d = dst.back().data();
      d += (SLOT - reinterpret_cast<uintptr_t>(d) % SLOT) % SLOT + align;
      parts.push_back({d, src.back().data(), bytes});
    }
    refuse = mode;
    if (mode) copy<CopyCrew<Scarce>>(parts);
    else copy<CopyCrew<>>(parts);
    for (size_t p = 0; p < parts.size(); ++p)
      if (memcmp(parts[p].dst, parts[p].src, parts[p].bytes) != 0 ||
          ((const char *)parts[p].dst)[parts[p].bytes] != char(0x5a)) {
        std::printf("FAILED %s", line);
        return 1;
      }
  }
  return 0;
}
