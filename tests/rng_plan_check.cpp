// Plans of draws read from standard input, one a line: "nseeds seed count ...";
// per plan the first and last streams' chunk states are printed.  Built with the
// host's sanitizers by test_cpu_rng_plan.py: the packed plan lies in an array
// of exactly rng_dev_bytes.
#include "../genetic_amd/csrc/rng_plan.h"
#include <cstdio>
#include <cstdlib>
#include <memory>

using namespace gic;

static void must(bool ok, const char *what) {
  if (ok) return;
  std::printf("FAILED %s\n", what);
  std::exit(1);
}

// the state at the start of chunk t, from the tables as the kernels form it
static void chunk_state(const RngDev &d, int kclog, long t, uint64_t *x, uint64_t &c) {
  uint64_t acc[9], r[9];
  memcpy(acc, d.y0.w, sizeof acc);
  for (int l = 0; l < RNG_DIGITS; ++l) {
    u576_mulmod(acc, &jump_table().w[((size_t(kclog) * RNG_DIGITS + l) * 64 + ((t >> (6 * l)) & 63)) * 9], r);
    memcpy(acc, r, sizeof acc);
  }
  decode_state(acc, x);
  c = 0;
  for (int i = 0; i < 12; ++i) {
    const int64_t v = int64_t(x[(i + 7) % 12]) - int64_t(x[i]) - int64_t(c);
    c = v < 0;
    x[i] = uint64_t(v) & MASK48;
  }
}

int main() {
  int n;
  while (std::scanf("%d", &n) == 1) {
    std::vector<RngStream> streams;
    size_t at = 0;
    for (int i = 0; i < n; ++i) {
      unsigned long seed;
      size_t count;
      must(std::scanf("%lu %zu", &seed, &count) == 2, "input");
      streams.push_back({seed, count, at});
      at += count;
    }
    RngPlan p;
    rng_plan(streams, p);
    const size_t bytes = rng_dev_bytes(p);
    std::unique_ptr<char[]> h(new char[bytes]);
    rng_dev_pack(p, h.get());
    must(rng_workspace_bytes(p) >= bytes + size_t(p.nseg) * (64 * (24 + 5) * 4 + 5 * 4 + 8) + 4, "workspace");
    const RngDev *d = reinterpret_cast<const RngDev *>(h.get());
    const uint32_t *of = reinterpret_cast<const uint32_t *>(h.get() + align256(n * sizeof(RngDev)));
    uint64_t seg = 0;
    std::printf("plan %d %ld\n", p.kclog, p.nseg);
    for (int i = 0; i < n; ++i) {
      must(d[i].seg0 == seg && d[i].nseg >= 1, "seg0");
      must(d[i].out0 == streams[i].out0 && d[i].total == streams[i].count, "targets");
      must(double(d[i].nseg) * 64 * p.ch() >= raw_needed(streams[i].count), "numbers");
      if (n > 1)
        for (uint64_t k = 0; k < d[i].nseg; ++k) must(of[seg + k] == uint32_t(i), "seg_stream");
      seg += d[i].nseg;
      if (i >= 40 && i < n - 12) continue;
      const long last = long(d[i].nseg) * 64 - 1;
      for (long t : {1l, last / 2, last}) {
        uint64_t x[12], c;
        chunk_state(d[i], p.kclog, t, x, c);
        std::printf("state %lu %ld %d", streams[i].seed, t << p.kclog, int(c));
        for (uint64_t w : x) std::printf(" %lu", (unsigned long)w);
        std::printf("\n");
      }
    }
    must(seg == uint64_t(p.nseg), "nseg");
  }
  return 0;
}
