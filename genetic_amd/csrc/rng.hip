// Parallel, bit-exact ranlxs2 + ziggurat Gaussians on gfx950.
//
// Replaces the serial draw loop of RandomFieldGenerator::drawRandomForSpecifiedGrid
// (genetIC/src/simulation/field/randomfieldgenerator.hpp:181-197), which calls
// gsl_ran_gaussian_ziggurat(ranlxs2, 1) once per cell in index order and
// continues the same stream across levels.
//
// ranlxs2 (Luescher's RANLUX at luxury p=397, GSL's 48-bit implementation)
// runs the subtract-with-borrow recurrence x_n = x_{n-5} - x_{n-12} - c_{n-1}
// (mod b = 2^48) and emits the 12 newest words after every 397 steps as 24
// 24-bit numbers (low half first, oldest word first).  The recurrence is an
// LCG in disguise: Z_n = sum_j a_j x_{n-12+j} + b c_{n-1} (mod m, m =
// b^12 - b^5 + 1, a_j = b^{j+1} - [j>=7] b^{j-6}) obeys Z_{n+1} = b^{-1} Z_n.
// So chunk t of the stream starts from a 576-bit modular product, is decoded
// to the 12-word state (the carry ambiguity of the decode disappears after
// 12 recurrence steps), and is then generated independently.
//
// gsl_ran_gaussian_ziggurat consumes 2 numbers per accepted iteration and
// 3 or 4 on the rare edge/tail tests, so the Gaussian index of a chunk is
// data dependent.  Pass 1 generates every chunk, parses it from the 4
// possible entry offsets (the parses merge after a few iterations) and scans
// the entry->(exit, count) maps across its wavefront; pass 2 scans the
// wavefronts' maps; pass 3 generates each chunk again, parses it from its
// true entry and writes the Gaussians to their cells.
//
// Generating twice is cheaper than keeping the numbers: a block of 24
// numbers takes about 3200 issue cycles of a wavefront (two instructions per
// recurrence step), writing and reading back its 64 x 24 words about 6100
// cycles of that SIMD's share of the memory bandwidth.
//
// One launch draws any number of independent streams (the shells of a
// Fourier-space draw, the realisations of a batch); every wavefront works on
// 64 consecutive chunks of one stream.
#include "rng.h"
#include "fft.h"
#include <cstring>
#include <cmath>
#include <mutex>
#include <string>

namespace gic {

#include "zig_tables.inc"

__constant__ double c_ytab[128];
__constant__ double c_wtab[128];
__constant__ unsigned int c_ktab[128];

// The generator's 12 words, oldest first, as 32 + 16 bits each: 48-bit words
// split this way need no masks (see swb_round)
struct Lux {
  uint32_t lo[12], hi[12];
  uint32_t c;   // borrow, 0 or 1
};

// One subtract-with-borrow step x[i] <- x[j] - x[i] - c in two instructions:
// the borrow stays in VCC, and the upper half is a 32-bit subtraction of
// zero-extended 16-bit values (SDWA), whose borrow is that of the 48-bit
// word and whose result is cut to 16 bits on the way out.  From the 64-bit
// C expression the compiler makes six.  gfx950 wants two wait states between
// a VALU write of VCC and its use as a carry, hence the s_nop.  Written for
// one wavefront the waits show; four wavefronts per SIMD fill them.
#define LUX_STEP(i, j)                                              \
  "v_subb_co_u32 %[l" #i "], vcc, %[l" #j "], %[l" #i "], vcc\n\t"  \
  "s_nop 1\n\t"                                                     \
  "v_subb_co_u32_sdwa %[h" #i "], vcc, %[h" #j "], %[h" #i "], vcc" \
  " dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:WORD_0 src1_sel:WORD_0\n\t" \
  "s_nop 1\n\t"
#define LUX_IO(x)                                                                                            \
  [l0] "+v"(x.lo[0]), [l1] "+v"(x.lo[1]), [l2] "+v"(x.lo[2]), [l3] "+v"(x.lo[3]), [l4] "+v"(x.lo[4]),        \
      [l5] "+v"(x.lo[5]), [l6] "+v"(x.lo[6]), [l7] "+v"(x.lo[7]), [l8] "+v"(x.lo[8]), [l9] "+v"(x.lo[9]),    \
      [l10] "+v"(x.lo[10]), [l11] "+v"(x.lo[11]), [h0] "+v"(x.hi[0]), [h1] "+v"(x.hi[1]), [h2] "+v"(x.hi[2]), \
      [h3] "+v"(x.hi[3]), [h4] "+v"(x.hi[4]), [h5] "+v"(x.hi[5]), [h6] "+v"(x.hi[6]), [h7] "+v"(x.hi[7]),    \
      [h8] "+v"(x.hi[8]), [h9] "+v"(x.hi[9]), [h10] "+v"(x.hi[10]), [h11] "+v"(x.hi[11]), [c] "+v"(x.c)
#define LUX_BEGIN "v_cmp_ne_u32 vcc, 0, %[c]\n\ts_nop 1\n\t"
#define LUX_END "v_cndmask_b32 %[c], 0, 1, vcc\n\ts_nop 1\n\t"

// 12 steps: every word is replaced once, x[0] stays the oldest
__device__ __forceinline__ void lux_round(Lux &x) {
  asm volatile(LUX_BEGIN LUX_STEP(0, 7) LUX_STEP(1, 8) LUX_STEP(2, 9) LUX_STEP(3, 10) LUX_STEP(4, 11) LUX_STEP(5, 0)
                   LUX_STEP(6, 1) LUX_STEP(7, 2) LUX_STEP(8, 3) LUX_STEP(9, 4) LUX_STEP(10, 5) LUX_STEP(11, 6) LUX_END
               : LUX_IO(x)
               :
               : "vcc");
}
__device__ __forceinline__ void lux_step0(Lux &x) {
  asm volatile(LUX_BEGIN LUX_STEP(0, 7) LUX_END : LUX_IO(x) : : "vcc");
}

// 397 steps (33 rounds of 12 plus one), the words rotated once at the end so
// that x[0] is the oldest again
__device__ __forceinline__ void lux_block(Lux &x) {
#pragma unroll 1
  for (int r = 0; r < 33; ++r) lux_round(x);
  lux_step0(x);
  uint32_t l = x.lo[0], h = x.hi[0];
#pragma unroll
  for (int i = 0; i < 11; ++i) {
    x.lo[i] = x.lo[i + 1];
    x.hi[i] = x.hi[i + 1];
  }
  x.lo[11] = l;
  x.hi[11] = h;
}
// the two 24-bit numbers of word k, in stream order
__device__ __forceinline__ uint32_t lux_first(const Lux &x, int k) { return x.lo[k] & 0xFFFFFFu; }
__device__ __forceinline__ uint32_t lux_second(const Lux &x, int k) {
  return __builtin_amdgcn_alignbit(x.hi[k], x.lo[k], 24);
}

// JumpTable's device copy
static __device__ uint64_t d_jump[RNG_KC_LOG][RNG_DIGITS][64][9];

__device__ __forceinline__ void lux_set(Lux &x, const uint64_t *w) {
#pragma unroll
  for (int i = 0; i < 12; ++i) {
    x.lo[i] = uint32_t(w[i]);
    x.hi[i] = uint32_t(w[i] >> 32);
  }
  x.c = 0;
}

__device__ __forceinline__ void chunk_start_state(const RngDev &p, int kclog, long t, Lux &x) {
  uint64_t acc[9];
  for (int i = 0; i < 9; ++i) acc[i] = p.y0.w[i];
#pragma unroll 1
  for (int l = 0; l < RNG_DIGITS; ++l) {
    long up = t >> (6 * l);
    if (l > 0 && up == 0) break;
    uint64_t r[9];
    u576_mulmod(acc, d_jump[kclog][l][up & 63], r);
    for (int i = 0; i < 9; ++i) acc[i] = r[i];
  }
  uint64_t w[12];
  decode_state(acc, w);
  lux_set(x, w);
  // 12 steps resolve the carry ambiguity and land on the chunk's start
  lux_round(x);
  if (t == 0) lux_set(x, p.seed_words);
}

// ---- ziggurat -------------------------------------------------------------------
// The ziggurat tables in LDS: the lookups are indexed by random bytes, so
// each lane reads a different entry (constant memory serves one address per
// wavefront)
struct ZigTabs {
  double y[128];
  double w[128];
  uint32_t k[128];
};
// all threads of the block call this before any of them returns
__device__ __forceinline__ void zig_tabs_load(ZigTabs &z) {
  for (int i = int(threadIdx.x); i < 128; i += int(blockDim.x)) {
    z.y[i] = c_ytab[i];
    z.w[i] = c_wtab[i];
    z.k[i] = c_ktab[i];
  }
  __syncthreads();
}

// A chunk is parsed window by window: with block q of the chunk come its 24
// numbers, and the iterations that may start at the 24 positions s = 0..23
// beginning 3 numbers before them can be finished (an iteration reads at
// most 4 numbers).  The 3 numbers before the first block are the newest ones
// of the chunk's start state.  So a chunk covers the starts from 3 numbers
// before its first block to 4 before its end, the parse enters it at s = 0,
// 1, 2 or 3, and the stream itself starts at s = 3 of chunk 0.
constexpr int ZIG_WIN = 27;   // numbers a window's iterations read
constexpr int ZIG_START = 3;

// An iteration of gsl_ran_gaussian_ziggurat starting at s reads number s
// (layer and sign) and s + 1 (abscissa); nearly always the abscissa lies in
// the layer's inner part and the iteration accepts with 2 numbers read.  Bit
// s of the result: it does.  No branches: the others are resolved after.
__device__ __forceinline__ uint32_t zig_fast(const uint32_t (&num)[ZIG_WIN], const ZigTabs &zt) {
  uint32_t f = 0;
#pragma unroll
  for (int s = 23; s >= 0; --s) {
    uint32_t d = num[s + 1] - zt.k[num[s] & 0x7Fu];   // both below 2^25: the sign bit is the comparison
    f = __builtin_amdgcn_alignbit(f, d, 31);
  }
  return f;
}

// the iteration's magnitude when it is accepted by the layer's own abscissa
__device__ __forceinline__ double zig_abscissa(uint32_t k1, uint32_t k2, const ZigTabs &zt) {
  return double(k2) * zt.w[k1 & 0x7Fu];
}

// An iteration that is not accepted at once: k1..k4 are the numbers from its
// start on.  Whether it accepts; x receives its magnitude.  It reads 4
// numbers in the tail (layer 127), otherwise 3.
__device__ __forceinline__ bool zig_slow(uint32_t k1, uint32_t k2, uint32_t k3, uint32_t k4, const ZigTabs &zt,
                                         double &x) {
  const double PARAM_R = 3.44428647676;
  uint32_t i = k1 & 0x7Fu;
  double y;
  if (i < 127) {
    x = zig_abscissa(k1, k2, zt);
    double y0 = zt.y[i], y1 = zt.y[i + 1];
    double U1 = k3 / 16777216.0;
    y = y1 + (y0 - y1) * U1;
  } else {
    double U1 = 1.0 - k3 / 16777216.0;
    double U2 = k4 / 16777216.0;
    x = PARAM_R - log(U1) / PARAM_R;
    y = exp(-PARAM_R * (x - 0.5 * PARAM_R)) * U2;
  }
  return y < exp(-0.5 * x * x);
}

// the window's numbers: the 3 kept from the block before, then this block's
__device__ __forceinline__ void zig_window(const Lux &x, uint32_t (&num)[ZIG_WIN]) {
  num[0] = num[24];
  num[1] = num[25];
  num[2] = num[26];
#pragma unroll
  for (int k = 0; k < 12; ++k) {
    num[3 + 2 * k] = lux_first(x, k);
    num[4 + 2 * k] = lux_second(x, k);
  }
}
// before the first block: the start state's newest numbers
__device__ __forceinline__ void zig_before(const Lux &x, uint32_t (&num)[ZIG_WIN]) {
  num[24] = lux_second(x, 10);
  num[25] = lux_first(x, 11);
  num[26] = lux_second(x, 11);
}
// length of the run of accepted 2-number iterations from s, in numbers; it
// stops at 24 or 25 at the latest
__device__ __forceinline__ int zig_run(uint32_t fast, int s) { return __ffs(int(~(fast >> s) & 0x55555555u)) - 1; }

constexpr int RNG_THREADS = 256;   // four wavefronts, each 64 consecutive chunks of one stream
constexpr int RNG_SEGS = RNG_THREADS / 64;

// entry offset -> exit offset (2 bits each in ex) and accepted count
struct Map4 {
  uint32_t ex;
  uint32_t cnt[4];
};
__device__ __forceinline__ uint32_t pick4(const uint32_t (&v)[4], uint32_t e) {
  // all four read first: selected by address they would live in memory
  const uint32_t a = v[0], b = v[1], c = v[2], d = v[3];
  const uint32_t lo = e & 1u ? b : a, hi = e & 1u ? d : c;
  return e & 2u ? hi : lo;
}
__device__ __forceinline__ Map4 compose(const Map4 &a, const Map4 &b) {   // a, then b
  Map4 r;
  r.ex = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    uint32_t m = (a.ex >> (2 * e)) & 3u;
    r.ex |= ((b.ex >> (2 * m)) & 3u) << (2 * e);
    r.cnt[e] = a.cnt[e] + pick4(b.cnt, m);
  }
  return r;
}
constexpr uint32_t MAP_ID = 0xE4u;   // e -> e
__device__ __forceinline__ Map4 load_map(const uint32_t *s, long t) {
  Map4 m;
  m.ex = s[t * 5];
  for (int e = 0; e < 4; ++e) m.cnt[e] = s[t * 5 + 1 + e];
  return m;
}
__device__ __forceinline__ void store_map(uint32_t *s, long t, const Map4 &m) {
  s[t * 5] = m.ex;
  for (int e = 0; e < 4; ++e) s[t * 5 + 1 + e] = m.cnt[e];
}
// Words 0..23 of chunk t's start state, 64 chunks side by side; the borrow
// rides in the free half of the first upper word
__device__ __forceinline__ size_t state_at(long seg, int k, int lane) { return (size_t(seg) * 24 + k) * 64 + lane; }

// Pass 1: per chunk the map from each of the four entry offsets, composed
// with those of the wavefront's earlier chunks (maps), per wavefront the
// whole (segmaps), and the chunk's start state for pass 3.  Bound by integer
// issue (the recurrence), four wavefronts per SIMD by registers.
// 1.1e9 Gaussians: 4.4 ms, where the 64-bit recurrence with an iteration at
// a time parsed from all entries, storing the numbers, took 10.6 ms; 20011
// Gaussians: 22 us against 125 us.
__global__ __launch_bounds__(RNG_THREADS) void k_rng_summary(const RngDev *__restrict__ streams,
                                                             const uint32_t *__restrict__ seg_stream, long nseg,
                                                             int kclog, uint32_t *__restrict__ state,
                                                             uint32_t *__restrict__ maps,
                                                             uint32_t *__restrict__ segmaps) {
  __shared__ uint32_t ring[ZIG_WIN * RNG_THREADS];   // a lane's numbers, for the slow iterations' indexed reads
  __shared__ ZigTabs zt;
  zig_tabs_load(zt);
  const int tid = threadIdx.x, lane = tid & 63;
  const long seg = long(blockIdx.x) * RNG_SEGS + __builtin_amdgcn_readfirstlane(tid >> 6);
  if (seg >= nseg) return;
  const RngDev &p = streams[seg_stream ? seg_stream[seg] : 0u];
  Lux x;
  chunk_start_state(p, kclog, (seg - long(p.seg0)) * 64 + lane, x);
#pragma unroll
  for (int k = 0; k < 12; ++k) {
    state[state_at(seg, k, lane)] = x.lo[k];
    state[state_at(seg, 12 + k, lane)] = k == 0 ? x.hi[k] | x.c << 16 : x.hi[k];
  }
  uint32_t num[ZIG_WIN];
  zig_before(x, num);
  int cur[4] = {0, 1, 2, 3};
  uint32_t cnt[4] = {0, 0, 0, 0};
  bool merged = false;   // one cursor is left: its acceptances count for all
  uint32_t shared_cnt = 0;
  const int kc = 1 << kclog;
#pragma unroll 1
  for (int q = 0; q < kc; ++q) {
    lux_block(x);
    zig_window(x, num);
#pragma unroll
    for (int s = 0; s < ZIG_WIN; ++s) ring[s * RNG_THREADS + tid] = num[s];
    const uint32_t fast = zig_fast(num, zt);
    // every start of the window that is not accepted at once, on a cursor's
    // way or not: about one in 42
    uint32_t acc = fast, four = 0;
    for (uint32_t z = ~fast & 0xFFFFFFu; z; z &= z - 1) {
      int s = __ffs(int(z)) - 1;
      const uint32_t *r = ring + s * RNG_THREADS + tid;
      uint32_t k1 = r[0];
      double v;
      if (zig_slow(k1, r[RNG_THREADS], r[2 * RNG_THREADS], r[3 * RNG_THREADS], zt, v)) acc |= 1u << s;
      if ((k1 & 0x7Fu) == 127u) four |= 1u << s;
    }
    auto walk = [&](int &pos) {
      uint32_t n = 0;
      int s = pos;
      while (s < 24) {
        int r = zig_run(fast, s);
        n += r >> 1;
        s += r;
        if (s >= 24) break;
        n += (acc >> s) & 1u;
        s += 3 + int((four >> s) & 1u);
      }
      pos = s - 24;
      return n;
    };
    if (merged) {
      shared_cnt += walk(cur[0]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) cnt[e] += walk(cur[e]);
      merged = cur[0] == cur[1] && cur[0] == cur[2] && cur[0] == cur[3];
    }
  }
  Map4 m;
  m.ex = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t own = uint32_t(cur[e]), one = uint32_t(cur[0]);
    m.ex |= (merged ? one : own) << (2 * e);
    m.cnt[e] = cnt[e] + shared_cnt;
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    Map4 a;
    a.ex = __shfl_up(m.ex, off);
#pragma unroll
    for (int e = 0; e < 4; ++e) a.cnt[e] = __shfl_up(m.cnt[e], off);
    if (lane >= off) m = compose(a, m);
  }
  if (lane == 63) store_map(segmaps, seg, m);
  Map4 before;
  before.ex = __shfl_up(m.ex, 1);
#pragma unroll
  for (int e = 0; e < 4; ++e) before.cnt[e] = __shfl_up(m.cnt[e], 1);
  if (lane == 0) before = Map4{MAP_ID, {0, 0, 0, 0}};
  store_map(maps, seg * 64 + lane, before);
}

// Pass 2: one workgroup per stream scans its wavefronts' maps; segstart[s] =
// (index of the stream's Gaussian the wavefront starts with << 2) | entry.
// *flag gets 1 if a stream holds fewer Gaussians than are wanted.
__global__ __launch_bounds__(1024) void k_rng_seg_scan(const RngDev *__restrict__ streams,
                                                       const uint32_t *__restrict__ segmaps,
                                                       uint64_t *__restrict__ segstart, uint32_t *__restrict__ flag,
                                                       int flag_stride) {
  __shared__ Map4 wave[16];
  const RngDev &p = streams[blockIdx.x];
  const long nseg = long(p.nseg), s0 = long(p.seg0);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const long per = (nseg + 1023) / 1024;
  const long b0 = min(nseg, tid * per), b1 = min(nseg, b0 + per);
  Map4 m{MAP_ID, {0, 0, 0, 0}};
  for (long t = b0; t < b1; ++t) m = compose(m, load_map(segmaps, s0 + t));
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    Map4 a;
    a.ex = __shfl_up(m.ex, off);
#pragma unroll
    for (int e = 0; e < 4; ++e) a.cnt[e] = __shfl_up(m.cnt[e], off);
    if (lane >= off) m = compose(a, m);
  }
  if (lane == 63) wave[w] = m;
  Map4 before;
  before.ex = __shfl_up(m.ex, 1);
#pragma unroll
  for (int e = 0; e < 4; ++e) before.cnt[e] = __shfl_up(m.cnt[e], 1);
  __syncthreads();
  uint32_t e = ZIG_START;
  uint64_t base = 0;
  for (int i = 0; i < w; ++i) {
    base += pick4(wave[i].cnt, e);
    e = (wave[i].ex >> (2 * e)) & 3u;
  }
  if (lane > 0) {
    base += pick4(before.cnt, e);
    e = (before.ex >> (2 * e)) & 3u;
  }
  for (long t = b0; t < b1; ++t) {
    segstart[s0 + t] = (base << 2) | uint64_t(e);
    Map4 a = load_map(segmaps, s0 + t);
    base += pick4(a.cnt, e);
    e = (a.ex >> (2 * e)) & 3u;
  }
  if (b1 == nseg && (b0 < b1 || nseg == 0) && base < p.total) flag[size_t(blockIdx.x) * flag_stride] = 1u;
}

struct LevelTargets {
  void *f[4];
  int n[4];        // grid size of a padded real field; 0 for a dense array
  size_t cum[4];   // cumulative Gaussian counts at the end of each target
  double scale;    // every value is stored as T(v * scale)
};

// Where a lane's next Gaussian goes: its cell and the cells left in its row
// (a dense target is one row)
template <typename T> struct CellCursor {
  T *p;
  uint64_t g;       // index of that Gaussian in the targets' order
  uint64_t end;     // end of the target it lies in
  uint32_t left;    // cells of the row from p on
  uint32_t n;
  __device__ __forceinline__ void seek(const LevelTargets &lt, uint64_t at) {
    g = at;
    int L = g < lt.cum[0] ? 0 : g < lt.cum[1] ? 1 : g < lt.cum[2] ? 2 : 3;
    size_t i = g - (L ? lt.cum[L - 1] : 0);
    end = lt.cum[L];
    n = uint32_t(lt.n[L]);
    if (n == 0) {
      p = reinterpret_cast<T *>(lt.f[L]) + i;
      left = uint32_t(min(uint64_t(0xFFFFFFFFu), end - g));
      return;
    }
    size_t row = i / n, z = i - row * n;
    p = reinterpret_cast<T *>(lt.f[L]) + row * (n + 2) + z;
    left = n - uint32_t(z);
  }
  // past m cells of the row (m <= left)
  __device__ __forceinline__ void step(const LevelTargets &lt, uint32_t m, uint64_t total) {
    p += m;
    g += m;
    left -= m;
    if (left == 0) {
      if (n != 0 && g < end) {
        p += 2;
        left = n;
      } else if (g < total) {
        seek(lt, g);
      }
    }
  }
};

// Pass 3 stages a lane's Gaussians in LDS and stores them four at a time as
// they complete (16 or 32 bytes a lane: a store of single values takes one
// address per lane, and four times as many).  A window adds at most 12 to
// the at most 3 left over.
constexpr int EMIT_STAGE = 16;
template <typename T> struct __attribute__((packed, aligned(sizeof(T)))) Four {
  T v[4];
};

// Pass 3: generate each chunk again, parse it from its true entry, write the
// Gaussians.  Bound by integer issue like pass 1, three wavefronts per SIMD
// (FP32) by LDS.  1.1e9 Gaussians in FP32: 5.4 ms, where reading stored
// numbers back, parsing an iteration at a time and storing runs
// cooperatively took 11.0 ms; 20011 Gaussians: 12 us against 56 us.
template <typename T>
__global__ __launch_bounds__(RNG_THREADS) void k_rng_emit(const RngDev *__restrict__ streams,
                                                          const uint32_t *__restrict__ seg_stream, long nseg,
                                                          int kclog, const uint32_t *__restrict__ state,
                                                          const uint32_t *__restrict__ maps,
                                                          const uint64_t *__restrict__ segstart, LevelTargets lt) {
  __shared__ uint32_t ring[ZIG_WIN * RNG_THREADS];
  __shared__ T stage[EMIT_STAGE * RNG_THREADS];
  __shared__ ZigTabs zt;
  zig_tabs_load(zt);
  const int tid = threadIdx.x, lane = tid & 63;
  const long seg = long(blockIdx.x) * RNG_SEGS + __builtin_amdgcn_readfirstlane(tid >> 6);
  if (seg >= nseg) return;
  const RngDev &p = streams[seg_stream ? seg_stream[seg] : 0u];
  const uint64_t ss = segstart[seg];
  Map4 before = load_map(maps, seg * 64 + lane);
  const uint32_t e = uint32_t(ss & 3u);
  // indexes in the targets' order from here on
  const uint64_t total = p.out0 + p.total;
  uint64_t g = p.out0 + (ss >> 2) + pick4(before.cnt, e);
  int pos = int((before.ex >> (2 * e)) & 3u);
  bool live = g < total;
  if (!__any(live)) return;
  Lux x;
#pragma unroll
  for (int k = 0; k < 12; ++k) {
    x.lo[k] = state[state_at(seg, k, lane)];
    x.hi[k] = state[state_at(seg, 12 + k, lane)];
  }
  x.c = x.hi[0] >> 16;
  x.hi[0] &= 0xFFFFu;
  CellCursor<T> cell;
  if (live) cell.seek(lt, g);
  uint32_t num[ZIG_WIN];
  zig_before(x, num);
  int head = 0, fill = 0;   // staged Gaussians: slots head .. head + fill - 1 (mod EMIT_STAGE)
  auto slot = [&](int i) -> T & { return stage[((head + i) & (EMIT_STAGE - 1)) * RNG_THREADS + tid]; };
  const int kc = 1 << kclog;
#pragma unroll 1
  for (int q = 0; q < kc; ++q) {
    if (!__any(live)) break;
    lux_block(x);
    zig_window(x, num);
#pragma unroll
    for (int s = 0; s < ZIG_WIN; ++s) ring[s * RNG_THREADS + tid] = num[s];
    const uint32_t fast = zig_fast(num, zt);
    // the accepted starts on the way (all), and those of them whose value is
    // the layer's abscissa (plain); the tail's values are staged here
    uint32_t all = 0, plain = 0;
    int s = live ? pos : 24;
    while (s < 24) {
      int r = zig_run(fast, s);
      uint32_t run = (0x555555u & ((1u << r) - 1u)) << s;
      all |= run;
      plain |= run;
      s += r;
      if (s >= 24) break;
      const uint32_t *k = ring + s * RNG_THREADS + tid;
      uint32_t k1 = k[0];
      bool tail = (k1 & 0x7Fu) == 127u;
      double v;
      if (zig_slow(k1, k[RNG_THREADS], k[2 * RNG_THREADS], k[3 * RNG_THREADS], zt, v)) {
        if (tail) slot(fill + __popc(all)) = T(((k1 & 0x80u) ? v : -v) * lt.scale);
        else plain |= 1u << s;
        all |= 1u << s;
      }
      s += tail ? 4 : 3;
    }
    pos = s - 24;
    // at most one of the starts 2k, 2k + 1 is on the way
#pragma unroll
    for (int k = 0; k < 12; ++k) {
      uint32_t b = (plain >> (2 * k)) & 3u;
      uint32_t k1 = b & 2u ? num[2 * k + 1] : num[2 * k], k2 = b & 2u ? num[2 * k + 2] : num[2 * k + 1];
      double v = zig_abscissa(k1, k2, zt);
      if (b) slot(fill + __popc(all & ((1u << (2 * k)) - 1u))) = T(((k1 & 0x80u) ? v : -v) * lt.scale);
    }
    fill += __popc(all);
    while (fill >= 4 && live) {
      T v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = slot(i);
      if (cell.left >= 4 && total - cell.g >= 4) {
        *reinterpret_cast<Four<T> *>(cell.p) = Four<T>{{v[0], v[1], v[2], v[3]}};
        cell.step(lt, 4, total);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (cell.g < total) {
            *cell.p = v[i];
            cell.step(lt, 1, total);
          }
      }
      head += 4;
      fill -= 4;
      live = cell.g < total;
    }
  }
  if (live)
    for (int i = 0; i < fill && cell.g < total; ++i) {
      *cell.p = slot(i);
      cell.step(lt, 1, total);
    }
}

// Raw 24-bit numbers in stream order (for bit-exactness checks).
__global__ __launch_bounds__(256) void k_rng_raw(RngDev p, int kclog, long nchunks, uint32_t *__restrict__ out,
                                                 size_t n) {
  long t = long(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= nchunks) return;
  Lux x;
  chunk_start_state(p, kclog, t, x);
  const int kc = 1 << kclog;
  size_t base = size_t(t) * (kc * 24);
  for (int q = 0; q < kc; ++q) {
    lux_block(x);
#pragma unroll
    for (int k = 0; k < 12; ++k) {
      size_t i = base + q * 24 + 2 * k;
      if (i < n) out[i] = lux_first(x, k);
      if (i + 1 < n) out[i + 1] = lux_second(x, k);
    }
  }
}

struct RngBufs {
  uint32_t *state, *maps, *segmaps;
  uint64_t *segstart;
  char *dev;
};
static RngBufs carve(const RngPlan &plan, void *ws, size_t bytes) {
  size_t ns = size_t(plan.nseg);
  char *p = (char *)ws;
  auto take = [&](size_t b) {
    char *r = p;
    p += align256(b);
    return r;
  };
  RngBufs r;
  r.state = (uint32_t *)take(ns * 64 * 24 * 4);
  r.maps = (uint32_t *)take(ns * 64 * 5 * 4);
  r.segmaps = (uint32_t *)take(ns * 5 * 4);
  r.segstart = (uint64_t *)take(ns * 8);
  r.dev = take(rng_dev_bytes(plan));
  if ((size_t)(p - (char *)ws) > bytes) throw std::runtime_error("RNG workspace too small");
  return r;
}

constexpr int RNG_MAX_DEVICES = 64;
static std::mutex g_tables_mu;
static bool g_tables_done[RNG_MAX_DEVICES];

// the ziggurat and jump tables into the current device's memory (each device
// has its own copy), once per device
static void upload_tables() {
  int dev = 0;
  GIC_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= RNG_MAX_DEVICES) throw std::runtime_error("RNG: device index out of range");
  std::lock_guard<std::mutex> g(g_tables_mu);
  if (g_tables_done[dev]) return;
  GIC_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_ytab), ZIG_YTAB, sizeof ZIG_YTAB));
  GIC_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_wtab), ZIG_WTAB, sizeof ZIG_WTAB));
  GIC_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_ktab), ZIG_KTAB, sizeof ZIG_KTAB));
  GIC_HIP(hipMemcpyToSymbol(HIP_SYMBOL(d_jump), jump_table().w.data(), sizeof(uint64_t) * jump_table().w.size()));
  g_tables_done[dev] = true;
}


// a stream's device copy, written by a kernel from its arguments
__global__ void k_rng_put_plan(RngDev d, RngDev *__restrict__ dst, uint32_t *__restrict__ flag) {
  const uint64_t *s = reinterpret_cast<const uint64_t *>(&d);
  uint64_t *o = reinterpret_cast<uint64_t *>(dst);
  for (int i = threadIdx.x; i < int(sizeof(RngDev) / 8); i += blockDim.x) o[i] = s[i];
  if (flag && threadIdx.x == 0) *flag = 0;
}
static_assert(sizeof(RngDev) % 8 == 0, "RngDev is copied as 64-bit words");

template <typename T>
static void draw_real_list(const RngPlan &plan, const RngLevelOut *levels, size_t nlev, void *ws, size_t ws_bytes,
                           hipStream_t st, TimingHook *hook, double scale, uint32_t *cover_flag, int flag_stride,
                           const void *dev_plan) {
  if (nlev < 1 || nlev > 4) throw std::runtime_error("real-space draw supports 1 to 4 levels");
  upload_tables();
  RngBufs b = carve(plan, ws, ws_bytes);
  const size_t n = plan.streams.size();
  LevelTargets lt;
  size_t acc = 0;
  for (size_t i = 0; i < 4; ++i) {
    lt.f[i] = i < nlev ? levels[i].field : nullptr;
    lt.n[i] = i < nlev ? levels[i].n : 0;
    if (i < nlev) acc += levels[i].count;
    lt.cum[i] = acc;
  }
  lt.scale = scale;
  for (auto &s : plan.streams)
    if (s.out0 > acc || s.count > acc - s.out0) throw std::runtime_error("RNG: a stream runs past the targets");
  // coverage: every stream must hold the Gaussians wanted of it; without a
  // caller's flag the check is this call's own, after the work
  uint32_t *flag = cover_flag;
  if (!flag) flag = (uint32_t *)(b.dev + rng_dev_bytes(plan));   // carve's slack
  const RngDev *pd = static_cast<const RngDev *>(dev_plan);
  std::vector<char> host;
  if (!pd) {
    pd = (const RngDev *)b.dev;
    if (n == 1) {
      hipLaunchKernelGGL(k_rng_put_plan, dim3(1), dim3(64), 0, st, to_dev(plan, 0), (RngDev *)b.dev,
                         cover_flag ? nullptr : flag);
      GIC_HIP(hipGetLastError());
    } else {
      // (host outlives the copy: without a caller's flag the call ends with a wait)
      if (cover_flag) throw std::runtime_error("internal error: several streams and a flag need a packed plan");
      host.resize(rng_dev_bytes(plan) + 4, 0);   // the flag follows
      rng_dev_pack(plan, host.data());
      GIC_HIP(hipMemcpyAsync(b.dev, host.data(), host.size(), hipMemcpyHostToDevice, st));
    }
  } else if (!cover_flag) {
    throw std::runtime_error("internal error: a draw from a packed plan needs a flag");
  }
  const uint32_t *of = n > 1 ? (const uint32_t *)((const char *)pd + align256(n * sizeof(RngDev))) : nullptr;
  const unsigned nblk = unsigned((plan.nseg + RNG_SEGS - 1) / RNG_SEGS);
  if (hook) hook->begin("rng_summary", st);
  hipLaunchKernelGGL(k_rng_summary, dim3(nblk), dim3(RNG_THREADS), 0, st, pd, of, plan.nseg, plan.kclog, b.state,
                     b.maps, b.segmaps);
  GIC_HIP(hipGetLastError());
  if (hook) hook->end("rng_summary", st);
  if (hook) hook->begin("rng_scan", st);
  hipLaunchKernelGGL(k_rng_seg_scan, dim3(unsigned(n)), dim3(1024), 0, st, pd, b.segmaps, b.segstart, flag,
                     cover_flag ? flag_stride : 0);
  GIC_HIP(hipGetLastError());
  if (hook) hook->end("rng_scan", st);
  if (hook) hook->begin("rng_emit", st);
  hipLaunchKernelGGL(k_rng_emit<T>, dim3(nblk), dim3(RNG_THREADS), 0, st, pd, of, plan.nseg, plan.kclog, b.state,
                     b.maps, b.segstart, lt);
  GIC_HIP(hipGetLastError());
  if (hook) hook->end("rng_emit", st);
  if (!cover_flag) {
    uint32_t few = 0;
    GIC_HIP(hipMemcpyAsync(&few, flag, 4, hipMemcpyDeviceToHost, st));
    GIC_HIP(hipStreamSynchronize(st));
    if (few) throw std::runtime_error("internal error: RNG plan produced too few Gaussians");
  }
}

template <typename T>
void rng_draw_real(const RngPlan &plan, const std::vector<RngLevelOut> &levels, void *ws, size_t ws_bytes,
                   hipStream_t st, TimingHook *hook, double scale, uint32_t *cover_flag, int flag_stride,
                   const void *dev_plan) {
  draw_real_list<T>(plan, levels.data(), levels.size(), ws, ws_bytes, st, hook, scale, cover_flag, flag_stride,
                    dev_plan);
}

template void rng_draw_real<float>(const RngPlan &, const std::vector<RngLevelOut> &, void *, size_t, hipStream_t,
                                   TimingHook *, double, uint32_t *, int, const void *);
template void rng_draw_real<double>(const RngPlan &, const std::vector<RngLevelOut> &, void *, size_t, hipStream_t,
                                    TimingHook *, double, uint32_t *, int, const void *);

// ---- draws with a fixed workspace ------------------------------------------------
// For callers that cannot allocate device memory: the draw's workspace (chunk
// states and maps, wavefront maps and starts, the plan) lives in this
// file-scope device array, one copy per GPU, held until the process ends.
// Its address on each device is looked up once (rng_scratch_setup, called by
// gic_create with the device current) and only that address is passed to
// kernels: the array's name in host code is a host-side stand-in.  The
// workspace needs no clearing (every pass writes what the next one reads).
// Calls that overlap on one GPU share the array and race.
constexpr size_t NOALLOC_SCRATCH_BYTES = size_t(13) << 20;
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[RNG_MAX_DEVICES];

void rng_scratch_setup(int device) {
  if (device < 0 || device >= RNG_MAX_DEVICES) throw std::runtime_error("RNG: device index out of range");
  upload_tables();
  std::lock_guard<std::mutex> g(g_scratch_mu);
  if (g_scratch_ptr[device]) return;
  void *p = nullptr;
  GIC_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  if (!p) throw std::runtime_error("RNG: no device address for the fixed workspace");
  g_scratch_ptr[device] = p;
}

size_t rng_noalloc_max_gaussians() { return size_t(1) << 20; }

void rng_gaussians_noalloc(int device, unsigned long seed, double *dev_out, size_t n, hipStream_t st) {
  if (n > rng_noalloc_max_gaussians())
    throw std::runtime_error("gic_gaussian_stream_noalloc: at most " + std::to_string(rng_noalloc_max_gaussians()) +
                             " Gaussians per call (the fixed workspace holds " +
                             std::to_string(NOALLOC_SCRATCH_BYTES >> 20) +
                             " MiB); gic_gaussian_stream draws longer streams");
  void *ws = nullptr;
  {
    std::lock_guard<std::mutex> g(g_scratch_mu);
    if (device >= 0 && device < RNG_MAX_DEVICES) ws = g_scratch_ptr[device];
  }
  if (!ws) throw std::runtime_error("gic_gaussian_stream_noalloc: the fixed workspace of this device is not set up");
  RngPlan plan;
  rng_plan(seed, n, plan);
  if (rng_workspace_bytes(plan) > NOALLOC_SCRATCH_BYTES)
    throw std::runtime_error("internal error: the fixed RNG workspace is too small for this draw");
  RngLevelOut out{dev_out, 0, n};
  draw_real_list<double>(plan, &out, 1, ws, NOALLOC_SCRATCH_BYTES, st, nullptr, 1.0, nullptr, 0, nullptr);
}

void rng_raw(const RngPlan &plan, uint32_t *d_out, size_t n, hipStream_t st) {
  upload_tables();
  size_t nc = (n + plan.ch() - 1) / plan.ch();
  if (nc > size_t(plan.nseg) * 64) throw std::runtime_error("rng_raw: plan too small");
  RngDev d = to_dev(plan, 0);
  hipLaunchKernelGGL(k_rng_raw, dim3((nc + 255) / 256), dim3(256), 0, st, d, plan.kclog, long(nc), d_out, n);
  GIC_HIP(hipGetLastError());
}

}  // namespace gic
