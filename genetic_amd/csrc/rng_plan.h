// The host's part of a draw: 576-bit arithmetic of the generator's jumps,
// the plan of a draw's streams and its copy for the device.  Plain C++ but for
// the functions that kernels share, so that it can be built without a device
// compiler.
#pragma once
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <stdexcept>
#include <vector>

#ifdef __HIPCC__
#define GIC_HD __host__ __device__
#else
#define GIC_HD
#endif

namespace gic {

// 576-bit numbers as 9 little-endian 64-bit limbs.
struct U576 {
  uint64_t w[9];
};

// One stream of a draw: its seed, the Gaussians wanted, and where the first
// of them goes, counted in the order of the draw's targets.
struct RngStream {
  unsigned long seed;
  size_t count;
  size_t out0;
};

// Host-side set-up of one real-space draw: its streams, the chunk length and
// how many wavefronts of 64 chunks each stream takes.
struct RngPlan {
  std::vector<RngStream> streams;
  int kclog = 6;                             // log2 of the ranlxs2 blocks (24 numbers) per chunk: 0..6
  int ch() const { return 24 << kclog; }     // raw numbers per chunk
  std::vector<long> seg0;                    // each stream's first wavefront
  long nseg = 0;                             // wavefronts in all
};

typedef unsigned __int128 u128;
static constexpr uint64_t MASK48 = (uint64_t(1) << 48) - 1;

// ---- 576-bit arithmetic mod m = 2^576 - 2^240 + 1 -------------------------
GIC_HD inline bool u576_geq_m(const uint64_t *a) {
  // m limbs: w0 = 1, w3 = 0xFFFF000000000000 (bits 240..255 clear... ) see below
  // m = 2^576 - 2^240 + 1: limbs 0..2: [1, 0, 0], limb 3: 2^64 - 2^48 (bits 48..63 set),
  // limbs 4..8: all ones.
  const uint64_t m[9] = {1, 0, 0, 0xFFFF000000000000ull, ~0ull, ~0ull, ~0ull, ~0ull, ~0ull};
  #pragma unroll
  for (int i = 8; i >= 0; --i) {
    if (a[i] != m[i]) return a[i] > m[i];
  }
  return true;
}
GIC_HD inline void u576_sub_m(uint64_t *a) {
  const uint64_t m[9] = {1, 0, 0, 0xFFFF000000000000ull, ~0ull, ~0ull, ~0ull, ~0ull, ~0ull};
  uint64_t borrow = 0;
  #pragma unroll
  for (int i = 0; i < 9; ++i) {
    u128 d = (u128)a[i] - m[i] - borrow;
    a[i] = (uint64_t)d;
    borrow = (uint64_t)(d >> 64) & 1;
  }
}

// s (nlimbs) <- L + H * 2^240 - H  with H given as hn limbs; result limbs
// written to out (length 14).  Requires H*2^240 >= H, true for any H >= 0.
template <int hn>
GIC_HD inline void fold(const uint64_t *L, const uint64_t *H, uint64_t *out) {
  uint64_t t[14];
  #pragma unroll
  for (int i = 0; i < 14; ++i) t[i] = 0;
  #pragma unroll
  for (int i = 0; i < 9; ++i) t[i] = L[i];
  // add H << 240 (= 3 limbs + 48 bits)
  u128 carry = 0;
  #pragma unroll
  for (int i = 0; i < 11; ++i) {
    uint64_t sh = 0;
    if (i < hn) sh |= H[i] << 48;
    if (i >= 1 && i - 1 < hn) sh |= H[i - 1] >> 16;
    u128 s = (u128)t[i + 3] + sh + carry;
    t[i + 3] = (uint64_t)s;
    carry = s >> 64;
  }
  // subtract H
  uint64_t borrow = 0;
  #pragma unroll
  for (int i = 0; i < 14; ++i) {
    uint64_t hv = i < hn ? H[i] : 0;
    u128 d = (u128)t[i] - hv - borrow;
    t[i] = (uint64_t)d;
    borrow = (uint64_t)(d >> 64) & 1;
  }
  #pragma unroll
  for (int i = 0; i < 14; ++i) out[i] = t[i];
}

GIC_HD inline void u576_mulmod(const uint64_t *a, const uint64_t *b, uint64_t *r) {
  uint64_t p[18];
  #pragma unroll
  for (int i = 0; i < 18; ++i) p[i] = 0;
  #pragma unroll
  for (int i = 0; i < 9; ++i) {
    uint64_t carry = 0;
    #pragma unroll
    for (int j = 0; j < 9; ++j) {
      u128 cur = (u128)a[i] * b[j] + p[i + j] + carry;
      p[i + j] = (uint64_t)cur;
      carry = (uint64_t)(cur >> 64);
    }
    p[i + 9] = carry;
  }
  uint64_t s[14];
  fold<9>(p, p + 9, s);          // < 2^576 + 2^816
  uint64_t s2[14];
  fold<5>(s, s + 9, s2);         // < 2^576 + 2^561
  #pragma unroll
  for (int i = 0; i < 9; ++i) r[i] = s2[i];
  // s2 fits in 9 limbs plus a possible carry bit in limb 9
  if (s2[9]) {
    // value >= 2^576 > m: subtract m once (2^576 - m = 2^240 - 1 < m)
    u576_sub_m(r);  // wraps limb 9 away
  }
  while (u576_geq_m(r)) u576_sub_m(r);
}

// 48-bit field at bit offset off of a little-endian limb array
GIC_HD inline uint64_t get48(const uint64_t *v, int off) {
  int li = off >> 6, bi = off & 63;
  uint64_t x = v[li] >> bi;
  if (bi > 16) x |= v[li + 1] << (64 - bi);
  return x & MASK48;
}
GIC_HD inline void put48(uint64_t *v, int off, uint64_t x) {
  int li = off >> 6, bi = off & 63;
  v[li] |= x << bi;
  if (bi > 16) v[li + 1] |= x >> (64 - bi);
}

// Decode V (the LCG state one step past the state S_n) into the 12 words of
// S_n with carry 0: V = A_low + (b^7 - 1) B + c, A_low the 7 oldest words,
// B the 5 newest.
GIC_HD inline void decode_state(const uint64_t *V, uint64_t *x) {
  // v0 = V mod 2^336, v1 = V >> 336
  uint64_t v0[7], v1[7];
  for (int i = 0; i < 7; ++i) v0[i] = v1[i] = 0;
  for (int i = 0; i < 5; ++i) v0[i] = V[i];
  v0[5] = V[5] & 0xFFFF;   // bits 320..335
  for (int i = 0; i < 4; ++i) v1[i] = (V[5 + i] >> 16) | (i + 6 < 9 ? V[6 + i] << 48 : 0);
  // v1 has at most 240 bits (4 limbs, top limb < 2^48)
  uint64_t s[7];
  u128 carry = 0;
  for (int i = 0; i < 7; ++i) {
    u128 t = (u128)v0[i] + v1[i] + carry;
    s[i] = (uint64_t)t;
    carry = t >> 64;
  }
  // compare s with D = 2^336 - 1 (limbs 0..4 all ones, limb 5 = 0xFFFF)
  bool ge = s[6] > 0 || s[5] > 0xFFFF ||
            (s[5] == 0xFFFF && s[4] == ~0ull && s[3] == ~0ull && s[2] == ~0ull && s[1] == ~0ull && s[0] == ~0ull);
  uint64_t B[7], R[7];
  for (int i = 0; i < 7; ++i) {
    B[i] = v1[i];
    R[i] = s[i];
  }
  if (ge) {
    // B += 1 ; R -= 2^336 - 1  (i.e. R = R - 2^336 + 1)
    u128 c = 1;
    for (int i = 0; i < 7; ++i) {
      u128 t = (u128)B[i] + c;
      B[i] = (uint64_t)t;
      c = t >> 64;
    }
    // R - 2^336 + 1: add 1 then clear bit 336 (R >= 2^336 - 1 so R+1 >= 2^336)
    c = 1;
    for (int i = 0; i < 7; ++i) {
      u128 t = (u128)R[i] + c;
      R[i] = (uint64_t)t;
      c = t >> 64;
    }
    // subtract 2^336 = limb 5 bit 16
    u128 d = (u128)R[5] - (uint64_t(1) << 16);
    R[5] = (uint64_t)d;
    if ((uint64_t)(d >> 64) & 1) R[6] -= 1;
  }
  // B >= 2^240 (only for V = m - 1): move one unit back into R
  if (B[3] >> 48) {
    uint64_t borrow = 1;
    for (int i = 0; i < 7; ++i) {
      u128 t = (u128)B[i] - borrow;
      B[i] = (uint64_t)t;
      borrow = (uint64_t)(t >> 64) & 1;
    }
    // R += 2^336 - 1
    u128 c = 0;
    const uint64_t D[7] = {~0ull, ~0ull, ~0ull, ~0ull, ~0ull, 0xFFFF, 0};
    for (int i = 0; i < 7; ++i) {
      u128 t = (u128)R[i] + D[i] + c;
      R[i] = (uint64_t)t;
      c = t >> 64;
    }
  }
  for (int j = 0; j < 7; ++j) x[j] = get48(R, 48 * j);
  for (int j = 0; j < 5; ++j) x[7 + j] = get48(B, 48 * j);
}

// The jump multipliers b^{-397 kc d 64^l} mod m for kc = 2^q blocks per
// chunk, digit d at base-64 position l of the chunk index: a chunk's start
// is at most RNG_DIGITS modular products from the stream's (a table of
// squarings takes one per bit set in any lane's index).  They depend on
// neither seed nor size.
constexpr int RNG_KC_LOG = 7;    // kc = 1 .. 64
constexpr int RNG_DIGITS = 5;    // 64^5 chunks a stream

// One stream of a draw
struct RngDev {
  uint64_t seed_words[12];
  U576 y0;          // the LCG state 12 steps before the stream's start
  uint64_t seg0;    // its first wavefront (64 chunks each)
  uint64_t nseg;
  uint64_t out0;    // where its first Gaussian goes, counted in the targets' order
  uint64_t total;   // Gaussians wanted
};

inline void seed_words(unsigned long s, uint64_t *xw) {
  // GSL ranlxs_set_lux / Luescher rlxs_init: bits of the seed drive a
  // 31-bit shift register clocked 48 times per word.
  if (s == 0) s = 1;
  long seed = (long)s;
  int i = (int)(seed & 0xFFFFFFFFUL);
  int xbit[31];
  for (int k = 0; k < 31; ++k) {
    xbit[k] = i % 2;
    i /= 2;
  }
  int ibit = 0, jbit = 18;
  for (int k = 0; k < 12; ++k) {
    int64_t xv = 0;
    for (int m = 1; m <= 48; ++m) {
      int64_t y = xbit[ibit];
      xv += xv + y;
      xbit[ibit] = (xbit[ibit] + xbit[jbit]) % 2;
      ibit = (ibit + 1) % 31;
      jbit = (jbit + 1) % 31;
    }
    xw[k] = (uint64_t)xv & MASK48;
  }
}

inline void u576_from_words(const uint64_t *x, int nw, uint64_t *out) {
  for (int i = 0; i < 9; ++i) out[i] = 0;
  for (int j = 0; j < nw; ++j) put48(out, 48 * j, x[j]);
}

inline void u576_powmod(const uint64_t *base, u128 e_lo, uint64_t *r) {
  uint64_t acc[9] = {1, 0, 0, 0, 0, 0, 0, 0, 0};
  uint64_t b[9];
  for (int i = 0; i < 9; ++i) b[i] = base[i];
  while (e_lo) {
    if (e_lo & 1) {
      uint64_t t[9];
      u576_mulmod(acc, b, t);
      memcpy(acc, t, sizeof acc);
    }
    uint64_t t[9];
    u576_mulmod(b, b, t);
    memcpy(b, t, sizeof b);
    e_lo >>= 1;
  }
  memcpy(r, acc, sizeof acc);
}

// The constants of the jumps: b^12 and the device table d_jump, computed
// once per process (about 2300 modular products)
struct JumpTable {
  uint64_t b12[9];
  std::vector<uint64_t> w;   // as d_jump
  JumpTable() : w(size_t(RNG_KC_LOG) * RNG_DIGITS * 64 * 9) {
    uint64_t one_b[9] = {0};
    put48(one_b, 48, 1);   // b
    u576_powmod(one_b, 12, b12);
    // b^{-1} = m - b^11 + b^4 (b^12 = b^5 - 1 mod m)
    uint64_t binv[9];
    const uint64_t m[9] = {1, 0, 0, 0xFFFF000000000000ull, ~0ull, ~0ull, ~0ull, ~0ull, ~0ull};
    uint64_t b11[9] = {0}, b4[9] = {0};
    put48(b11, 48 * 11, 1);
    put48(b4, 48 * 4, 1);
    uint64_t borrow = 0;
    for (int i = 0; i < 9; ++i) {
      u128 d = (u128)m[i] - b11[i] - borrow;
      binv[i] = (uint64_t)d;
      borrow = (uint64_t)(d >> 64) & 1;
    }
    u128 c = 0;
    for (int i = 0; i < 9; ++i) {
      u128 t = (u128)binv[i] + b4[i] + c;
      binv[i] = (uint64_t)t;
      c = t >> 64;
    }
    for (int q = 0; q < RNG_KC_LOG; ++q) {
      uint64_t step[9];   // one unit of the digit
      u576_powmod(binv, (u128)397 << q, step);
      for (int l = 0; l < RNG_DIGITS; ++l) {
        uint64_t v[9] = {1, 0, 0, 0, 0, 0, 0, 0, 0}, t[9];
        for (int d = 0; d < 64; ++d) {
          memcpy(&w[((size_t(q) * RNG_DIGITS + l) * 64 + d) * 9], v, sizeof v);
          u576_mulmod(v, step, t);
          memcpy(v, t, sizeof v);
        }
        memcpy(step, v, sizeof step);   // step^64
      }
    }
  }
};
inline const JumpTable &jump_table() {
  static const JumpTable t;
  return t;
}

// The LCG state 12 steps before the stream's start: b^12 V_0, V_0 the state
// one step past the seed (carry 0).  The device decodes V at 12 steps before
// a chunk's start and runs 12 steps.
inline void start_value(const uint64_t *words, U576 &y0) {
  // A = sum_j x_j b^j (12 words), B = sum_j x_{7+j} b^j (5 words), V_0 = A - B (mod m)
  uint64_t A[9], B[9], V[9];
  u576_from_words(words, 12, A);
  u576_from_words(words + 7, 5, B);
  while (u576_geq_m(A)) u576_sub_m(A);   // A < 2^576 but may exceed m
  uint64_t borrow = 0;
  for (int i = 0; i < 9; ++i) {
    u128 d = (u128)A[i] - B[i] - borrow;
    V[i] = (uint64_t)d;
    borrow = (uint64_t)(d >> 64) & 1;
  }
  if (borrow) {
    const uint64_t m[9] = {1, 0, 0, 0xFFFF000000000000ull, ~0ull, ~0ull, ~0ull, ~0ull, ~0ull};
    u128 c = 0;
    for (int i = 0; i < 9; ++i) {
      u128 t = (u128)V[i] + m[i] + c;
      V[i] = (uint64_t)t;
      c = t >> 64;
    }
  }
  u576_mulmod(jump_table().b12, V, y0.w);
}

// Raw numbers to have ready for n Gaussians: 2 per Gaussian plus rejections
// (~1.2% of iterations take 3-4 numbers and may repeat); 2.2x plus slack is
// never exceeded in practice and is checked after the scan.
inline double raw_needed(size_t n) { return 2.2 * double(n) + 4096.0; }

inline void rng_plan(const std::vector<RngStream> &streams, RngPlan &plan) {
  if (streams.empty()) throw std::runtime_error("RNG: no streams");
  plan.streams = streams;
  plan.seg0.clear();
  double need = 0;
  for (auto &s : streams) need += raw_needed(s.count);
  // Chunks of kc blocks: long chunks amortise the jump to each chunk's start
  // (about four blocks' time), and a small draw takes shorter ones so that
  // it still has about 64k chunks (a wavefront per SIMD) to run on.
  plan.kclog = RNG_KC_LOG - 1;
  while (plan.kclog > 0 && need / (24.0 * (1 << plan.kclog)) < 65536.0) --plan.kclog;
  plan.nseg = 0;
  for (auto &s : streams) {
    plan.seg0.push_back(plan.nseg);
    // (the jump tables reach a chunk from its own stream's start)
    const double chunks = raw_needed(s.count) / plan.ch() + 2;
    if (chunks > double(1L << (6 * RNG_DIGITS)) - 64) throw std::runtime_error("RNG: stream too long");
    plan.nseg += (long(chunks) + 63) / 64;
  }
}
inline void rng_plan(unsigned long seed, size_t n_gaussians, RngPlan &plan) {
  rng_plan(std::vector<RngStream>{{seed, n_gaussians, 0}}, plan);
}

inline size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

inline size_t rng_dev_bytes(const RngPlan &plan) {
  size_t n = plan.streams.size();
  return align256(n * sizeof(RngDev)) + (n > 1 ? align256(size_t(plan.nseg) * 4) : 0);
}
// Per chunk its start state (24 words) and map (5), per wavefront its map
// and start; then the streams, and for several of them each wavefront's.
inline size_t rng_workspace_bytes(const RngPlan &plan) {
  size_t ns = size_t(plan.nseg);
  return align256(ns * 64 * 24 * 4) + align256(ns * 64 * 5 * 4) + align256(ns * 5 * 4) + align256(ns * 8) +
         rng_dev_bytes(plan) + 256;
}
inline RngDev to_dev(const RngPlan &plan, size_t i) {
  RngDev d;
  seed_words(plan.streams[i].seed, d.seed_words);
  start_value(d.seed_words, d.y0);
  d.seg0 = uint64_t(plan.seg0[i]);
  d.nseg = uint64_t((i + 1 < plan.seg0.size() ? plan.seg0[i + 1] : plan.nseg) - plan.seg0[i]);
  d.out0 = plan.streams[i].out0;
  d.total = plan.streams[i].count;
  return d;
}
inline void rng_dev_pack(const RngPlan &plan, void *host_dst) {
  size_t n = plan.streams.size();
  RngDev *d = (RngDev *)host_dst;
  for (size_t i = 0; i < n; ++i) d[i] = to_dev(plan, i);
  if (n == 1) return;
  uint32_t *of = (uint32_t *)((char *)host_dst + align256(n * sizeof(RngDev)));
  for (size_t i = 0; i < n; ++i)
    for (uint64_t k = 0; k < d[i].nseg; ++k) of[d[i].seg0 + k] = uint32_t(i);
}

}  // namespace gic
