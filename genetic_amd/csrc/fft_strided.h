#pragma once
// 3D real<->complex FFT for the padded FFTW layout, written for gfx950: the
// stages of a transform and the strided passes along y and x.
//
// Replaces the FFTW calls behind FieldFourierManager::performTransform
// (genetIC/src/tools/numerics/fourier.hpp:479-563): in-place r2c / c2r over
// [N][N][N+2] reals <-> [N][N][N/2+1] complex, forward sign e^{-2 pi i k.x/N}.
// The reference's pad/unpad copies (fourier.hpp:368-405) disappear because
// the real-space field stays padded in HBM.
//
// One kernel launch per axis:
//   z  : contiguous rows, N/2-point complex Stockham FFT of the packed
//        (even, odd) samples plus the r2c post-/c2r pre-twiddle (fft_rows.h);
//   y,x: strided lines, a tile of C adjacent kz columns is staged in LDS so
//        every global access is a C*sizeof(complex)-byte contiguous segment.
// Stages are radix-8 (plus one radix-4 or radix-16 stage) Stockham autosort steps;
// the first stage reads HBM, the last writes HBM, the rest go through LDS.
// Twiddles come from an N-entry table generated in FP64 on the host.
#include "gic_common.h"
#include "fft_api.h"
#include "fft_tiles.h"
#include <algorithm>
#include <vector>
#include <cmath>
#include <map>
#include <mutex>
#include <string>
#include <type_traits>

namespace gic {

constexpr int ilog2(int n) { return n <= 1 ? 0 : 1 + ilog2(n / 2); }

// WIDE: where the radix-8 stages leave a factor 2, the first stage takes 16
// points instead (one stage, and one pass through LDS, fewer).  It pays
// where the first stage has no |k|^2 operator (none, or a y pass's k_y / k_z
// factor); with a filter or table the 16 slots' factors take more registers
// than two blocks per CU allow.
template <int L, bool WIDE = false> struct RadixPlan {
  static constexpr int lg = ilog2(L);
  static constexpr int rem = lg % 3;
  static constexpr bool r16 = WIDE && rem == 1 && lg >= 4;
  static constexpr int nstages = r16 ? (lg - 4) / 3 + 1 : lg / 3 + (rem ? 1 : 0);
  static constexpr int radix(int s) { return s == 0 ? (r16 ? 16 : rem ? (1 << rem) : 8) : 8; }
  static constexpr int pbefore(int s) {
    int p = 1;
    for (int i = 0; i < s; ++i) p *= radix(i);
    return p;
  }
};

// multiply by i*DIR
template <int DIR, typename C> __device__ __forceinline__ C mul_i(C a) {
  return DIR > 0 ? C{-a.y, a.x} : C{a.y, -a.x};
}

template <int R, int DIR, typename T> struct Dft;

template <int DIR, typename T> struct Dft<1, DIR, T> {
  __device__ __forceinline__ static void run(cx<T> *) {}
};
template <int DIR, typename T> struct Dft<2, DIR, T> {
  __device__ __forceinline__ static void run(cx<T> *x) {
    cx<T> a = x[0];
    x[0] = cadd(a, x[1]);
    x[1] = csub(a, x[1]);
  }
};
template <int DIR, typename T> struct Dft<4, DIR, T> {
  __device__ __forceinline__ static void run(cx<T> *x) {
    cx<T> a0 = cadd(x[0], x[2]), a1 = csub(x[0], x[2]);
    cx<T> a2 = cadd(x[1], x[3]), a3 = mul_i<DIR>(csub(x[1], x[3]));
    x[0] = cadd(a0, a2);
    x[2] = csub(a0, a2);
    x[1] = cadd(a1, a3);
    x[3] = csub(a1, a3);
  }
};
template <int DIR, typename T> struct Dft<8, DIR, T> {
  __device__ __forceinline__ static void run(cx<T> *x) {
    cx<T> e[4] = {x[0], x[2], x[4], x[6]};
    cx<T> o[4] = {x[1], x[3], x[5], x[7]};
    Dft<4, DIR, T>::run(e);
    Dft<4, DIR, T>::run(o);
    const T h = T(0.70710678118654752440084436210484903928);
    // w8^1 = (1 + DIR i)/sqrt2, w8^2 = DIR i, w8^3 = (-1 + DIR i)/sqrt2
    cx<T> o1 = o[1], o3 = o[3];
    cx<T> t1 = cx<T>{h * (o1.x - DIR * o1.y), h * (o1.y + DIR * o1.x)};
    cx<T> t2 = mul_i<DIR>(o[2]);
    cx<T> t3 = cx<T>{h * (-o3.x - DIR * o3.y), h * (-o3.y + DIR * o3.x)};
    x[0] = cadd(e[0], o[0]);
    x[4] = csub(e[0], o[0]);
    x[1] = cadd(e[1], t1);
    x[5] = csub(e[1], t1);
    x[2] = cadd(e[2], t2);
    x[6] = csub(e[2], t2);
    x[3] = cadd(e[3], t3);
    x[7] = csub(e[3], t3);
  }
};

// 16 points as 4 x 4: DFT-4 of the four decimated columns, the W16^(jk)
// twiddles, DFT-4 of the rows; output k + 4m in natural order
template <int DIR, typename T> struct Dft<16, DIR, T> {
  __device__ __forceinline__ static cx<T> rot(cx<T> a, T c, T s) {   // a * (c + DIR s i)
    return cx<T>{a.x * c - T(DIR) * s * a.y, a.y * c + T(DIR) * s * a.x};
  }
  __device__ __forceinline__ static void run(cx<T> *x) {
    const T c1 = T(0.92387953251128675612818318939678828682), s1 = T(0.38268343236508977172845998403039886676);
    const T h = T(0.70710678118654752440084436210484903928);
    cx<T> a[4][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int m = 0; m < 4; ++m) a[j][m] = x[j + 4 * m];
      Dft<4, DIR, T>::run(a[j]);
    }
    a[1][1] = rot(a[1][1], c1, s1);    // W^1
    a[1][2] = rot(a[1][2], h, h);      // W^2
    a[1][3] = rot(a[1][3], s1, c1);    // W^3
    a[2][1] = rot(a[2][1], h, h);      // W^2
    a[2][2] = mul_i<DIR>(a[2][2]);     // W^4
    a[2][3] = rot(a[2][3], -h, h);     // W^6
    a[3][1] = rot(a[3][1], s1, c1);    // W^3
    a[3][2] = rot(a[3][2], -h, h);     // W^6
    a[3][3] = rot(a[3][3], -c1, -s1);  // W^9
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      cx<T> b[4] = {a[0][k], a[1][k], a[2][k], a[3][k]};
      Dft<4, DIR, T>::run(b);
#pragma unroll
      for (int m = 0; m < 4; ++m) x[k + 4 * m] = b[m];
    }
  }
};

// XCD-aware tile order: consecutive tiles land on the same XCD (the
// dispatcher places workgroup b on XCD b % 8), so tiles that share 128-byte
// lines are served by one L2.
__device__ __forceinline__ int xcd_tile(int b, int nblk) {
  if ((nblk & 7) != 0) return b;
  return (b & 7) * (nblk >> 3) + (b >> 3);
}

// One Stockham stage.  Butterfly q is mapped to (line, i): LINE_FAST puts
// adjacent q on adjacent lines (strided passes), otherwise on adjacent points.
// An operator on the first stage's loads has a real factor per (line, point)
// that depends only on the mode (factor) and combines it with the loaded
// value (apply).
struct NoOp {};

template <typename T, int L, int NL, int THREADS, int S, int DIR, bool LINE_FAST, bool WIDE, class Ld, class St,
          class Op = NoOp>
__device__ __forceinline__ void stage(const cx<T> *__restrict__ tw, int twmul, Ld ld, St st, bool sync_between,
                                      Op op = Op()) {
  using P = RadixPlan<L, WIDE>;
  constexpr int R = P::radix(S);
  constexpr int p = P::pbefore(S);
  constexpr int NB = NL * (L / R);
  constexpr int PER = (NB + THREADS - 1) / THREADS;
  const int tid = threadIdx.x;
  cx<T> v[PER][R];
#pragma unroll
  for (int b = 0; b < PER; ++b) {
    int q = tid + b * THREADS;
    if (NB % THREADS == 0 || q < NB) {
      int line = LINE_FAST ? q % NL : q / (L / R);
      int i = LINE_FAST ? q / NL : q % (L / R);
#pragma unroll
      for (int r = 0; r < R; ++r) v[b][r] = ld(line, i + r * (L / R));
    }
  }
  // operators: every factor is formed while the loads are in flight (they
  // depend only on the mode), and only then applied to the loaded values
  if constexpr (!std::is_same<Op, NoOp>::value) {
    // all slots' factors in one call; an idle slot (no butterfly) takes
    // line 0 and point r L/R, inside the tile, and its factor is unused
    int ln[PER * R], pp[PER * R];
#pragma unroll
    for (int b = 0; b < PER; ++b) {
      int q = tid + b * THREADS;
      bool has = NB % THREADS == 0 || q < NB;
      int line = has ? (LINE_FAST ? q % NL : q / (L / R)) : 0;
      int i = has ? (LINE_FAST ? q / NL : q % (L / R)) : 0;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        ln[b * R + r] = line;
        pp[b * R + r] = i + r * (L / R);
      }
    }
    // in groups of four slots: enough chains to interleave, few enough
    // registers for two blocks per CU.  Each group is applied as soon as it
    // is formed, so that only its four factors are held and it waits only on
    // its own loads (the later slots' loads stay in flight)
    constexpr int NSL = PER * R, CH = NSL % 4 == 0 ? 4 : NSL;
#pragma unroll
    for (int c0 = 0; c0 < NSL; c0 += CH) {
      int lc[CH], pc[CH];
      T fc[CH];
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        lc[j] = ln[c0 + j];
        pc[j] = pp[c0 + j];
      }
      op.factors(lc, pc, fc);
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        const int b = (c0 + j) / R, r = (c0 + j) % R;
        if (NB % THREADS == 0 || tid + b * THREADS < NB) v[b][r] = op.apply(v[b][r], fc[j]);
      }
    }
  }
  if (sync_between) __syncthreads();
#pragma unroll
  for (int b = 0; b < PER; ++b) {
    int q = tid + b * THREADS;
    if (NB % THREADS == 0 || q < NB) {
      int line = LINE_FAST ? q % NL : q / (L / R);
      int i = LINE_FAST ? q / NL : q % (L / R);
      int k = i % p;
      if (p > 1) {
#pragma unroll
        for (int r = 1; r < R; ++r) {
          cx<T> w = tw[(r * k * (L / (p * R))) * twmul];
          if (DIR > 0) w.y = -w.y;
          v[b][r] = cmul(v[b][r], w);
        }
      }
      Dft<R, DIR, T>::run(v[b]);
      int j = (i - k) * R + k;
#pragma unroll
      for (int s = 0; s < R; ++s) st(line, j + s * p, v[b][s]);
    }
  }
}

// Run all stages: stage 0 loads with gld, the last stage stores with gst, the
// others go through LDS laid out by lidx(line, point).  GLD_LDS / GST_LDS say
// whether gld / gst themselves touch LDS, in which case the stage must put a
// barrier between its loads and its stores.
template <typename T, int L, int NL, int THREADS, int DIR, bool LINE_FAST, bool GLD_LDS, bool GST_LDS, int S,
          bool WIDE, class GLd, class GSt, class LIdx, class Op = NoOp>
__device__ __forceinline__ void run_stages(cx<T> *lds, const cx<T> *tw, int twmul, GLd gld, GSt gst, LIdx lidx,
                                           Op op = Op()) {
  using P = RadixPlan<L, WIDE>;
  constexpr int NS = P::nstages;
  auto lds_ld = [&](int line, int pt) { return lds[lidx(line, pt)]; };
  auto lds_st = [&](int line, int pt, cx<T> v) { lds[lidx(line, pt)] = v; };
  if constexpr (NS == 1) {
    stage<T, L, NL, THREADS, 0, DIR, LINE_FAST, WIDE>(tw, twmul, gld, gst, GLD_LDS && GST_LDS, op);
  } else if constexpr (S == 0) {
    stage<T, L, NL, THREADS, 0, DIR, LINE_FAST, WIDE>(tw, twmul, gld, lds_st, GLD_LDS, op);
    __syncthreads();
    run_stages<T, L, NL, THREADS, DIR, LINE_FAST, GLD_LDS, GST_LDS, 1, WIDE>(lds, tw, twmul, gld, gst, lidx);
  } else if constexpr (S == NS - 1) {
    stage<T, L, NL, THREADS, S, DIR, LINE_FAST, WIDE>(tw, twmul, lds_ld, gst, GST_LDS);
  } else {
    stage<T, L, NL, THREADS, S, DIR, LINE_FAST, WIDE>(tw, twmul, lds_ld, lds_st, true);
    __syncthreads();
    run_stages<T, L, NL, THREADS, DIR, LINE_FAST, GLD_LDS, GST_LDS, S + 1, WIDE>(lds, tw, twmul, gld, gst, lidx);
  }
}

// ---- strided c2c pass (y or x) ------------------------------------------------
// Lines of length L along one axis; a tile holds C adjacent kz columns of one
// `outer` index.  Input and output may differ (out-of-place) and the output
// may keep only a window of the line (pruned inverse transforms, where the
// line's output is a spatial coordinate).  Optional k-space operators:
//   PRE  (inverse x pass, input indexed by kx=pt, ky=outer, kz=col):
//        PRE_TABLE: v *= tab[kx^2+ky^2+kz^2]
//   POST (forward x pass, output indexed by kx=pt, ky=outer, kz=col):
//        POST_TABLE: v *= tab[kx^2+ky^2+kz^2]
//        POST_AUX:   out = tab[|k|^2] aux + v, aux a spectrum laid out as out
enum { PRE_NONE = FFT_PRE_NONE, PRE_TABLE = FFT_PRE_TABLE };
enum { POST_NONE = 0, POST_TABLE = 1, POST_AUX = 2 };

// FilterInline prepared for single precision on the host: per filter the
// cut kc and 1 / (0.1 kc), the scale, kMin and 1 / kMin^2
struct FilterF {
  int nf, zero, over_k2;
  int kind[8];
  float kc[8], inv_w[8];
  float scale, kmin, inv_kmin2;
};

template <typename T> struct StridedArgs {
  const cx<T> *in;
  cx<T> *out;
  long in_ls, in_os, out_ls, out_os;
  int ncol, nkzb;
  int n;            // full grid size, for signed wavenumbers
  const T *tab;     // |k|^2-indexed factor table (or nullptr)
  int win0, wlen;   // output keeps line points (pt - win0) mod n < wlen
  T scale;
  int accum;        // POST ops: add to the output instead of storing
  const cx<T> *aux;        // POST_AUX: the spectrum added after its table
  double inv_k2, kmin_d;   // PRE ops without a table: factor inv_k2 / (|k|^2 kmin_d^2)
  FilterInline fil;        // FP32: the table's filter product formed in the pass (fil.nf >= 0)
  int in_win0, in_wlen;   // if 0 < in_wlen < n: the input holds only line points (pt - in_win0) mod n < in_wlen,
                          // stored at index (pt - in_win0) mod n
  FilterF ff;             // FP32: fil in single precision with its divisions turned into products (set by strided())
  float inv_k2_f;         // FP32: inv_k2 / kMin^2 (set by strided())
  int nbatch, nouter;     // nbatch > 1: that many fields, in_bs / out_bs elements apart, nouter outer lines each
  long in_bs, out_bs;
  const int *in_win0_b;   // if given: in_win0 of each field of the batch (device array)
};

__device__ __forceinline__ int signed_k(int i, int n) { return i > n / 2 ? i - n : i; }

// The factor of FilterInline at |k|^2 = ksq (filter_table's product) in
// single precision, with hardware reciprocal and square root (1 ulp each)
// and the host's reciprocals: no division per mode.
__device__ __forceinline__ float filter_fast_f(const FilterF &F, int ksq) {
  if (F.zero) return 0.f;
  float fk = float(ksq);
  float k = __builtin_amdgcn_sqrtf(fk) * F.kmin;
  float v = F.scale;
  // a fixed bound with a uniform exit: the parameters are indexed by
  // constants and stay in scalar registers
#pragma unroll
  for (int i = 0; i < FILTER_INLINE_MAX; ++i) {
    if (i >= F.nf) break;
    float lp = __builtin_amdgcn_rcpf(1.f + __expf((k - F.kc[i]) * F.inv_w[i]));
    v *= F.kind[i] == 0 ? lp : F.kind[i] == 1 ? __builtin_amdgcn_sqrtf(fmaxf(1.f - lp * lp, 0.f)) : 1.f - lp;
  }
  if (F.over_k2) v = ksq == 0 ? 0.f : v * F.inv_kmin2 * __builtin_amdgcn_rcpf(fk);
  return v;
}
// filter_fast_f for NS values of |k|^2 at once, one factor at a time across
// them: the parameter tests are taken once for all values and their
// exp / rcp / sqrt chains interleave.  The same arithmetic per value.
template <int NS>
__device__ __forceinline__ void filter_fast_f_n(const FilterF &F, const int (&ksq)[NS], float (&out)[NS]) {
  if (F.zero) {
#pragma unroll
    for (int s = 0; s < NS; ++s) out[s] = 0.f;
    return;
  }
  float k[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    k[s] = __builtin_amdgcn_sqrtf(float(ksq[s])) * F.kmin;
    out[s] = F.scale;
  }
#pragma unroll
  for (int i = 0; i < FILTER_INLINE_MAX; ++i) {
    if (i >= F.nf) break;
    const float kc = F.kc[i], iw = F.inv_w[i];
    const int kind = F.kind[i];
    float lp[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) lp[s] = __builtin_amdgcn_rcpf(1.f + __expf((k[s] - kc) * iw));
    if (kind == 0) {
#pragma unroll
      for (int s = 0; s < NS; ++s) out[s] *= lp[s];
    } else if (kind == 1) {
#pragma unroll
      for (int s = 0; s < NS; ++s) out[s] *= __builtin_amdgcn_sqrtf(fmaxf(1.f - lp[s] * lp[s], 0.f));
    } else {
#pragma unroll
      for (int s = 0; s < NS; ++s) out[s] *= 1.f - lp[s];
    }
  }
  if (F.over_k2) {
#pragma unroll
    for (int s = 0; s < NS; ++s)
      out[s] = ksq[s] == 0 ? 0.f : out[s] * F.inv_kmin2 * __builtin_amdgcn_rcpf(float(ksq[s]));
  }
}
template <typename T, class A> __device__ __forceinline__ T kfactor(const A &a, int ksq) {
  if constexpr (sizeof(T) == 4) {
    if (a.ff.nf >= 0) return filter_fast_f(a.ff, ksq);
    if (!a.tab) return ksq == 0 ? 0.f : a.inv_k2_f * __builtin_amdgcn_rcpf(float(ksq));
  }
  return a.tab ? a.tab[ksq] : T(ksq == 0 ? 0.0 : (1.0 / (double(ksq) * a.kmin_d * a.kmin_d)) * a.inv_k2);
}

// PASS only names the pass (0 x, 1 y, 2 windowed x, 3 windowed y) so that
// profiles tell the launches apart.
// The part of the field one tile of a strided pass works on: C adjacent kz
// columns of one outer line (of one field of a batch).
template <typename T> struct TileG {
  int col0, nc, ky2, iw0;
  const cx<T> *ib;
  cx<T> *ob;
};
template <typename T, int C> __device__ __forceinline__ TileG<T> tile_geom(const StridedArgs<T> &a, int tile) {
  TileG<T> g;
  int outer = tile / a.nkzb, kzb = tile - outer * a.nkzb;
  g.col0 = kzb * C;
  g.nc = min(C, a.ncol - g.col0);
  long boff_in = 0, boff_out = 0;
  int b = 0;
  if (a.nbatch > 1) {
    b = outer / a.nouter;
    outer -= b * a.nouter;
    boff_in = b * a.in_bs;
    boff_out = b * a.out_bs;
  }
  g.iw0 = a.in_win0_b ? a.in_win0_b[b] : a.in_win0;
  g.ib = a.in + boff_in + outer * a.in_os + g.col0;
  g.ob = a.out + boff_out + outer * a.out_os + g.col0;
  const int ky = signed_k(outer, a.n);
  g.ky2 = ky * ky;
  return g;
}
// input value at (line, point) of a tile: zero past the last column and, for
// a pruned input, outside its window
template <typename T, int L>
__device__ __forceinline__ cx<T> tile_in(int in_wlen, long in_ls, const TileG<T> &g, int line, int pt) {
  if (line >= g.nc) return cx<T>{0, 0};
  if (in_wlen > 0 && in_wlen < L) {
    int o = pt - g.iw0;
    if (o < 0) o += L;
    if (o >= in_wlen) return cx<T>{0, 0};
    return g.ib[o * in_ls + line];
  }
  return g.ib[pt * in_ls + line];
}
// the operator's parameters, copied out of the kernel arguments once per
// tile (read through a reference they were reloaded for every mode)
template <typename T> struct PreArgs {
  const T *tab;
  int ncol, n;
  double inv_k2, kmin_d;
  FilterF ff;
  float inv_k2_f;
};
// the factor of |k|^2 of PRE_TABLE: the caller's table, its filter formed
// here (FP32), or inv_k2 / (|k|^2 kMin^2) formed exactly as filter_table
// forms it
template <typename T> struct PreOp {
  PreArgs<T> a;
  int col0, ky2;
  __device__ __forceinline__ int ksq(int line, int pt) const {
    int kx = signed_k(pt, a.n), kz = col0 + line;
    return kx * kx + ky2 + kz * kz;
  }
  // NS slots at once; FP32 filters go through filter_fast_f_n.  Past the last
  // column (its loads are zero) no table is read.
  template <int NS>
  __device__ __forceinline__ void factors(const int (&line)[NS], const int (&pt)[NS], T (&f)[NS]) const {
    if constexpr (sizeof(T) == 4) {
      if (a.ff.nf >= 0) {
        int k[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) k[s] = ksq(line[s], pt[s]);
        float base[NS];
        filter_fast_f_n<NS>(a.ff, k, base);
#pragma unroll
        for (int s = 0; s < NS; ++s) f[s] = col0 + line[s] >= a.ncol ? T(0) : base[s];
        return;
      }
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) f[s] = col0 + line[s] >= a.ncol ? T(0) : kfactor<T>(a, ksq(line[s], pt[s]));
  }
  __device__ __forceinline__ cx<T> apply(cx<T> v, T f) const { return cx<T>{v.x * f, v.y * f}; }
};
// One tile of a strided pass; ld supplies the first stage's inputs.
template <typename T, int L, int C, int DIR, int THREADS, int PRE, int POST, class Ld>
__device__ __forceinline__ void strided_tile(const StridedArgs<T> &a, const cx<T> *__restrict__ tw, cx<T> *lds,
                                             const TileG<T> &g, Ld gld) {
  const int col0 = g.col0, nc = g.nc, ky2 = g.ky2;
  cx<T> *ob = g.ob;
  PreOp<T> op{PreArgs<T>{a.tab, a.ncol, a.n, a.inv_k2, a.kmin_d, a.ff, a.inv_k2_f}, col0, ky2};
  constexpr bool WIDE = PRE == PRE_NONE;
  // the store path's parameters, read once per tile
  const int wlen = a.wlen, win0 = a.win0, accum = a.accum;
  const long out_ls = a.out_ls;
  const T scale = a.scale;
  const cx<T> *aux = a.aux, *out0 = a.out;
  auto gst = [&](int line, int pt, cx<T> v) {
    if (line >= nc) return;
    int o = pt;
    if (wlen < L) {
      o = pt - win0;
      if (o < 0) o += L;
      if (o >= wlen) return;
    }
    T s = scale;
    if constexpr (POST == POST_TABLE) {
      int kx = signed_k(pt, op.a.n), kz = col0 + line;
      s *= kfactor<T>(op.a, kx * kx + ky2 + kz * kz);
    }
    if constexpr (POST == POST_NONE || POST == POST_TABLE) {
      if (accum) {
        cx<T> &dst = ob[o * out_ls + line];
        cx<T> prev = dst;
        dst = cx<T>{prev.x + v.x * s, prev.y + v.y * s};
        return;
      }
    }
    if constexpr (POST == POST_AUX) {
      // the added spectrum is read here, at the store: fetched before the
      // first stage it held 16 more registers through the transform and left
      // one block per CU instead of two
      int kx = signed_k(pt, op.a.n), kz = col0 + line;
      T f = kfactor<T>(op.a, kx * kx + ky2 + kz * kz);
      cx<T> x = aux[long(o) * out_ls + line + (ob - out0)];
      ob[o * out_ls + line] = cx<T>{x.x * f + v.x * s, x.y * f + v.y * s};
      return;
    }
    ob[o * out_ls + line] = cx<T>{v.x * s, v.y * s};
  };
  auto lidx = [](int line, int pt) { return pt * C + line; };
  if constexpr (PRE == PRE_NONE) {
    run_stages<T, L, C, THREADS, DIR, true, false, false, 0, WIDE>(lds, tw, 1, gld, gst, lidx);
  } else {
    run_stages<T, L, C, THREADS, DIR, true, false, false, 0, WIDE>(lds, tw, 1, gld, gst, lidx, op);
  }
}

// One tile per block, tiles in XCD order.
template <typename T, int L, int C, int DIR, int THREADS, int PRE, int POST, int PASS>
__global__ __launch_bounds__(THREADS) void k_fft_strided(StridedArgs<T> a, const cx<T> *__restrict__ tw) {
  extern __shared__ char smem_raw[];
  cx<T> *lds = reinterpret_cast<cx<T> *>(smem_raw);
  // the L twiddles in LDS after the tile: the stages after the first read
  // them there instead of through the vector memory path (the first stage
  // needs none, and the barrier after it publishes the copy)
  cx<T> *ltw = lds + C * L;
  for (int i = int(threadIdx.x); i < L; i += THREADS) ltw[i] = tw[i];
  TileG<T> g = tile_geom<T, C>(a, xcd_tile(blockIdx.x, gridDim.x));
  const int in_wlen = a.in_wlen;   // read once, not per load
  const long in_ls = a.in_ls;
  strided_tile<T, L, C, DIR, THREADS, PRE, POST>(
      a, ltw, lds, g, [&](int line, int pt) { return tile_in<T, L>(in_wlen, in_ls, g, line, pt); });
}

}  // namespace gic
