// Fused passes of the 3D transforms: one launch transforms several fields, or
// makes several fields of one, so that a field is read once for all that is
// made of it.  The displacement map, its transpose, the second-order source
// and the batches are built of these; fft_passes.h has the plain passes.
//
// A strided tile (C adjacent kz columns of one line direction) is held in
// registers, E points a thread; LDS only exchanges points between the stages
// of a transform.  So a tile's spectrum stays in registers while one inverse
// transform after the other is made of it.
#pragma once
#include "fft_passes.h"

namespace gic {

// Radices of a line and points per thread.  FP32 lines of 128 points and
// more take 16 points a thread where the radices allow: one exchange fewer
// at 256 and 1024; FP64 takes 8 (16 would leave two wavefronts per SIMD).
template <typename T, int L> struct LinePlan;
#define GIC_LINE_PLAN(T, L, e, ...)                      \
  template <> struct LinePlan<T, L> {                    \
    static constexpr int E = e;                          \
    static constexpr int R[] = {__VA_ARGS__};            \
    static constexpr int NS = sizeof(R) / sizeof(R[0]);  \
  };
GIC_LINE_PLAN(float, 4, 4, 4)
GIC_LINE_PLAN(float, 8, 8, 8)
GIC_LINE_PLAN(float, 16, 16, 16)
GIC_LINE_PLAN(float, 32, 8, 4, 8)
GIC_LINE_PLAN(float, 64, 8, 8, 8)
GIC_LINE_PLAN(float, 128, 16, 16, 8)
GIC_LINE_PLAN(float, 256, 16, 16, 16)
GIC_LINE_PLAN(float, 512, 8, 8, 8, 8)
GIC_LINE_PLAN(float, 1024, 16, 16, 8, 8)
GIC_LINE_PLAN(double, 4, 4, 4)
GIC_LINE_PLAN(double, 8, 8, 8)
GIC_LINE_PLAN(double, 16, 8, 2, 8)
GIC_LINE_PLAN(double, 32, 8, 4, 8)
GIC_LINE_PLAN(double, 64, 8, 8, 8)
GIC_LINE_PLAN(double, 128, 8, 2, 8, 8)
GIC_LINE_PLAN(double, 256, 8, 4, 8, 8)
GIC_LINE_PLAN(double, 512, 8, 8, 8, 8)
GIC_LINE_PLAN(double, 1024, 8, 2, 8, 8, 8)
#undef GIC_LINE_PLAN

// Columns of a tile: 128-byte segments where a tile and its twiddles leave
// two blocks per CU, 64-byte ones for lines of 1024 points (and FP64): there
// one block of 16 columns a CU loads, transforms and stores by turns, two of 8
// overlap.  1024^3 FP32, the y pass of 2 fields into 3: 7.2 -> 6.0 ms, of 3
// into 6: 11.4 -> 9.8.
template <typename T, int L> struct FusedCols {
  static constexpr int x = sizeof(T) == 4 ? (L == 1024 ? 8 : 16) : (L == 1024 ? 4 : 8);
  static constexpr int y = x;
};

// One line transform of the tile in registers.  REV runs the radices in
// reverse order, so that an inverse transform starts from the points where a
// forward one ended.  A thread holds line tid % C; its element e is the point
// i0 + at<R>(e), i0 = tid / C, before the first stage and after the last (R
// that stage's radix): one offset a thread and constants for the rest, so
// that addresses take one register.  The caller makes sure that LDS is free.
template <typename T, int L, int C, int DIR, bool REV> struct LineFft {
  using P = LinePlan<T, L>;
  static constexpr int E = P::E, NS = P::NS, TH = C * L / E;
  static constexpr int radix(int s) { return P::R[REV ? NS - 1 - s : s]; }
  static constexpr int first = radix(0), last = radix(NS - 1);
  static constexpr int pbefore(int s) {
    int p = 1;
    for (int i = 0; i < s; ++i) p *= radix(i);
    return p;
  }
  template <int R> __host__ __device__ static constexpr int at(int e) { return (e / R) * (L / E) + (e % R) * (L / R); }
  template <int S>
  __device__ __forceinline__ static void stages(cx<T> (&v)[E], cx<T> *lds, const cx<T> *tw, int i0, int line) {
    constexpr int R = radix(S), p = pbefore(S), PER = E / R;
#pragma unroll
    for (int b = 0; b < PER; ++b) {
      const int i = i0 + b * (L / E), k = i % p;
      if constexpr (p > 1) {
#pragma unroll
        for (int r = 1; r < R; ++r) {
          cx<T> w = tw[r * k * (L / (p * R))];
          if (DIR > 0) w.y = -w.y;
          v[b * R + r] = cmul(v[b * R + r], w);
        }
      }
      Dft<R, DIR, T>::run(v + b * R);
    }
    if constexpr (S < NS - 1) {
      if constexpr (S > 0) __syncthreads();   // the stage before has read
#pragma unroll
      for (int b = 0; b < PER; ++b) {
        const int i = i0 + b * (L / E), k = i % p, j = (i - k) * R + k;
        cx<T> *o = lds + j * C + line;
#pragma unroll
        for (int s = 0; s < R; ++s) o[s * p * C] = v[b * R + s];
      }
      __syncthreads();
      constexpr int R2 = radix(S + 1);
      const cx<T> *o = lds + i0 * C + line;
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = o[at<R2>(e) * C];
      stages<S + 1>(v, lds, tw, i0, line);
    }
  }
  __device__ __forceinline__ static void run(cx<T> (&v)[E], cx<T> *lds, const cx<T> *tw) {
    stages<0>(v, lds, tw, fresh(int(threadIdx.x)) / C, fresh(int(threadIdx.x)) % C);
  }
  // a value the compiler takes as new: indexes formed from it are formed
  // where they are used, not held in registers through every stage
  __device__ __forceinline__ static int fresh(int x) {
    asm volatile("" : "+v"(x));
    return x;
  }
  // element e from / to base + (i0 + at<R>(e)) ls + line; base and ls are the
  // same for the whole block, the thread's part fits 32 bits of bytes
  __device__ __forceinline__ static uint32_t offset(long ls) {
    const int t = fresh(int(threadIdx.x));
    return uint32_t((t / C) * uint32_t(ls) + t % C) * uint32_t(sizeof(cx<T>));
  }
  template <int R> __device__ __forceinline__ static void load(cx<T> (&v)[E], const cx<T> *base, long ls, int nc) {
    const uint32_t off = offset(ls);
    if (int(threadIdx.x) % C < nc) {
#pragma unroll
      for (int e = 0; e < E; ++e)
        v[e] = *reinterpret_cast<const cx<T> *>(reinterpret_cast<const char *>(base + at<R>(e) * ls) + off);
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = cx<T>{0, 0};
    }
  }
  // the same of an input that holds only the points [win0, win0 + wlen)
  template <int R>
  __device__ __forceinline__ static void load_window(cx<T> (&v)[E], const cx<T> *base, long ls, int nc, int win0,
                                                     int wlen) {
    const int i0 = fresh(int(threadIdx.x)) / C, line = int(threadIdx.x) % C;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      int o = i0 + at<R>(e) - win0;
      if (o < 0) o += L;
      v[e] = line < nc && o < wlen ? base[o * ls + line] : cx<T>{0, 0};
    }
  }
  template <int R>
  __device__ __forceinline__ static void store(const cx<T> (&v)[E], cx<T> *base, long ls, int nc, int win0, int wlen) {
    if (int(threadIdx.x) % C >= nc) return;
    if (wlen < L) {
      const int i0 = fresh(int(threadIdx.x)) / C, line = int(threadIdx.x) % C;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        int o = i0 + at<R>(e) - win0;
        if (o < 0) o += L;
        if (o < wlen) base[o * ls + line] = v[e];
      }
      return;
    }
    const uint32_t off = offset(ls);
#pragma unroll
    for (int e = 0; e < E; ++e) *reinterpret_cast<cx<T> *>(reinterpret_cast<char *>(base + at<R>(e) * ls) + off) = v[e];
  }
};

// ---- x passes ---------------------------------------------------------------------
// What an x pass makes of a spectrum m(k): the inverse x transforms of
//   out[0]: m (f0 m with the filter given as plain0)   out[1]: f m
//   out[2]: i k_x f m (0 at +Nyquist)                    out[3]: k_x^2 f m
// f is the |k|^2 factor of kfactor (a table, a filter product or inv_k2 /
// k^2).  With FWD the input is a field already transformed along z and y: it
// is transformed along x first, scaled by norm and post[|k|^2], and stored as
// the spectrum spec (if given).  Outputs keep the points [win0, win0 + wlen);
// a FWD input holds the points [iwin0, iwin0 + iwlen) and is 0 elsewhere.
template <typename T> struct XArgs {
  const cx<T> *in;
  cx<T> *spec, *out[4];
  long in_bs, spec_bs, out_bs;   // from one field of a batch (blockIdx.y) to the next
  const T *post;
  T norm, kmin;
  PreArgs<T> f;
  const T *tab0;   // the filter of out[0] where f divides it by k^2 (FP64)
  int plain0;
  int nkzb, win0, wlen, iwin0, iwlen;
};

template <typename T, int L, int C, bool FWD>
__global__ __launch_bounds__((LineFft<T, L, C, 1, true>::TH), 2) void k_fft_x_fused(XArgs<T> a,
                                                                                   const cx<T> *__restrict__ tw) {
  using Fw = LineFft<T, L, C, -1, false>;
  using Bw = LineFft<T, L, C, 1, true>;
  constexpr int E = Bw::E, NZ = L / 2 + 1, R = Bw::first;   // the spectrum's points: at<R>
  constexpr long LS = long(L) * NZ;                          // from one x to the next
  extern __shared__ char smem_raw[];
  cx<T> *lds = reinterpret_cast<cx<T> *>(smem_raw), *ltw = lds + C * L;
  for (int i = int(threadIdx.x); i < L; i += Bw::TH) ltw[i] = tw[i];
  const int tile = xcd_tile(blockIdx.x, gridDim.x), outer = tile / a.nkzb, col0 = (tile - outer * a.nkzb) * C;
  const int nc = min(C, NZ - col0), ky = signed_k(outer, L), ky2 = ky * ky;
  const long base = long(outer) * NZ + col0;
  const cx<T> *in = a.in + long(blockIdx.y) * a.in_bs + base;
  cx<T> v[E];
  if constexpr (FWD) {
    if (a.iwlen < L) Fw::template load_window<Fw::first>(v, in, LS, nc, a.iwin0, a.iwlen);
    else Fw::template load<Fw::first>(v, in, LS, nc);
    __syncthreads();   // the twiddles
    Fw::run(v, lds, ltw);
  } else {
    Bw::template load<R>(v, in, LS, nc);
  }
  // |k|^2 of element e; past the last column any entry of the table
  auto ksq_at = [&](int i0, int kz, int e) {
    const int kx = signed_k(i0 + Bw::template at<R>(e), L);
    return kx * kx + ky2 + kz * kz;
  };
  auto own = [&](int &i0, int &kz) {
    const int t = Bw::fresh(int(threadIdx.x));
    i0 = t / C;
    kz = min(col0 + t % C, NZ - 1);
  };
  if constexpr (FWD) {
    int i0, kz;
    own(i0, kz);
    if (a.post) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const T s = a.norm * a.post[ksq_at(i0, kz, e)];
        v[e] = cx<T>{v[e].x * s, v[e].y * s};
      }
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = cx<T>{v[e].x * a.norm, v[e].y * a.norm};
    }
  }
  if (a.spec) Bw::template store<R>(v, a.spec + long(blockIdx.y) * a.spec_bs + base, LS, nc, 0, L);
  const PreArgs<T> fa = a.f;
  T f[E];
#pragma unroll 1
  for (int s = 0; s < 4; ++s) {
    cx<T> *out = a.out[s];
    const bool more = s == 0 && (a.out[1] || a.out[2] || a.out[3]);
    cx<T> t[E];
    int i0, kz;
    own(i0, kz);
    if (s == 0) {
      if (out) {
        if (a.plain0) {
#pragma unroll
          for (int e = 0; e < E; ++e) {
            T g;
            if constexpr (sizeof(T) == 4) {
              FilterF F = fa.ff;
              F.over_k2 = 0;
              g = filter_fast_f(F, ksq_at(i0, kz, e));
            } else {
              g = a.tab0[ksq_at(i0, kz, e)];
            }
            t[e] = cx<T>{v[e].x * g, v[e].y * g};
          }
        } else {
#pragma unroll
          for (int e = 0; e < E; ++e) t[e] = v[e];
        }
      }
      if (more) {
        bool done = false;
        if constexpr (sizeof(T) == 4) {
          if (fa.ff.nf >= 0) {
            // one factor at a time across four elements (see filter_fast_f_n)
#pragma unroll
            for (int c0 = 0; c0 < E; c0 += 4) {
              const int k4[4] = {ksq_at(i0, kz, c0), ksq_at(i0, kz, c0 + 1), ksq_at(i0, kz, c0 + 2),
                                 ksq_at(i0, kz, c0 + 3)};
              float f4[4];
              filter_fast_f_n<4>(fa.ff, k4, f4);
#pragma unroll
              for (int j = 0; j < 4; ++j) f[c0 + j] = f4[j];
            }
            done = true;
          }
        }
        if (!done) {
#pragma unroll
          for (int e = 0; e < E; ++e) f[e] = kfactor<T>(fa, ksq_at(i0, kz, e));
        }
      }
    }
    if (!out) continue;
    if (s > 0) {
      const T kmin = a.kmin;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int kx = signed_k(i0 + Bw::template at<R>(e), L);
        const T k = T(kx) * kmin;
        T g = f[e];
        if (s == 2) g = kx == L / 2 ? T(0) : g * k;
        if (s == 3) g = g * (k * k);
        t[e] = s == 2 ? cx<T>{-v[e].y * g, v[e].x * g} : cx<T>{v[e].x * g, v[e].y * g};
      }
    }
    __syncthreads();   // the twiddles; that the transform before has read LDS
    Bw::run(t, lds, ltw);
    Bw::template store<Bw::last>(t, out + long(blockIdx.y) * a.out_bs + base, LS, nc, a.win0, a.wlen);
  }
}

// The transpose of a displacement map's x passes: from h1 and h0, transformed
// along z and y, the inverse x transform of
//   tab[|k|^2] norm ( -i k_x X h1 + X h0 ),   X the forward x transform,
// (0 for the first term at +Nyquist), plus the same of a second pair with a
// table of its own, if given; inputs of the points [iwin0, iwin0 + iwlen).
// Without h1 the first term is left out.
template <typename T> struct XAdjArgs {
  cx<T> *out;
  const cx<T> *h1, *h0, *g1, *g0;
  const T *tab, *gtab;
  T norm, kmin;
  int nkzb, iwin0, iwlen;
};
template <typename T, int L, int C>
__global__ __launch_bounds__((LineFft<T, L, C, 1, true>::TH), 2) void k_fft_x_adjoint(XAdjArgs<T> a,
                                                                                     const cx<T> *__restrict__ tw) {
  using Fw = LineFft<T, L, C, -1, false>;
  using Bw = LineFft<T, L, C, 1, true>;
  constexpr int E = Bw::E, NZ = L / 2 + 1, R = Bw::first;
  constexpr long LS = long(L) * NZ;
  extern __shared__ char smem_raw[];
  cx<T> *lds = reinterpret_cast<cx<T> *>(smem_raw), *ltw = lds + C * L;
  for (int i = int(threadIdx.x); i < L; i += Bw::TH) ltw[i] = tw[i];
  const int tile = xcd_tile(blockIdx.x, gridDim.x), outer = tile / a.nkzb, col0 = (tile - outer * a.nkzb) * C;
  const int nc = min(C, NZ - col0), ky = signed_k(outer, L), ky2 = ky * ky;
  const long base = long(outer) * NZ + col0;
  cx<T> v[E], acc[E];
#pragma unroll
  for (int e = 0; e < E; ++e) acc[e] = cx<T>{0, 0};
#pragma unroll 1
  for (int s = 0; s < 4; ++s) {
    const cx<T> *h = s == 0 ? a.h1 : s == 1 ? a.h0 : s == 2 ? a.g1 : a.g0;
    const T *tab = s < 2 ? a.tab : a.gtab;
    if (!h) continue;
    if (a.iwlen < L) Fw::template load_window<Fw::first>(v, h + base, LS, nc, a.iwin0, a.iwlen);
    else Fw::template load<Fw::first>(v, h + base, LS, nc);
    __syncthreads();   // LDS is free, the twiddles are there
    Fw::run(v, lds, ltw);
    const int t = Bw::fresh(int(threadIdx.x)), i0 = t / C, kz = min(col0 + t % C, NZ - 1);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int kx = signed_k(i0 + Bw::template at<R>(e), L);
      const T f = a.norm * tab[kx * kx + ky2 + kz * kz];
      if (s & 1) {
        acc[e].x += f * v[e].x;
        acc[e].y += f * v[e].y;
      } else {
        const T g = kx == L / 2 ? T(0) : f * (T(kx) * a.kmin);
        acc[e].x += g * v[e].y;
        acc[e].y -= g * v[e].x;
      }
    }
  }
  __syncthreads();
  Bw::run(acc, lds, ltw);
  Bw::template store<Bw::last>(acc, a.out + base, LS, nc, 0, L);
}

// ---- y passes ---------------------------------------------------------------------
// Inverse: job j (blockIdx.y) transforms its input times FFT_YZ_* factors of
// (k_y, k_z), up to three fields from one read; outputs keep the points
// [win0, win0 + wlen).  An output may be the input's own memory.
template <typename T> struct YArgs {
  struct Job {
    const cx<T> *in;
    cx<T> *out[3];
    int op[3];
  } job[FUSED_JOBS];
  long in_bs, out_bs;   // batch (blockIdx.z)
  long in_os, out_os;   // from one outer line to the next
  int nkzb, win0, wlen;
  T kmin;
};
template <typename T, int L, int C>
__global__ __launch_bounds__((LineFft<T, L, C, 1, false>::TH), (LineFft<T, L, C, 1, false>::TH > 512 ? 1 : 2)) void
k_fft_y_fused(YArgs<T> a, const cx<T> *__restrict__ tw) {
  using Bw = LineFft<T, L, C, 1, false>;
  constexpr int E = Bw::E, NZ = L / 2 + 1, R = Bw::first;
  extern __shared__ char smem_raw[];
  cx<T> *lds = reinterpret_cast<cx<T> *>(smem_raw), *ltw = lds + C * L;
  for (int i = int(threadIdx.x); i < L; i += Bw::TH) ltw[i] = tw[i];
  const auto &job = a.job[blockIdx.y];
  const int tile = xcd_tile(blockIdx.x, gridDim.x), outer = tile / a.nkzb, col0 = (tile - outer * a.nkzb) * C;
  const int nc = min(C, NZ - col0);
  cx<T> v[E];
  Bw::template load<R>(v, job.in + long(blockIdx.z) * a.in_bs + outer * a.in_os + col0, NZ, nc);
#pragma unroll 1
  for (int s = 0; s < 3; ++s) {
    cx<T> *out = job.out[s];
    if (!out) break;
    const YzOp op = yz_op(job.op[s]);
    const int t0 = Bw::fresh(int(threadIdx.x)), i0 = t0 / C;
    const T gz = k_power<T>(op.pz, col0 + t0 % C, L / 2, a.kmin), kmin = a.kmin;
    cx<T> t[E];
#pragma unroll
    for (int e = 0; e < E; ++e)
      t[e] = rot_mul<T>(op.rot, v[e], gz * k_power<T>(op.py, signed_k(i0 + Bw::template at<R>(e), L), L / 2, kmin));
    __syncthreads();   // the twiddles; later, that LDS has been read
    Bw::run(t, lds, ltw);
    Bw::template store<Bw::last>(t, out + long(blockIdx.z) * a.out_bs + outer * a.out_os + col0, NZ, nc, a.win0,
                                 a.wlen);
  }
}

// Forward: out = Y in (op[0] one), or with a second input
// out = -i k_y Y in - i k_z Y in2 (0 at +Nyquist): the y passes of the
// transpose of psi_y and psi_z, whose x passes they share.
template <typename T> struct YFwdArgs {
  struct Job {
    const cx<T> *in, *in2;
    cx<T> *out;
  } job[FUSED_JOBS];
  long bs;
  int nkzb, iwin0, iwlen;
  T kmin;
};
template <typename T, int L, int C>
__global__ __launch_bounds__((LineFft<T, L, C, 1, false>::TH), (LineFft<T, L, C, 1, false>::TH > 512 ? 1 : 2)) void
k_fft_y_forward(YFwdArgs<T> a, const cx<T> *__restrict__ tw) {
  using Fw = LineFft<T, L, C, -1, false>;
  constexpr int E = Fw::E, NZ = L / 2 + 1, R = Fw::last;
  extern __shared__ char smem_raw[];
  cx<T> *lds = reinterpret_cast<cx<T> *>(smem_raw), *ltw = lds + C * L;
  for (int i = int(threadIdx.x); i < L; i += Fw::TH) ltw[i] = tw[i];
  const auto &job = a.job[blockIdx.y];
  const int tile = xcd_tile(blockIdx.x, gridDim.x), outer = tile / a.nkzb, col0 = (tile - outer * a.nkzb) * C;
  const int nc = min(C, NZ - col0);
  const long at = long(blockIdx.z) * a.bs + long(outer) * L * NZ + col0;
  const long in = long(blockIdx.z) * a.bs + long(outer) * a.iwlen * NZ + col0;
  cx<T> v[E];
  auto load = [&](const cx<T> *p) {
    if (a.iwlen < L) Fw::template load_window<Fw::first>(v, p + in, NZ, nc, a.iwin0, a.iwlen);
    else Fw::template load<Fw::first>(v, p + in, NZ, nc);
  };
  load(job.in);
  __syncthreads();
  Fw::run(v, lds, ltw);
  if (job.in2) {
    cx<T> r[E];
    {
      const int i0 = Fw::fresh(int(threadIdx.x)) / C;
#pragma unroll
      for (int e = 0; e < E; ++e)
        r[e] = rot_mul<T>(3, v[e], k_power<T>(1, signed_k(i0 + Fw::template at<R>(e), L), L / 2, a.kmin));
    }
    load(job.in2);
    __syncthreads();
    Fw::run(v, lds, ltw);
    const T gz = k_power<T>(1, col0 + Fw::fresh(int(threadIdx.x)) % C, L / 2, a.kmin);
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = cadd(r[e], rot_mul<T>(3, v[e], gz));
  }
  Fw::template store<R>(v, job.out + at, NZ, nc, 0, L);
}

// ---- launches ---------------------------------------------------------------------
template <typename T, int N> struct FftFused {
  using F = FftN<T, N>;
  using Rows = RowLaunch<T, N>;
  static constexpr int NZ = N / 2 + 1;
  static constexpr int CX = FusedCols<T, N>::x, CY = FusedCols<T, N>::y;
  static constexpr double FIELD = double(N) * N * NZ * sizeof(cx<T>);   // bytes of a spectrum
  static cx<T> *c(T *p) { return reinterpret_cast<cx<T> *>(p); }
  static const cx<T> *c(const T *p) { return reinterpret_cast<const cx<T> *>(p); }
  template <class K, class... A>
  static void launch(K kern, dim3 grid, int threads, size_t shm, const char *name, double bytes, hipStream_t st,
                     TimingHook *hook, const A &...args) {
    if (shm > 65536)
      GIC_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
    std::string tag;
    if (hook) {
      tag = std::string(name) + "." + std::to_string(N);
      hook->begin(tag.c_str(), st);
      hook->bytes(tag.c_str(), bytes);
    }
    hipLaunchKernelGGL(kern, grid, dim3(threads), shm, st, args..., twtable<T>().get(N));
    GIC_HIP(hipGetLastError());
    if (hook) hook->end(tag.c_str(), st);
  }
  static size_t tile_lds(int cols) { return sizeof(cx<T>) * (cols + 1) * N; }

  static void x(const FftX<T> &q, hipStream_t st, TimingHook *hook) {
    XArgs<T> a{};
    a.in = c(q.in);
    a.spec = c(q.spec);
    for (int i = 0; i < 4; ++i) a.out[i] = c(q.out[i]);
    a.in_bs = q.in_bs / 2;
    a.spec_bs = q.spec_bs / 2;
    a.out_bs = q.out_bs / 2;
    a.post = q.post;
    a.norm = F::norm();
    a.kmin = T(q.kmin);
    StridedArgs<T> s{};   // the factor's parameters, as the plain passes prepare them
    s.tab = q.tab;
    s.kmin_d = q.kmin;
    s.inv_k2 = q.inv_k2;
    if (q.fil) s.fil = *q.fil;
    F::prepare_factor(s);
    a.f = PreArgs<T>{s.tab, NZ, N, s.inv_k2, s.kmin_d, s.ff, s.inv_k2_f};
    a.tab0 = q.tab0;
    a.plain0 = q.plain0 ? 1 : 0;
    if ((q.out[1] || q.out[2] || q.out[3]) && !q.tab && q.inv_k2 == 0 && s.ff.nf < 0)
      throw std::runtime_error("fft_x: outputs without a factor");
    if (q.plain0 && (!q.fil || !q.tab0)) throw std::runtime_error("fft_x: plain0 without its filter");
    a.nkzb = (NZ + CX - 1) / CX;
    a.win0 = q.wlen > 0 ? q.win0 : 0;
    a.wlen = q.wlen > 0 ? q.wlen : N;
    a.iwin0 = q.iwlen > 0 ? q.iwin0 : 0;
    a.iwlen = q.iwlen > 0 ? q.iwlen : N;
    int outs = 0;
    for (auto *o : q.out) outs += o ? 1 : 0;
    double bytes = q.nb * FIELD * (double(a.iwlen) / N + (q.spec ? 1.0 : 0.0) + outs * double(a.wlen) / N);
    constexpr int TH = LineFft<T, N, CX, 1, true>::TH;
    dim3 grid(N * a.nkzb, q.nb);
    if (q.forward)
      launch(k_fft_x_fused<T, N, CX, true>, grid, TH, tile_lds(CX), "fft_x_fwd_inv", bytes, st, hook, a);
    else
      launch(k_fft_x_fused<T, N, CX, false>, grid, TH, tile_lds(CX), q.wlen > 0 ? "fft_x_multi_win" : "fft_x_multi",
             bytes, st, hook, a);
  }
  static void y(const FftY<T> &q, hipStream_t st, TimingHook *hook) {
    YArgs<T> a{};
    double fields = 0;
    a.win0 = q.wlen > 0 ? q.win0 : 0;
    a.wlen = q.wlen > 0 ? q.wlen : N;
    for (int j = 0; j < q.njob; ++j) {
      a.job[j].in = c(q.job[j].in);
      fields += 1;
      for (int i = 0; i < 3; ++i) {
        a.job[j].out[i] = c(q.job[j].out[i]);
        a.job[j].op[i] = q.job[j].op[i];
        if (q.job[j].out[i]) fields += double(a.wlen) / N;
      }
    }
    const int nouter = q.nouter > 0 ? q.nouter : N;
    a.in_bs = q.in_bs / 2;
    a.out_bs = q.out_bs / 2;
    a.in_os = long(N) * NZ;
    a.out_os = long(a.wlen) * NZ;
    a.nkzb = (NZ + CY - 1) / CY;
    a.kmin = T(q.kmin);
    constexpr int TH = LineFft<T, N, CY, 1, false>::TH;
    launch(k_fft_y_fused<T, N, CY>, dim3(nouter * a.nkzb, q.njob, q.nb), TH, tile_lds(CY),
           q.wlen > 0 ? "fft_y_multi_win" : "fft_y_multi", q.nb * FIELD * fields * nouter / N, st, hook, a);
  }
  static void y_forward(const FftYFwd<T> &q, hipStream_t st, TimingHook *hook) {
    YFwdArgs<T> a{};
    double fields = 0;
    for (int j = 0; j < q.njob; ++j) {
      a.job[j].in = c(q.job[j].in);
      a.job[j].in2 = c(q.job[j].in2);
      a.job[j].out = c(q.job[j].out);
      fields += 1 + (q.job[j].in2 ? 2 : 1) * double(q.iwlen > 0 ? q.iwlen : N) / N;
    }
    const int nouter = q.nouter > 0 ? q.nouter : N;
    a.iwin0 = q.iwlen > 0 ? q.iwin0 : 0;
    a.iwlen = q.iwlen > 0 ? q.iwlen : N;
    a.bs = q.bs / 2;
    a.nkzb = (NZ + CY - 1) / CY;
    a.kmin = T(q.kmin);
    constexpr int TH = LineFft<T, N, CY, 1, false>::TH;
    launch(k_fft_y_forward<T, N, CY>, dim3(nouter * a.nkzb, q.njob, q.nb), TH, tile_lds(CY), "fft_y_fwd_multi",
           q.nb * FIELD * fields * nouter / N, st, hook, a);
  }
  static void x_adjoint(const FftXAdj<T> &q, hipStream_t st, TimingHook *hook) {
    XAdjArgs<T> a{c(q.out), c(q.h1), c(q.h0), c(q.g1), c(q.g0), q.tab, q.gtab, F::norm(), T(q.kmin), (NZ + CX - 1) / CX,
                  q.iwlen > 0 ? q.iwin0 : 0, q.iwlen > 0 ? q.iwlen : N};
    constexpr int TH = LineFft<T, N, CX, 1, true>::TH;
    launch(k_fft_x_adjoint<T, N, CX>, dim3(N * a.nkzb), TH, tile_lds(CX), "fft_x_adjoint",
           FIELD * (1 + (q.g1 ? 4 : 2) * double(a.iwlen) / N), st, hook, a);
  }
  static void z(const FftZ<T> &q, hipStream_t st, TimingHook *hook) {
    ZArgs<T> a{};
    double fields = 0;
    for (int j = 0; j < q.njob; ++j) {
      a.job[j] = {q.job[j].in, q.job[j].out, q.job[j].dense, q.job[j].op};
      fields += 1 + (q.job[j].out ? 1 : 0) + (q.job[j].dense ? 1 : 0);
    }
    a.in_bs = q.in_bs;
    a.out_bs = q.out_bs;
    a.dense_bs = q.dense_bs;
    a.nrows = long(N) * N;
    a.iters = Rows::iters(a.nrows, long(q.njob) * q.nb);
    a.scale = F::norm() * T(q.scale);
    a.kmin = T(q.kmin);
    F::rows_launch(k_fft_z_c2r<T, N, Rows::TH, false>, a, q.njob, q.nb, "fft_z_c2r_multi", q.nb * FIELD * fields, st,
                   hook);
  }
  static void z_forward(const FftZFwd<T> &q, hipStream_t st, TimingHook *hook) {
    ZFwdArgs<T> a{};
    for (int j = 0; j < q.njob; ++j) a.job[j] = {q.job[j].src, q.job[j].out, q.job[j].dense ? long(N) : long(N + 2)};
    a.src_bs = q.src_bs;
    a.out_bs = q.out_bs;
    a.nrows = long(N) * N;
    a.iters = Rows::iters(a.nrows, long(q.njob) * q.nb);
    F::rows_launch(k_fft_z_r2c<T, N, Rows::TH, false>, a, q.njob, q.nb, "fft_z_r2c_multi", q.nb * FIELD * 2 * q.njob, st,
                   hook);
  }
  static void z_lpt(T *px, T *py, T *pz, const T *xx, const T *yy, const T *xy, T *S, bool psi, double kmin,
                    hipStream_t st, TimingHook *hook) {
    const long nrows = long(N) * N;
    ZLptArgs<T> a{px, py, pz, xx, yy, xy, S, nrows, Rows::iters(nrows, 1), F::norm(), T(kmin)};
    if (psi) F::rows_launch(k_fft_z_lpt<T, N, Rows::TH, true>, a, 1, 1, "fft_z_lpt", FIELD * 10, st, hook);
    else F::rows_launch(k_fft_z_lpt<T, N, Rows::TH, false>, a, 1, 1, "fft_z_lpt", FIELD * 7, st, hook);
  }
};

template <typename T, int N> FftApi<T> fft_api_of() {
  using F = FftN<T, N>;
  using G = FftFused<T, N>;
  FftApi<T> a;
  a.r2c = F::r2c;
  a.r2c_batch = F::r2c_batch;
  a.r2c_boxes = F::r2c_boxes;
  a.c2r = F::c2r;
  a.c2r_from = F::c2r_from;
  a.c2r_window = F::c2r_window;
  a.r2c_window = F::r2c_window;
  a.r2c_window_zy = F::r2c_window_zy;
  a.r2c_z_window = F::r2c_z_window;
  a.z_window = F::z_window;
  a.x = G::x;
  a.y = G::y;
  a.y_forward = G::y_forward;
  a.x_adjoint = G::x_adjoint;
  a.z = G::z;
  a.z_forward = G::z_forward;
  a.z_lpt = G::z_lpt;
  return a;
}
#ifndef GIC_FFT_SPLIT
template <typename T, int N> const FftApi<T> &fft_api() {
  static const FftApi<T> a = fft_api_of<T, N>();
  return a;
}
#endif

}  // namespace gic
