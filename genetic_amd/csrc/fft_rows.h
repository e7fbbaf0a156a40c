// The passes along z: real rows to half-length complex rows and back.
//
// A row belongs to M / E lanes of one wavefront (N = 2 M reals, E points a
// lane), so that the stages of its transform exchange points through LDS
// without a barrier of the block, and each wavefront loads, transforms and
// stores on its own.  The pairs k, M - k that a real transform combines are
// read twice (from the row itself, the second time from the cache) instead of
// being rearranged in LDS first.  Twiddles lie in LDS in the order in which a
// stage's lanes read them.
//
// Rows whose points went through LDS for the whole block before the first
// stage took 86 vector instructions a complex point (54 % of the issue slots
// at 1024^3 FP32, 71 % in the second-order pass); measured before and now:
// c2r of three fields 1024^3 FP32 6.7 -> 5.4 ms (4.7 TB/s), 256^3 77 -> 59 us,
// 64^3 10.9 -> 5.6 us; of one field 512^3 FP64 496 -> 405 us (5.3 TB/s); the
// second-order pass at 1024^3 FP32 16.9 -> 11.6 ms (3.7 TB/s); r2c, which
// memory bounds, 1.6 -> 1.7 ms at 1024^3 FP32 and 397 -> 401 us at 512^3 FP64.
#pragma once
#include "fft_strided.h"

namespace gic {

// Radices of a row of M complex points, and points a lane.
template <int M> struct RowPlan;
#define GIC_ROW_PLAN(M, e, ...)                          \
  template <> struct RowPlan<M> {                        \
    static constexpr int E = e;                          \
    static constexpr int R[] = {__VA_ARGS__};            \
    static constexpr int NS = sizeof(R) / sizeof(R[0]);  \
  };
GIC_ROW_PLAN(2, 2, 2)
GIC_ROW_PLAN(4, 4, 4)
GIC_ROW_PLAN(8, 8, 8)
GIC_ROW_PLAN(16, 8, 2, 8)
GIC_ROW_PLAN(32, 8, 4, 8)
GIC_ROW_PLAN(64, 8, 8, 8)
GIC_ROW_PLAN(128, 8, 2, 8, 8)
GIC_ROW_PLAN(256, 8, 4, 8, 8)
GIC_ROW_PLAN(512, 8, 8, 8, 8)
#undef GIC_ROW_PLAN

template <typename T, int M> struct RowFft {
  using P = RowPlan<M>;
  static constexpr int E = P::E, NS = P::NS, LPR = M / E, RPW = 64 / LPR;
  static constexpr int LEN = M >= 8 ? M + M / 8 : M;   // a row in LDS, a gap after every 8 points
  static constexpr int first = P::R[0], last = P::R[NS - 1];
  static_assert(LPR <= 64 && 64 % LPR == 0, "a row belongs to one wavefront");
  __device__ __forceinline__ static constexpr int idx(int pt) { return M >= 8 ? pt + pt / 8 : pt; }
  static constexpr int pbefore(int s) {
    int p = 1;
    for (int i = 0; i < s; ++i) p *= P::R[i];
    return p;
  }
  // stage s >= 1 reads its factor r (1..R-1) for k (0..p-1) at tw_at(s) + (r - 1) p + k
  static constexpr int tw_at(int s) {
    int o = 0;
    for (int i = 1; i < s; ++i) o += (P::R[i] - 1) * pbefore(i);
    return o;
  }
  static constexpr int TW = tw_at(NS);      // the stages' factors, then exp(-2 pi i k / N), k < M
  static constexpr int TABLE = TW + M;
  // point of element e: i0 + at<R>(e), R the first stage's radix before the
  // transform, the last stage's after it
  template <int R> __host__ __device__ static constexpr int at(int e) { return (e / R) * (M / E) + (e % R) * (M / R); }

  // the table from the N-point factors; the caller's barrier publishes it
  template <int S = 1> __device__ __forceinline__ static void table(cx<T> *ltw, const cx<T> *__restrict__ twN, int threads) {
    if constexpr (S < NS) {
      constexpr int R = P::R[S], p = pbefore(S), cnt = (R - 1) * p;
      for (int i = int(threadIdx.x); i < cnt; i += threads)
        ltw[tw_at(S) + i] = twN[2 * (i / p + 1) * (i % p) * (M / (p * R))];
      table<S + 1>(ltw, twN, threads);
    } else {
      for (int i = int(threadIdx.x); i < M; i += threads) ltw[TW + i] = twN[i];
    }
  }
  // orders a wavefront's LDS accesses (which complete in order) for the compiler
  __device__ __forceinline__ static void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  template <int DIR, int S = 0>
  __device__ __forceinline__ static void run(cx<T> (&v)[E], cx<T> *row, const cx<T> *ltw, int i0) {
    constexpr int R = P::R[S], p = pbefore(S), PER = E / R;
#pragma unroll
    for (int b = 0; b < PER; ++b) {
      const int k = (i0 + b * (M / E)) % p;
      if constexpr (p > 1) {
#pragma unroll
        for (int r = 1; r < R; ++r) {
          cx<T> w = ltw[tw_at(S) + (r - 1) * p + k];
          if (DIR > 0) w.y = -w.y;
          v[b * R + r] = cmul(v[b * R + r], w);
        }
      }
      Dft<R, DIR, T>::run(v + b * R);
    }
    if constexpr (S < NS - 1) {
      wave_sync();   // what was read before has been
#pragma unroll
      for (int b = 0; b < PER; ++b) {
        const int i = i0 + b * (M / E), k = i % p, j = (i - k) * R + k;
#pragma unroll
        for (int s = 0; s < R; ++s) row[idx(j + s * p)] = v[b * R + s];
      }
      wave_sync();
      constexpr int R2 = P::R[S + 1];
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = row[idx(i0 + at<R2>(e))];
      run<DIR, S + 1>(v, row, ltw, i0);
    }
  }
  // A complex row X (its points i0 + at<first>(e) in v, M minus those in m) as
  // the half-length transform's input; the imaginary parts of k_z = 0 and
  // +Nyquist are ignored, as a c2r does.
  __device__ __forceinline__ static void pack(cx<T> (&v)[E], cx<T> (&m)[E], const cx<T> *ltw, int i0) {
    if (i0 == 0) v[0].y = m[0].y = T(0);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      cx<T> w = ltw[TW + i0 + at<first>(e)];
      w.y = -w.y;
      const cx<T> o = cmul(cx<T>{v[e].x - m[e].x, v[e].y + m[e].y}, w);
      v[e] = cx<T>{v[e].x + m[e].x - o.y, v[e].y - m[e].y + o.x};
    }
  }
};

// which rows a wavefront works on, of its job's nrows
template <typename T, int M, int WAVES> struct RowSpan {
  using F = RowFft<T, M>;
  int lane, i0, sub;
  long row0;
  __device__ __forceinline__ RowSpan() {
    lane = int(threadIdx.x) % 64;
    i0 = lane % F::LPR;
    sub = lane / F::LPR;
  }
  // false past the last row; a lane without a row repeats the last one
  __device__ __forceinline__ bool at(long it, long nrows) {
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / 64);
    row0 = (it * WAVES + wave) * F::RPW;
    return row0 < nrows;
  }
  __device__ __forceinline__ bool live(long nrows) const { return row0 + sub < nrows; }
  __device__ __forceinline__ int row(long nrows) const {
    const int left = int(min(nrows - row0, long(F::RPW)));
    return min(sub, left - 1);
  }
};

// FFT_YZ_* as i^rot k_y^py k_z^pz, the first powers 0 at +Nyquist
struct YzOp {
  int rot, py, pz;
};
__device__ __forceinline__ YzOp yz_op(int op) {
  YzOp r{0, 0, 0};
  switch (op) {
    case FFT_YZ_IKY: return {1, 1, 0};
    case FFT_YZ_IKZ: return {1, 0, 1};
    case FFT_YZ_MIKY: return {3, 1, 0};
    case FFT_YZ_KYKY: return {0, 2, 0};
    case FFT_YZ_KY: return {0, 1, 0};
  }
  return r;
}
template <typename T> __device__ __forceinline__ T k_power(int p, int k, int nyq, T kmin) {
  const T f = T(k) * kmin;
  return p == 0 ? T(1) : p == 2 ? f * f : k == nyq ? T(0) : f;
}
template <typename T> __device__ __forceinline__ cx<T> rot_mul(int rot, cx<T> v, T f) {
  if (rot == 0) return cx<T>{v.x * f, v.y * f};
  if (rot == 3) f = -f;
  return cx<T>{-v.y * f, v.x * f};
}

// the row at base (+ 32-bit offset) times i^rot k_z^pz, ready for run<+1>
template <typename T, int M>
__device__ __forceinline__ void row_load(cx<T> (&v)[RowPlan<M>::E], const cx<T> *base, int row, int i0, YzOp op, T kmin,
                                         const cx<T> *ltw) {
  using F = RowFft<T, M>;
  constexpr int E = F::E, R = F::first;
  const uint32_t o = uint32_t(row) * uint32_t(M + 1), up = o + uint32_t(i0), dn = o + uint32_t(M - i0);
  cx<T> m[E];
#pragma unroll
  for (int e = 0; e < E; ++e) v[e] = base[up + uint32_t(F::template at<R>(e))];
#pragma unroll
  for (int e = 0; e < E; ++e) m[e] = base[dn - uint32_t(F::template at<R>(e))];
  if (op.rot | op.pz) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int k = i0 + F::template at<R>(e);
      v[e] = rot_mul<T>(op.rot, v[e], k_power<T>(op.pz, k, M, kmin));
      m[e] = rot_mul<T>(op.rot, m[e], k_power<T>(op.pz, M - k, M, kmin));
    }
  }
  F::pack(v, m, ltw, i0);
}

// c2r of several fields (blockIdx.y) of a batch (blockIdx.z): complex rows
// times a factor of k_z (FFT_YZ_ONE or FFT_YZ_IKZ), the real rows
// to the padded field out (may be the input), a dense array, or both.  WIN:
// only the points [z0, z0 + wz) mod N, to dense rows of wz reals.
constexpr int FUSED_JOBS = 6;
template <typename T> struct ZArgs {
  struct Job {
    const T *in;
    T *out, *dense;
    int op;
  } job[FUSED_JOBS];
  long in_bs, out_bs, dense_bs;   // reals
  long nrows;
  int iters, z0, wz;
  T scale, kmin;
};

template <typename T, int N, int TH, bool WIN>
__global__ __launch_bounds__(TH) void k_fft_z_c2r(ZArgs<T> a, const cx<T> *__restrict__ twN) {
  constexpr int M = N / 2, WAVES = TH / 64;
  using F = RowFft<T, M>;
  constexpr int E = F::E, R = F::last;
  extern __shared__ char smem_raw[];
  cx<T> *ltw = reinterpret_cast<cx<T> *>(smem_raw);
  RowSpan<T, M, WAVES> s;
  cx<T> *lrow = ltw + F::TABLE + (int(threadIdx.x) / F::LPR) * F::LEN;
  F::table(ltw, twN, TH);
  __syncthreads();
  const auto &job = a.job[blockIdx.y];
  const cx<T> *in = reinterpret_cast<const cx<T> *>(job.in + long(blockIdx.z) * a.in_bs);
  const YzOp op = yz_op(job.op);
#pragma unroll 1
  for (int it = 0; it < a.iters; ++it) {
    if (!s.at(long(blockIdx.x) * a.iters + it, a.nrows)) return;
    cx<T> v[E];
    const int row = s.row(a.nrows);
    row_load<T, M>(v, in + s.row0 * (M + 1), row, s.i0, op, a.kmin, ltw);
    F::template run<+1>(v, lrow, ltw, s.i0);
    if (!s.live(a.nrows)) continue;
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = cx<T>{v[e].x * a.scale, v[e].y * a.scale};
    if constexpr (WIN) {
      T *o = job.dense + s.row0 * a.wz + uint32_t(row) * uint32_t(a.wz);
#pragma unroll
      for (int e = 0; e < E; ++e) {
        // complex point pt holds the reals 2 pt, 2 pt + 1
        int z = 2 * (s.i0 + F::template at<R>(e)) - a.z0, z1 = z + 1;
        z += z < 0 ? N : 0;
        z1 += z1 < 0 ? N : 0;
        if (z < a.wz) o[z] = v[e].x;
        if (z1 < a.wz) o[z1] = v[e].y;
      }
    } else {
      if (job.out) {
        cx<T> *o = reinterpret_cast<cx<T> *>(job.out + long(blockIdx.z) * a.out_bs) + s.row0 * (M + 1);
        const uint32_t at0 = uint32_t(row) * uint32_t(M + 1) + uint32_t(s.i0);
#pragma unroll
        for (int e = 0; e < E; ++e) o[at0 + uint32_t(F::template at<R>(e))] = v[e];
      }
      if (job.dense) {
        cx<T> *o = reinterpret_cast<cx<T> *>(job.dense + long(blockIdx.z) * a.dense_bs) + s.row0 * M;
        const uint32_t at0 = uint32_t(row) * uint32_t(M) + uint32_t(s.i0);
#pragma unroll
        for (int e = 0; e < E; ++e) o[at0 + uint32_t(F::template at<R>(e))] = v[e];
      }
    }
  }
}

// r2c of several fields: real rows from a padded field or a dense array (row
// stride srs reals) to padded complex rows (may be the input).  WIN: the rows
// hold the points [z0, z0 + wz) mod N, wz reals each, and are 0 elsewhere.
template <typename T> struct ZFwdArgs {
  struct Job {
    const T *src;
    T *out;
    long srs;
  } job[FUSED_JOBS];
  long src_bs, out_bs, nrows;
  int iters, z0, wz;
};
template <typename T, int N, int TH, bool WIN>
__global__ __launch_bounds__(TH) void k_fft_z_r2c(ZFwdArgs<T> a, const cx<T> *__restrict__ twN) {
  constexpr int M = N / 2, WAVES = TH / 64;
  using F = RowFft<T, M>;
  constexpr int E = F::E, R = F::first, RL = F::last;
  extern __shared__ char smem_raw[];
  cx<T> *ltw = reinterpret_cast<cx<T> *>(smem_raw);
  RowSpan<T, M, WAVES> s;
  cx<T> *lrow = ltw + F::TABLE + (int(threadIdx.x) / F::LPR) * F::LEN;
  F::table(ltw, twN, TH);
  __syncthreads();
  const auto &job = a.job[blockIdx.y];
#pragma unroll 1
  for (int it = 0; it < a.iters; ++it) {
    if (!s.at(long(blockIdx.x) * a.iters + it, a.nrows)) return;
    cx<T> v[E];
    const int row = s.row(a.nrows);
    if constexpr (WIN) {
      const T *in = job.src + s.row0 * a.wz + uint32_t(row) * uint32_t(a.wz);
#pragma unroll
      for (int e = 0; e < E; ++e) {
        int z = 2 * (s.i0 + F::template at<R>(e)) - a.z0, z1 = z + 1;
        z += z < 0 ? N : 0;
        z1 += z1 < 0 ? N : 0;
        v[e].x = z < a.wz ? in[z] : T(0);
        v[e].y = z1 < a.wz ? in[z1] : T(0);
      }
    } else {
      const cx<T> *in = reinterpret_cast<const cx<T> *>(job.src + long(blockIdx.z) * a.src_bs) + s.row0 * (job.srs / 2);
      const uint32_t at0 = uint32_t(row) * uint32_t(job.srs / 2) + uint32_t(s.i0);
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = in[at0 + uint32_t(F::template at<R>(e))];
    }
    F::template run<-1>(v, lrow, ltw, s.i0);
    // X_k of Z_k and Z_{M-k}
    F::wave_sync();
#pragma unroll
    for (int e = 0; e < E; ++e) lrow[F::idx(s.i0 + F::template at<RL>(e))] = v[e];
    F::wave_sync();
    cx<T> *o = reinterpret_cast<cx<T> *>(job.out + long(blockIdx.z) * a.out_bs) + s.row0 * (M + 1);
    const uint32_t at0 = uint32_t(row) * uint32_t(M + 1) + uint32_t(s.i0);
    const bool live = s.live(a.nrows);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int k = s.i0 + F::template at<RL>(e);
      const cx<T> zk = v[e], zm = lrow[F::idx((M - k) % M)];
      const cx<T> f{(zk.x + zm.x) * T(0.5), (zk.y - zm.y) * T(0.5)};
      const cx<T> d{(zk.x - zm.x) * T(0.5), (zk.y + zm.y) * T(0.5)};
      const cx<T> g = cmul(ltw[F::TW + k], cx<T>{d.y, -d.x});
      if (live) o[at0 + uint32_t(F::template at<RL>(e))] = cx<T>{f.x + g.x, f.y + g.y};
      if (e == 0 && live && s.i0 == 0) o[at0 + uint32_t(M)] = cx<T>{f.x - g.x, -(f.y - g.y)};   // k = M
    }
  }
}

// The second-order source and the first-order displacements of one level
// from six fields transformed along x and y:
//   px: of i k_x f m   py: of k_y f m times X0   pz: of f m   (X0, X1 of the x pass)
//   xx: of k_x^2 f m   yy: of k_y^2 f m           xy: of k_x k_y f m
// psi_x = Z px, psi_y = Z i py, psi_z = Z i k_z pz, phi_xz = Z (-i k_z) px,
// phi_yz = Z k_z py, phi_zz = Z k_z^2 pz, and
//   S = xx yy + (xx + yy) zz - xy^2 - xz^2 - yz^2
// so that each of the six is read once from memory for the nine transforms
// made of it.  With PSI the displacements go over px, py, pz; S to a padded
// field.
template <typename T> struct ZLptArgs {
  T *px, *py, *pz;
  const T *xx, *yy, *xy;
  T *S;
  long nrows;
  int iters;
  T scale, kmin;
};
template <typename T, int N, int TH, bool PSI>
__global__ __launch_bounds__(TH, (sizeof(T) == 4 ? 4 : 2)) void k_fft_z_lpt(ZLptArgs<T> a,
                                                                           const cx<T> *__restrict__ twN) {
  constexpr int M = N / 2, WAVES = TH / 64;
  using F = RowFft<T, M>;
  constexpr int E = F::E, R = F::last;
  extern __shared__ char smem_raw[];
  cx<T> *ltw = reinterpret_cast<cx<T> *>(smem_raw);
  RowSpan<T, M, WAVES> sp;
  cx<T> *lrow = ltw + F::TABLE + (int(threadIdx.x) / F::LPR) * F::LEN;
  F::table(ltw, twN, TH);
  __syncthreads();
#pragma unroll 1
  for (int it = 0; it < a.iters; ++it) {
    if (!sp.at(long(blockIdx.x) * a.iters + it, a.nrows)) return;
    const bool live = sp.live(a.nrows);
    const int row = sp.row(a.nrows);
    cx<T> S[E], A[E];
    // one piece of code for the nine transforms; indexes formed anew in each
    // (they would fill the registers that S and A need)
#pragma unroll 1
    for (int s = 0; s < (PSI ? 9 : 6); ++s) {
      // xx, yy, zz, xy, xz, yz, then the displacements, each over its own rows,
      // whose last reading this is
      T *own = s == 6 ? a.px : s == 7 ? a.py : a.pz;
      const T *src = s == 0 ? a.xx : s == 1 ? a.yy : s == 2 ? a.pz : s == 3 ? a.xy : s == 4 ? a.px : s == 5 ? a.py : own;
      const YzOp f = s == 2 ? YzOp{0, 0, 2} : s == 4 ? YzOp{3, 0, 1} : s == 5 ? YzOp{0, 0, 1} : s == 7 ? YzOp{1, 0, 0}
                     : s == 8 ? YzOp{1, 0, 1} : YzOp{0, 0, 0};
      int i0 = sp.i0;
      asm volatile("" : "+v"(i0));
      cx<T> v[E];
      row_load<T, M>(v, reinterpret_cast<const cx<T> *>(src) + sp.row0 * (M + 1), row, i0, f, a.kmin, ltw);
      F::template run<+1>(v, lrow, ltw, i0);
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const cx<T> x{v[e].x * a.scale, v[e].y * a.scale};
        if (s == 0) {
          A[e] = x;
        } else if (s == 1) {
          S[e] = cx<T>{A[e].x * x.x, A[e].y * x.y};
          A[e] = cadd(A[e], x);
        } else if (s == 2) {
          S[e] = cx<T>{S[e].x + A[e].x * x.x, S[e].y + A[e].y * x.y};
        } else if (s < 6) {
          S[e] = cx<T>{S[e].x - x.x * x.x, S[e].y - x.y * x.y};
        } else {
          A[e] = x;
        }
      }
      if (s >= 5 && live) {
        T *dst = s == 5 ? a.S : own;
        cx<T> *o = reinterpret_cast<cx<T> *>(dst) + sp.row0 * (M + 1);
        const uint32_t at0 = uint32_t(row) * uint32_t(M + 1) + uint32_t(i0);
#pragma unroll
        for (int e = 0; e < E; ++e) {
          // both read, then chosen: chosen by address they would live in memory
          const cx<T> vs = S[e], va = A[e];
          o[at0 + uint32_t(F::template at<R>(e))] = cx<T>{s == 5 ? vs.x : va.x, s == 5 ? vs.y : va.y};
        }
      }
    }
  }
}

// Threads and rows of a launch.  Blocks of one wavefront where rows are short
// (64^3 reals: 4096 rows of 4 lanes are 256 wavefronts), of four else, which
// share a table; a wavefront takes up to 8 groups of rows one after the other
// (the table is read once for them) while 4096 blocks are left.
template <typename T, int N> struct RowLaunch {
  using F = RowFft<T, N / 2>;
  static constexpr int TH = N <= 64 ? 64 : 256, WAVES = TH / 64;
  static constexpr size_t LDS = sizeof(cx<T>) * (F::TABLE + WAVES * F::RPW * F::LEN);
  static int iters(long nrows, long jobs) {
    const long groups = (nrows + WAVES * F::RPW - 1) / (WAVES * F::RPW);
    return int(std::min(8l, std::max(1l, groups * jobs / 4096)));
  }
  static unsigned blocks(long nrows, int iters) {
    const long per = long(WAVES) * F::RPW * iters;
    return unsigned((nrows + per - 1) / per);
  }
};

}  // namespace gic
