// 3D FFT entry points and the per-kernel event timer hook.
#pragma once
#include "gic_common.h"

namespace gic {

// Called around every kernel launch when event timing is enabled; the
// implementation records hipEvents on the launch stream.
struct TimingHook {
  virtual ~TimingHook() = default;
  virtual void begin(const char *name, hipStream_t st) = 0;
  virtual void end(const char *name, hipStream_t st) = 0;
  // the algorithmic HBM bytes of one launch under this name: each input
  // element read once, each output element written once (reads of an
  // accumulated output counted too); tables and indices are not counted
  virtual void bytes(const char *, double) {}
};

// In-place 3D transform of a padded field (N*N*(N+2) reals of type T).
// dir < 0: r2c (real -> FFTW layout), dir > 0: c2r (with Hermitian mirroring
// of the kz = 0, N/2 planes).  Both directions scale by N^-1.5, as
// FieldFourierManager::performTransform does.
template <typename T> void fft3d(T *d, int n, int dir, hipStream_t st, TimingHook *hook);

// k-space operators applied inside the x pass
enum { FFT_PRE_NONE = 0, FFT_PRE_TABLE = 1 };

// A product of Fermi level filters, formed inside a transform's pass instead
// of read from a |k|^2 table (used by FP32 transforms, whose table reads are
// scattered): scale * prod_i f_i(k), f = LP, sqrt(1 - LP^2) or 1 - LP for
// kind 0, 1, 2 with LP = 1 / (1 + exp((k - kc) / (0.1 kc))); over_k2 divides
// by k^2 (0 at k = 0); zero makes every factor 0.  nf < 0: not given.
// the most factors a FilterInline may hold (more: use a table)
constexpr int FILTER_INLINE_MAX = 4;
struct FilterInline {
  int nf = -1;
  int kind[8];
  double kc[8];
  double scale = 1.0;
  int over_k2 = 0;
  int zero = 0;
};

// r2c whose last pass multiplies each mode by post[kx^2+ky^2+kz^2] (if non-null).
// With src non-null the real input is read from the dense n^3 array src (z
// fastest, no padding) and the spectrum lands in d.
template <typename T>
void fft_r2c_post(T *d, int n, const T *post, hipStream_t st, TimingHook *hook, const T *src = nullptr);
// r2c of nb padded n^3 fields stored back to back, each mode times post[|k|^2] if post is given
template <typename T> void fft_r2c_batch(T *d, int n, int nb, const T *post, hipStream_t st, TimingHook *hook);
// r2c of nb fields that vanish outside boxes of wl x wl cells in (x, y), all
// z: box b starts at (winx[b], winy[b]) mod n (device int arrays).  rows
// holds the boxes' rows as dense rows of n reals, row (b wl + i) wl + j for
// x = winx[b]+i, y = winy[b]+j; nrows >= nb wl^2, rows past those are
// transformed but unused.
// zbuf (nrows (n/2+1) complex) and ybuf (nb wl n (n/2+1) complex) are
// scratch; field b's spectrum times post[|k|^2] goes to spec + b spec_stride.
template <typename T>
void fft_r2c_boxes(const T *rows, int n, long nrows, int nb, int wl, const int *winx, const int *winy, T *zbuf, T *ybuf,
                   T *spec, long spec_stride, const T *post, hipStream_t st, TimingHook *hook);
// out <- c2r(op(spec)), out-of-place from a spectrum that is left untouched.
// op: FFT_PRE_TABLE multiplies by tab[|k|^2].
template <typename T>
void fft_c2r_from(const T *spec, T *out, int n, int pre, const T *tab, double kmin, hipStream_t st, TimingHook *hook);
// Factors of (k_y, k_z) that the fused y and z passes multiply a field by
enum {
  FFT_YZ_ONE = 0,    // 1
  FFT_YZ_IKY = 1,    // i k_y (0 at k_y = +Nyquist)
  FFT_YZ_IKZ = 2,    // i k_z (0 at k_z = +Nyquist)
  FFT_YZ_MIKY = 3,   // -i k_y (0 at k_y = +Nyquist)
  FFT_YZ_KYKY = 4,   // k_y^2
  FFT_YZ_KY = 5      // k_y (0 at k_y = +Nyquist)
};
// ---- fused passes (fft_fused.h) ----------------------------------------------------
// Fields are padded (n * n * (n + 2) values of T); nb of them form a batch,
// *_bs values apart.

// One pass along x over a spectrum, or (forward) over fields transformed
// along z and y, which are transformed along x first, scaled by n^-1.5 and
// post[|k|^2] (if given) and stored as the spectrum spec (if given).  Of the
// spectrum m it makes the inverse x transforms
//   out[0]: m (times the filter alone with plain0)   out[1]: f m
//   out[2]: i k_x f m (0 at +Nyquist)                  out[3]: k_x^2 f m
// (those not null), f the table tab[|k|^2], the filter product fil in its place
// (FP32), or inv_k2 / (|k|^2 kmin^2) (0 at k = 0).  plain0: fil holds a filter over k^2 and tab0 the filter's table.
// With wlen > 0 the outputs keep the points [win0, win0 + wlen) mod n, as
// wlen planes; with iwlen > 0 (forward) the input is the iwlen planes from
// iwin0 on of fields that are 0 elsewhere.  Outputs may be the input where
// their windows are the same.
constexpr int FFT_JOBS = 6;
template <typename T> struct FftX {
  const T *in = nullptr;
  bool forward = false;
  T *spec = nullptr, *out[4] = {nullptr, nullptr, nullptr, nullptr};
  long in_bs = 0, spec_bs = 0, out_bs = 0;
  int nb = 1;
  const T *post = nullptr, *tab = nullptr, *tab0 = nullptr;
  const FilterInline *fil = nullptr;
  bool plain0 = false;
  double inv_k2 = 0, kmin = 0;
  int win0 = 0, wlen = 0, iwin0 = 0, iwlen = 0;
};
template <typename T> void fft_x(const FftX<T> &x, int n, hipStream_t st, TimingHook *hook);

// Inverse y passes: each job's input (of nouter planes, 0: n) times factors
// FFT_YZ_*, up to three outputs (the first null one ends them).  With
// wlen > 0 the outputs keep the points [win0, win0 + wlen) mod n of each
// plane.  An output may be its job's input.
template <typename T> struct FftY {
  struct Job {
    const T *in;
    T *out[3];
    int op[3];
  } job[FFT_JOBS] = {};
  int njob = 0, nb = 1, nouter = 0, win0 = 0, wlen = 0;
  long in_bs = 0, out_bs = 0;
  double kmin = 0;
  void add(const T *in, T *o0, int p0, T *o1 = nullptr, int p1 = 0, T *o2 = nullptr, int p2 = 0) {
    job[njob++] = Job{in, {o0, o1, o2}, {p0, p1, p2}};
  }
};
template <typename T> void fft_y(const FftY<T> &y, int n, hipStream_t st, TimingHook *hook);

// c2r along z, scaled by scale n^-1.5: each job's complex rows times FFT_YZ_ONE
// or FFT_YZ_IKZ to a padded field, a dense array or both
template <typename T> struct FftZ {
  struct Job {
    const T *in;
    T *out, *dense;
    int op;
  } job[FFT_JOBS] = {};
  int njob = 0, nb = 1;
  long in_bs = 0, out_bs = 0, dense_bs = 0;
  double kmin = 0, scale = 1;
  void add(const T *in, T *out, T *dense, int op) { job[njob++] = Job{in, out, dense, op}; }
};
template <typename T> void fft_z(const FftZ<T> &z, int n, hipStream_t st, TimingHook *hook);

// c2r along z of nrows complex rows into the points [z0, z0 + wz) mod n of each
template <typename T>
void fft_z_window(const T *in, T *out, long nrows, int z0, int wz, int n, hipStream_t st, TimingHook *hook);

// r2c along z of each job's padded (dense false) or dense field
template <typename T> struct FftZFwd {
  struct Job {
    const T *src;
    T *out;
    bool dense;
  } job[FFT_JOBS] = {};
  int njob = 0, nb = 1;
  long src_bs = 0, out_bs = 0;
  void add(const T *src, T *out, bool dense) { job[njob++] = Job{src, out, dense}; }
};
template <typename T> void fft_z_forward(const FftZFwd<T> &z, int n, hipStream_t st, TimingHook *hook);

// forward y passes: out = Y in, or with a second input -i k_y Y in - i k_z Y in2.
// With iwlen > 0 each of the nouter input planes holds the iwlen rows from
// iwin0 on and is 0 elsewhere.
template <typename T> struct FftYFwd {
  struct Job {
    const T *in, *in2;
    T *out;
  } job[FFT_JOBS] = {};
  int njob = 0, nb = 1, nouter = 0, iwin0 = 0, iwlen = 0;
  long bs = 0;
  double kmin = 0;
  void add(const T *in, const T *in2, T *out) { job[njob++] = Job{in, in2, out}; }
};
template <typename T> void fft_y_forward(const FftYFwd<T> &y, int n, hipStream_t st, TimingHook *hook);

// out <- inverse x transform of tab[|k|^2] n^-1.5 (-i k_x X h1 + X h0), plus the
// same of g1, g0 with gtab if given (X the forward x transform).  With
// iwlen > 0 the inputs are the iwlen planes from iwin0 on of fields that are 0
// elsewhere; without, out may be h1.
template <typename T> struct FftXAdj {
  T *out = nullptr;
  const T *h1 = nullptr, *h0 = nullptr, *tab = nullptr, *g1 = nullptr, *g0 = nullptr, *gtab = nullptr;
  int iwin0 = 0, iwlen = 0;
  double kmin = 0;
};
template <typename T> void fft_x_adjoint(const FftXAdj<T> &x, int n, hipStream_t st, TimingHook *hook);
// r2c along z of nrows rows given as their points [z0, z0 + wz) mod n, 0 elsewhere
template <typename T>
void fft_r2c_z_window(const T *win, T *out, long nrows, int z0, int wz, int n, hipStream_t st, TimingHook *hook);

// The z passes of the second-order source S = xx yy + (xx + yy) zz - xy^2 -
// xz^2 - yz^2, and with psi of the displacements over px, py, pz, from the
// fields transformed along x and y of X0 = x pass of f m, X1 of i k_x f m, X2
// of k_x^2 f m: px = y(X1), py = y(k_y X0), pz = y(X0), xx = y(X2),
// yy = y(k_y^2 X0), xy = y(-i k_y X1)
template <typename T>
void fft_z_lpt(T *px, T *py, T *pz, const T *xx, const T *yy, const T *xy, T *S, bool psi, int n, double kmin,
               hipStream_t st, TimingHook *hook);

// Spectrum (r2c, N^-1.5) of a field that is zero outside the real-space window
// [w0, w0+wl) (per axis, wrapping mod n), given as the dense window win
// (wl[0]*wl[1]*wl[2] reals, z fastest): pruned z and y passes and a full x
// pass that scales by post[|k|^2] (if non-null) and stores into, or with
// accumulate adds to, the padded spectrum spec.  bufB holds
// wl[0]*wl[1]*(n+2) reals, bufA wl[0]*n*(n/2+1) complex.
// With aux (a spectrum of the same layout) the result is spec = post * aux +
// r2c(win) instead: post then scales aux, not the transform.
template <typename T>
void fft_r2c_window(const T *win, int n, const int *w0, const int *wl, T *bufB, T *bufA, T *spec, const T *post,
                    bool accumulate, hipStream_t st, TimingHook *hook, const T *aux = nullptr,
                    const FilterInline *fil = nullptr, double kmin = 0);
// its z and y passes alone: bufA <- the window's planes transformed along z and y
template <typename T>
void fft_r2c_window_zy(const T *win, int n, const int *w0, const int *wl, T *bufB, T *bufA, hipStream_t st,
                       TimingHook *hook);
// Only the real-space window [w0, w0+wl) (per axis, wrapping mod n) of
// c2r(op(spec)), via pruned passes: bufA holds wl[0]*n*(n/2+1) complex,
// bufB wl[0]*wl[1]*(n/2+1) complex, out wl[0]*wl[1]*wl[2] reals.
template <typename T>
void fft_c2r_window(const T *spec, int n, int pre, const T *tab, double kmin, const int *w0, const int *wl,
                    T *bufA, T *bufB, T *out, hipStream_t st, TimingHook *hook, const FilterInline *fil = nullptr);

}  // namespace gic
