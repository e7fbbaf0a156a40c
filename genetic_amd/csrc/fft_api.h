// The passes of one precision and size, as a table of functions (see FftN in
// fft_passes.h for what each does).
#pragma once
#include "fft.h"

namespace gic {

template <typename T> struct FftApi {
  void (*r2c)(T *d, const T *post, hipStream_t st, TimingHook *hook, const T *src);
  void (*r2c_batch)(T *d, int nb, const T *post, hipStream_t st, TimingHook *hook);
  void (*r2c_boxes)(const T *rows, long nrows, int nb, int wl, const int *winx, const int *winy, T *zbuf, T *ybuf,
                    T *spec, long spec_stride, const T *post, hipStream_t st, TimingHook *hook);
  void (*c2r)(T *d, hipStream_t st, TimingHook *hook);
  void (*c2r_from)(const T *spec, T *out, int pre, const T *tab, double kmin, hipStream_t st, TimingHook *hook);
  void (*c2r_window)(const T *spec, int pre, const T *tab, double kmin, const int *w0, const int *wl, T *bufA,
                     T *bufB, T *out, hipStream_t st, TimingHook *hook, const FilterInline *fil);
  void (*r2c_window)(const T *win, const int *w0, const int *wl, T *bufB, T *bufA, T *spec, const T *post, bool accum,
                     hipStream_t st, TimingHook *hook, const T *aux, const FilterInline *fil, double kmin);
  void (*r2c_window_zy)(const T *win, const int *w0, const int *wl, T *bufB, T *bufA, hipStream_t st, TimingHook *hook);
  void (*r2c_z_window)(const T *win, T *out, long nrows, int z0, int wz, hipStream_t st, TimingHook *hook);
  void (*z_window)(const T *in, T *out, long nrows, int z0, int wz, hipStream_t st, TimingHook *hook);
  // fused passes
  void (*x)(const FftX<T> &q, hipStream_t st, TimingHook *hook);
  void (*y)(const FftY<T> &q, hipStream_t st, TimingHook *hook);
  void (*y_forward)(const FftYFwd<T> &q, hipStream_t st, TimingHook *hook);
  void (*x_adjoint)(const FftXAdj<T> &q, hipStream_t st, TimingHook *hook);
  void (*z)(const FftZ<T> &q, hipStream_t st, TimingHook *hook);
  void (*z_forward)(const FftZFwd<T> &q, hipStream_t st, TimingHook *hook);
  void (*z_lpt)(T *px, T *py, T *pz, const T *xx, const T *yy, const T *xy, T *S, bool psi, double kmin,
                hipStream_t st, TimingHook *hook);
};

template <typename T, int N> const FftApi<T> &fft_api();

}  // namespace gic
