// Entry points of the transforms, by size.  With GIC_FFT_SPLIT every size's
// passes are compiled in a unit of its own (fft_size.hip), without it all of
// them here.
#include "fft_api.h"
#include <cmath>
#include <string>
#ifndef GIC_FFT_SPLIT
#include "fft_fused.h"
#endif

namespace gic {

template <typename T> static const FftApi<T> &api(int n) {
  switch (n) {
    case 4: return fft_api<T, 4>();
    case 8: return fft_api<T, 8>();
    case 16: return fft_api<T, 16>();
    case 32: return fft_api<T, 32>();
    case 64: return fft_api<T, 64>();
    case 128: return fft_api<T, 128>();
    case 256: return fft_api<T, 256>();
    case 512: return fft_api<T, 512>();
    case 1024: return fft_api<T, 1024>();
  }
  throw std::runtime_error("FFT size " + std::to_string(n) + " is not supported (powers of two 4..1024)");
}

template <typename T> void fft3d(T *d, int n, int dir, hipStream_t st, TimingHook *hook) {
  if (dir < 0) {
    api<T>(n).r2c(d, nullptr, st, hook, nullptr);
  } else {
    api<T>(n).c2r(d, st, hook);
  }
}
template <typename T> void fft_r2c_post(T *d, int n, const T *post, hipStream_t st, TimingHook *hook, const T *src) {
  api<T>(n).r2c(d, post, st, hook, src);
}
template <typename T> void fft_r2c_batch(T *d, int n, int nb, const T *post, hipStream_t st, TimingHook *hook) {
  if (nb < 1) throw std::runtime_error("fft_r2c_batch: no fields");
  api<T>(n).r2c_batch(d, nb, post, st, hook);
}
template <typename T>
void fft_r2c_boxes(const T *rows, int n, long nrows, int nb, int wl, const int *winx, const int *winy, T *zbuf, T *ybuf,
                   T *spec, long spec_stride, const T *post, hipStream_t st, TimingHook *hook) {
  if (nb < 1 || wl < 1 || wl >= n) throw std::runtime_error("fft_r2c_boxes: bad box count or size");
  if (nrows < long(nb) * wl * wl) throw std::runtime_error("fft_r2c_boxes: bad row count");
  api<T>(n).r2c_boxes(rows, nrows, nb, wl, winx, winy, zbuf, ybuf, spec, spec_stride, post, st, hook);
}
template <typename T>
void fft_c2r_from(const T *spec, T *out, int n, int pre, const T *tab, double kmin, hipStream_t st,
                  TimingHook *hook) {
  api<T>(n).c2r_from(spec, out, pre, tab, kmin, st, hook);
}
template <typename T>
void fft_r2c_window_zy(const T *win, int n, const int *w0, const int *wl, T *bufB, T *bufA, hipStream_t st,
                       TimingHook *hook) {
  for (int a = 0; a < 3; ++a)
    if (wl[a] < 1 || wl[a] > n || w0[a] < 0 || w0[a] >= n) throw std::runtime_error("fft_r2c_window: bad window");
  api<T>(n).r2c_window_zy(win, w0, wl, bufB, bufA, st, hook);
}
template <typename T>
void fft_r2c_window(const T *win, int n, const int *w0, const int *wl, T *bufB, T *bufA, T *spec, const T *post,
                    bool accumulate, hipStream_t st, TimingHook *hook, const T *aux, const FilterInline *fil,
                    double kmin) {
  for (int a = 0; a < 3; ++a)
    if (wl[a] < 1 || wl[a] > n || w0[a] < 0 || w0[a] >= n) throw std::runtime_error("fft_r2c_window: bad window");
  if (aux && (!post || accumulate)) throw std::runtime_error("fft_r2c_window: aux needs a table and no accumulation");
  api<T>(n).r2c_window(win, w0, wl, bufB, bufA, spec, post, accumulate, st, hook, aux, fil, kmin);
}
template <typename T>
void fft_c2r_window(const T *spec, int n, int pre, const T *tab, double kmin, const int *w0, const int *wl,
                    T *bufA, T *bufB, T *out, hipStream_t st, TimingHook *hook, const FilterInline *fil) {
  for (int a = 0; a < 3; ++a)
    if (wl[a] < 1 || wl[a] > n || w0[a] < 0 || w0[a] >= n) throw std::runtime_error("fft_c2r_window: bad window");
  api<T>(n).c2r_window(spec, pre, tab, kmin, w0, wl, bufA, bufB, out, st, hook, fil);
}

template <typename T> void fft_x(const FftX<T> &x, int n, hipStream_t st, TimingHook *hook) {
  if (x.wlen < 0 || x.wlen > n || x.win0 < 0 || x.win0 >= n) throw std::runtime_error("fft_x: bad window");
  api<T>(n).x(x, st, hook);
}
template <typename T> void fft_y(const FftY<T> &y, int n, hipStream_t st, TimingHook *hook) {
  if (y.njob < 1 || y.njob > FFT_JOBS || y.nouter < 0 || y.nouter > n || y.wlen < 0 || y.wlen > n || y.win0 < 0 ||
      y.win0 >= n)
    throw std::runtime_error("fft_y: bad jobs or window");
  api<T>(n).y(y, st, hook);
}
template <typename T> void fft_z(const FftZ<T> &z, int n, hipStream_t st, TimingHook *hook) {
  if (z.njob < 1 || z.njob > FFT_JOBS) throw std::runtime_error("fft_z: bad jobs");
  api<T>(n).z(z, st, hook);
}
template <typename T>
void fft_z_window(const T *in, T *out, long nrows, int z0, int wz, int n, hipStream_t st, TimingHook *hook) {
  if (nrows < 1 || wz < 1 || wz > n || z0 < 0 || z0 >= n) throw std::runtime_error("fft_z_window: bad window");
  api<T>(n).z_window(in, out, nrows, z0, wz, st, hook);
}
template <typename T> void fft_z_forward(const FftZFwd<T> &z, int n, hipStream_t st, TimingHook *hook) {
  if (z.njob < 1 || z.njob > FFT_JOBS) throw std::runtime_error("fft_z_forward: bad jobs");
  api<T>(n).z_forward(z, st, hook);
}
template <typename T> void fft_y_forward(const FftYFwd<T> &y, int n, hipStream_t st, TimingHook *hook) {
  if (y.njob < 1 || y.njob > FFT_JOBS) throw std::runtime_error("fft_y_forward: bad jobs");
  api<T>(n).y_forward(y, st, hook);
}
template <typename T> void fft_x_adjoint(const FftXAdj<T> &x, int n, hipStream_t st, TimingHook *hook) {
  api<T>(n).x_adjoint(x, st, hook);
}
template <typename T>
void fft_r2c_z_window(const T *win, T *out, long nrows, int z0, int wz, int n, hipStream_t st, TimingHook *hook) {
  if (nrows < 1 || wz < 1 || wz > n || z0 < 0 || z0 >= n) throw std::runtime_error("fft_r2c_z_window: bad window");
  api<T>(n).r2c_z_window(win, out, nrows, z0, wz, st, hook);
}
template <typename T>
void fft_z_lpt(T *px, T *py, T *pz, const T *xx, const T *yy, const T *xy, T *S, bool psi, int n, double kmin,
               hipStream_t st, TimingHook *hook) {
  api<T>(n).z_lpt(px, py, pz, xx, yy, xy, S, psi, kmin, st, hook);
}

#define GIC_FFT_INST(T)                                                                                     \
  template void fft_x<T>(const FftX<T> &, int, hipStream_t, TimingHook *);                                  \
  template void fft_y<T>(const FftY<T> &, int, hipStream_t, TimingHook *);                                  \
  template void fft_z<T>(const FftZ<T> &, int, hipStream_t, TimingHook *);                                  \
  template void fft_z_window<T>(const T *, T *, long, int, int, int, hipStream_t, TimingHook *);             \
  template void fft_z_forward<T>(const FftZFwd<T> &, int, hipStream_t, TimingHook *);                       \
  template void fft_y_forward<T>(const FftYFwd<T> &, int, hipStream_t, TimingHook *);                       \
  template void fft_x_adjoint<T>(const FftXAdj<T> &, int, hipStream_t, TimingHook *);                       \
  template void fft_r2c_z_window<T>(const T *, T *, long, int, int, int, hipStream_t, TimingHook *);         \
  template void fft_z_lpt<T>(T *, T *, T *, const T *, const T *, const T *, T *, bool, int, double,         \
                             hipStream_t, TimingHook *);                                                     \
  template void fft_r2c_post<T>(T *, int, const T *, hipStream_t, TimingHook *, const T *);                 \
  template void fft_r2c_batch<T>(T *, int, int, const T *, hipStream_t, TimingHook *);                      \
  template void fft_r2c_boxes<T>(const T *, int, long, int, int, const int *, const int *, T *, T *, T *, long,  \
                                 const T *, hipStream_t, TimingHook *);                                       \
  template void fft_c2r_from<T>(const T *, T *, int, int, const T *, double, hipStream_t, TimingHook *);      \
  template void fft_r2c_window_zy<T>(const T *, int, const int *, const int *, T *, T *, hipStream_t, TimingHook *); \
  template void fft_r2c_window<T>(const T *, int, const int *, const int *, T *, T *, T *, const T *, bool,      \
                                  hipStream_t, TimingHook *, const T *, const FilterInline *, double);         \
  template void fft_c2r_window<T>(const T *, int, int, const T *, double, const int *, const int *, T *, T *, \
                                  T *, hipStream_t, TimingHook *, const FilterInline *);
GIC_FFT_INST(float)
GIC_FFT_INST(double)

template void fft3d<float>(float *, int, int, hipStream_t, TimingHook *);
template void fft3d<double>(double *, int, int, hipStream_t, TimingHook *);

}  // namespace gic
