#pragma once
// The transforms of one precision and size (FftN), built of the strided
// passes and the row passes, and the mirroring of the Hermitian planes.
#include "fft_rows.h"

namespace gic {

// ---- Hermitian mirror of the kz=0 and kz=N/2 planes ------------------------------
// ensureFourierModesAreMirrored (fourier.hpp:331-357): for kx in [0,N/2] and
// ky from N/2 down to -N/2+1 the conjugate of mode (kx,ky) is copied into
// (-kx,-ky).  Equivalent closed form: a destination (kx',ky') with kx' > N/2,
// or kx' in {0,N/2} and ky' > N/2 receives conj(mode(-kx',-ky')); the
// self-conjugate modes get their imaginary part negated.
template <typename T>
__global__ void k_mirror_planes(cx<T> *data, int n) {
  int nz = n / 2 + 1;
  long t = long(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= long(n) * n) return;
  int kx = int(t / n), ky = int(t % n);
  int h = n / 2;
  int sx = (n - kx) % n, sy = (n - ky) % n;
  bool xedge = (kx == 0 || kx == h);
  bool dest = kx > h || (xedge && ky > h);
  bool self = xedge && (ky == 0 || ky == h);
  for (int kz : {0, h}) {
    if (dest) {
      cx<T> s = data[(long(sx) * n + sy) * nz + kz];
      data[(long(kx) * n + ky) * nz + kz] = cx<T>{s.x, -s.y};
    } else if (self) {
      cx<T> &v = data[(long(kx) * n + ky) * nz + kz];
      v.y = -v.y;
    }
  }
}

// ----------------------------------------------------------------------------------
template <typename T> struct TwTable {
  std::map<int, cx<T> *> tabs;
  std::mutex mu;
  const cx<T> *get(int n) {
    std::lock_guard<std::mutex> g(mu);
    auto it = tabs.find(n);
    if (it != tabs.end()) return it->second;
    std::vector<cx<T>> h(n);
    for (int k = 0; k < n; ++k) {
      // FP64-generated twiddles, rounded to T
      double a = -2.0 * M_PI * double(k) / double(n);
      h[k] = cx<T>{T(cos(a)), T(sin(a))};
    }
    cx<T> *d = nullptr;
    GIC_HIP(hipMalloc(&d, sizeof(cx<T>) * n));
    GIC_HIP(hipMemcpy(d, h.data(), sizeof(cx<T>) * n, hipMemcpyHostToDevice));
    tabs[n] = d;
    return d;
  }
};
template <typename T> TwTable<T> &twtable() {
  static TwTable<T> t;
  return t;
}

// Tile shape of the strided passes: the tuned table, or one shape for every
// size when a tuning build names it (GIC_TUNE_THREADS, GIC_TUNE_COLS).
template <typename T, int N> constexpr int strided_threads() {
#ifdef GIC_TUNE_THREADS
  return GIC_TUNE_THREADS;
#else
  return TileShape<T, N>::threads;
#endif
}
template <typename T, int N> constexpr int strided_cols() {
#ifdef GIC_TUNE_COLS
  return sizeof(T) == 4 ? GIC_TUNE_COLS : (GIC_TUNE_COLS > 8 ? 8 : GIC_TUNE_COLS);
#else
  return TileShape<T, N>::cols;
#endif
}

// y passes' tile shape: YTileShape where fft_tiles.h gives one, else the
// x passes'
template <typename T, int N, class = void> struct YShape {
  static constexpr int threads = strided_threads<T, N>();
  static constexpr int cols = strided_cols<T, N>();
};
#ifndef GIC_TUNE_THREADS   // the tuner times one shape for every pass
template <typename T, int N> struct YShape<T, N, std::void_t<decltype(YTileShape<T, N>::cols)>> {
  static constexpr int threads = YTileShape<T, N>::threads;
  static constexpr int cols = YTileShape<T, N>::cols;
};
#endif

template <typename T, int N> struct FftN {
  static constexpr int C = strided_cols<T, N>();
  static constexpr int M = N / 2;
  static constexpr int NZ = N / 2 + 1;
  using Rows = RowLaunch<T, N>;

  static constexpr int STHREADS = strided_threads<T, N>();
  // FP32: the factor's filter and 1/k^2 in single precision
  static void prepare_factor(StridedArgs<T> &a) {
    a.ff.nf = -1;
    if (sizeof(T) == 4) {
      if (a.fil.nf >= 0) {
        if (a.fil.nf > FILTER_INLINE_MAX) throw std::runtime_error("FilterInline: at most 4 factors");
        a.ff.nf = a.fil.nf;
        a.ff.zero = a.fil.zero;
        a.ff.over_k2 = a.fil.over_k2;
        for (int i = 0; i < a.fil.nf; ++i) {
          a.ff.kind[i] = a.fil.kind[i];
          a.ff.kc[i] = float(a.fil.kc[i]);
          a.ff.inv_w[i] = 1.f / (float(a.fil.kc[i]) * 0.1f);
        }
        a.ff.scale = float(a.fil.scale);
        a.ff.kmin = float(a.kmin_d);
        a.ff.inv_kmin2 = a.kmin_d > 0 ? float(1.0 / (a.kmin_d * a.kmin_d)) : 0.f;
      }
      a.inv_k2_f = a.kmin_d > 0 ? float(a.inv_k2 / (a.kmin_d * a.kmin_d)) : 0.f;
    }
  }
  template <int DIR, int PRE, int POST, int PASS = 0>
  static void strided(const StridedArgs<T> &a0, int nouter, hipStream_t st, TimingHook *hook, const char *name) {
    constexpr bool YP = PASS == 1 || PASS == 3 || PASS == 5;
    constexpr int CP = YP ? YShape<T, N>::cols : C;
    constexpr int TP = YP ? YShape<T, N>::threads : STHREADS;
    StridedArgs<T> a = a0;
    prepare_factor(a);
    a.ncol = NZ;
    a.nkzb = (NZ + CP - 1) / CP;
    a.n = N;
    a.nouter = nouter;
    int nblk = nouter * a.nkzb * (a.nbatch > 1 ? a.nbatch : 1);
    size_t shm = sizeof(cx<T>) * (CP + 1) * N;   // the tile, then the line's twiddles
    const cx<T> *tw = twtable<T>().get(N);
    auto kern = k_fft_strided<T, N, CP, DIR, TP, PRE, POST, PASS>;
    if (shm > 65536) GIC_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
    std::string tag = std::string(name) + "." + std::to_string(N);
    if (hook) {
      hook->begin(tag.c_str(), st);
      // lines of the pass; a pruned input or output moves only its window
      double lines = double(nouter) * NZ * (a.nbatch > 1 ? a.nbatch : 1);
      double rd = lines * ((a.in_wlen > 0 && a.in_wlen < N) ? a.in_wlen : N);
      double wr = lines * (a.wlen < N ? a.wlen : N);
      bool reads_out = a.accum || POST == POST_AUX;   // accumulated output, or the spectrum it adds
      hook->bytes(tag.c_str(), sizeof(cx<T>) * (rd + wr + (reads_out ? wr : 0.0)));
    }
    hipLaunchKernelGGL(kern, dim3(nblk), dim3(TP), shm, st, a, tw);
    GIC_HIP(hipGetLastError());
    if (hook) hook->end(tag.c_str(), st);
  }
  // in-place plain pass over a full field: y (line stride NZ) or x (line stride N*NZ)
  static StridedArgs<T> plain(cx<T> *d, bool xpass, T scale) {
    StridedArgs<T> a{};
    a.in = d;
    a.out = d;
    a.in_ls = a.out_ls = xpass ? long(N) * NZ : NZ;
    a.in_os = a.out_os = xpass ? NZ : long(N) * NZ;
    a.tab = nullptr;
    a.win0 = 0;
    a.wlen = N;
    a.in_win0 = 0;
    a.in_wlen = N;
    a.scale = scale;
    return a;
  }
  template <class K, class A>
  static void rows_launch(K kern, const A &a, int jobs, int nb, const char *name, double bytes, hipStream_t st,
                          TimingHook *hook) {
    if (Rows::LDS > 65536)
      GIC_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)Rows::LDS));
    std::string tag;
    if (hook) {
      tag = std::string(name) + "." + std::to_string(N);
      hook->begin(tag.c_str(), st);
      hook->bytes(tag.c_str(), bytes);
    }
    hipLaunchKernelGGL(kern, dim3(Rows::blocks(a.nrows, a.iters), jobs, nb), dim3(Rows::TH), Rows::LDS, st, a,
                       twtable<T>().get(N));
    GIC_HIP(hipGetLastError());
    if (hook) hook->end(tag.c_str(), st);
  }
  // r2c (dir < 0) or c2r of nrows padded rows of d; src (if non-null) holds
  // the dense rows that the r2c reads
  static void zpass(T *d, T scale, int dir, long nrows, hipStream_t st, TimingHook *hook, const char *name,
                    const T *src = nullptr) {
    const double bytes = double(nrows) * (2 * N + 2) * sizeof(T);   // N reals one way, N+2 the other
    if (dir < 0) {
      ZFwdArgs<T> a{};
      a.job[0] = {src ? src : d, d, src ? long(N) : long(N + 2)};
      a.nrows = nrows;
      a.iters = Rows::iters(nrows, 1);
      rows_launch(k_fft_z_r2c<T, N, Rows::TH, false>, a, 1, 1, name, bytes, st, hook);
    } else {
      ZArgs<T> a{};
      a.job[0] = {d, d, nullptr, FFT_YZ_ONE};
      a.nrows = nrows;
      a.iters = Rows::iters(nrows, 1);
      a.scale = scale;
      rows_launch(k_fft_z_c2r<T, N, Rows::TH, false>, a, 1, 1, name, bytes, st, hook);
    }
  }
  static T norm() { return T(1.0 / pow(double(N), 1.5)); }
  static void mirror(cx<T> *c, hipStream_t st, TimingHook *hook) {
    int nt = 256;
    long nn = long(N) * N;
    std::string tag = "fft_mirror." + std::to_string(N);
    if (hook) {
      hook->begin(tag.c_str(), st);
      hook->bytes(tag.c_str(), 2.0 * nn * sizeof(cx<T>));   // half of two planes read, half written
    }
    hipLaunchKernelGGL(k_mirror_planes<T>, dim3((nn + nt - 1) / nt), dim3(nt), 0, st, c, N);
    GIC_HIP(hipGetLastError());
    if (hook) hook->end(tag.c_str(), st);
  }
  static void r2c(T *d, const T *post, hipStream_t st, TimingHook *hook, const T *src = nullptr) {
    cx<T> *c = reinterpret_cast<cx<T> *>(d);
    zpass(d, T(1), -1, long(N) * N, st, hook, "fft_z_r2c", src);
    strided<-1, PRE_NONE, POST_NONE, 1>(plain(c, false, T(1)), N, st, hook, "fft_y_fwd");
    StridedArgs<T> ax = plain(c, true, norm());
    if (post) {
      ax.tab = post;
      strided<-1, PRE_NONE, POST_TABLE>(ax, N, st, hook, "fft_x_post");
    } else {
      strided<-1, PRE_NONE, POST_NONE>(ax, N, st, hook, "fft_x_fwd");
    }
  }
  // r2c of nb padded fields stored back to back (no dense source), the
  // post table applied by the last pass of each
  static void r2c_batch(T *d, int nb, const T *post, hipStream_t st, TimingHook *hook) {
    cx<T> *c = reinterpret_cast<cx<T> *>(d);
    long fs = long(N) * N * NZ;
    zpass(d, T(1), -1, long(N) * N * nb, st, hook, "fft_z_r2c_batch");
    StridedArgs<T> ay = plain(c, false, T(1));
    ay.nbatch = nb;
    ay.in_bs = ay.out_bs = fs;
    strided<-1, PRE_NONE, POST_NONE, 1>(ay, N, st, hook, "fft_y_fwd_batch");
    StridedArgs<T> ax = plain(c, true, norm());
    ax.nbatch = nb;
    ax.in_bs = ax.out_bs = fs;
    if (post) {
      ax.tab = post;
      strided<-1, PRE_NONE, POST_TABLE>(ax, N, st, hook, "fft_x_post_batch");
    } else {
      strided<-1, PRE_NONE, POST_NONE>(ax, N, st, hook, "fft_x_fwd_batch");
    }
  }
  // r2c of nb fields that are zero outside a box of wl x wl cells in (x, y)
  // (all z), box b starting at (winx[b], winy[b]) (mod N; device arrays).
  // rows: the boxes' rows, nrows dense rows of N reals,
  // row (b wl + i) wl + j holding x = winx[b]+i, y = winy[b]+j; zbuf (nrows
  // rows of NZ complex) and ybuf (nb wl N NZ complex) are scratch.  Field b's
  // spectrum, times post[|k|^2], goes to spec + b * spec_stride (complex).
  static void r2c_boxes(const T *rows, long nrows, int nb, int wl, const int *winx, const int *winy, T *zbuf,
                        T *ybuf, T *spec, long spec_stride, const T *post, hipStream_t st, TimingHook *hook) {
    zpass(zbuf, T(1), -1, nrows, st, hook, "fft_z_r2c_boxes", rows);
    // y pass: per field, tiles (i, kz block), lines over ky from the wl rows j
    StridedArgs<T> ay{};
    ay.in = reinterpret_cast<const cx<T> *>(zbuf);
    ay.out = reinterpret_cast<cx<T> *>(ybuf);
    ay.in_ls = NZ;
    ay.in_os = long(wl) * NZ;
    ay.out_ls = NZ;
    ay.out_os = long(N) * NZ;
    ay.win0 = 0;
    ay.wlen = N;
    ay.in_win0 = 0;
    ay.in_wlen = wl;
    ay.scale = T(1);
    ay.nbatch = nb;
    ay.in_bs = long(wl) * wl * NZ;
    ay.out_bs = long(wl) * N * NZ;
    ay.in_win0_b = winy;
    strided<-1, PRE_NONE, POST_NONE, 5>(ay, wl, st, hook, "fft_y_fwd_boxes");
    // x pass: per field, tiles (ky, kz block), lines over kx from the wl planes i
    StridedArgs<T> ax{};
    ax.in = reinterpret_cast<const cx<T> *>(ybuf);
    ax.out = reinterpret_cast<cx<T> *>(spec);
    ax.in_ls = long(N) * NZ;
    ax.in_os = NZ;
    ax.out_ls = long(N) * NZ;
    ax.out_os = NZ;
    ax.win0 = 0;
    ax.wlen = N;
    ax.in_win0 = 0;
    ax.in_wlen = wl;
    ax.scale = norm();
    ax.tab = post;
    ax.nbatch = nb;
    ax.in_bs = long(wl) * N * NZ;
    ax.out_bs = spec_stride;
    ax.in_win0_b = winx;
    if (post) strided<-1, PRE_NONE, POST_TABLE, 4>(ax, N, st, hook, "fft_x_fwd_boxes");
    else strided<-1, PRE_NONE, POST_NONE, 4>(ax, N, st, hook, "fft_x_fwd_boxes");
  }
  static void c2r(T *d, hipStream_t st, TimingHook *hook) {
    cx<T> *c = reinterpret_cast<cx<T> *>(d);
    mirror(c, st, hook);
    strided<+1, PRE_NONE, POST_NONE>(plain(c, true, T(1)), N, st, hook, "fft_x");
    strided<+1, PRE_NONE, POST_NONE, 1>(plain(c, false, T(1)), N, st, hook, "fft_y");
    zpass(d, norm(), +1, long(N) * N, st, hook, "fft_z_c2r");
  }
  // out <- c2r(op(spec)) with op applied while the x pass reads the spectrum
  static void c2r_from(const T *spec, T *out, int pre, const T *tab, double kmin, hipStream_t st, TimingHook *hook) {
    const cx<T> *ci = reinterpret_cast<const cx<T> *>(spec);
    cx<T> *co = reinterpret_cast<cx<T> *>(out);
    StridedArgs<T> ax = plain(co, true, T(1));
    ax.in = ci;
    ax.tab = tab;
    ax.kmin_d = kmin;
    if (!tab && pre != PRE_NONE) throw std::runtime_error("c2r_from: operator without a table");
    if (pre == PRE_TABLE) strided<+1, PRE_TABLE, POST_NONE>(ax, N, st, hook, "fft_x_pre");
    else strided<+1, PRE_NONE, POST_NONE>(ax, N, st, hook, "fft_x");
    strided<+1, PRE_NONE, POST_NONE, 1>(plain(co, false, T(1)), N, st, hook, "fft_y");
    zpass(out, norm(), +1, long(N) * N, st, hook, "fft_z_c2r");
  }
  // real-space window [w0, w0+wl) (per axis, mod N) of c2r(op(spec)):
  // bufA holds wl[0] x-planes after the x pass, bufB wl[0]*wl[1] rows after
  // the y pass; out receives wl[0]*wl[1]*wl[2] reals.
  static void c2r_window(const T *spec, int pre, const T *tab, double kmin, const int *w0, const int *wl, T *bufA,
                         T *bufB, T *out, hipStream_t st, TimingHook *hook, const FilterInline *fil = nullptr) {
    const cx<T> *ci = reinterpret_cast<const cx<T> *>(spec);
    cx<T> *ca = reinterpret_cast<cx<T> *>(bufA);
    cx<T> *cb = reinterpret_cast<cx<T> *>(bufB);
    // x pass: tiles (ky, kz block), lines over kx, keep x in window; A = [wl0][N][NZ]
    StridedArgs<T> ax{};
    ax.in = ci;
    ax.out = ca;
    ax.in_ls = long(N) * NZ;
    ax.in_os = NZ;
    ax.out_ls = long(N) * NZ;
    ax.out_os = NZ;
    ax.tab = tab;
    ax.kmin_d = kmin;
    if (fil) ax.fil = *fil;
    ax.win0 = w0[0];
    ax.wlen = wl[0];
    ax.scale = T(1);
    if (pre == PRE_TABLE) {
      strided<+1, PRE_TABLE, POST_NONE, 2>(ax, N, st, hook, "fft_x_pre_win");
    } else {
      strided<+1, PRE_NONE, POST_NONE, 2>(ax, N, st, hook, "fft_x_win");
    }
    // y pass: tiles (x_local, kz block), lines over ky, keep y in window; B = [wl0][wl1][NZ]
    StridedArgs<T> ay{};
    ay.in = ca;
    ay.out = cb;
    ay.in_ls = NZ;
    ay.in_os = long(N) * NZ;
    ay.out_ls = NZ;
    ay.out_os = long(wl[1]) * NZ;
    ay.tab = nullptr;
    ay.win0 = w0[1];
    ay.wlen = wl[1];
    ay.scale = T(1);
    strided<+1, PRE_NONE, POST_NONE, 3>(ay, wl[0], st, hook, "fft_y_win");
    z_window(bufB, out, long(wl[0]) * wl[1], w0[2], wl[2], st, hook);
  }
  // c2r of nrows complex rows, z in [z0, z0 + wz) (mod N) of each kept
  static void z_window(const T *in, T *out, long nrows, int z0, int wz, hipStream_t st, TimingHook *hook) {
    ZArgs<T> a{};
    a.job[0] = {in, nullptr, out, FFT_YZ_ONE};
    a.nrows = nrows;
    a.iters = Rows::iters(nrows, 1);
    a.z0 = z0;
    a.wz = wz;
    a.scale = norm();
    rows_launch(k_fft_z_c2r<T, N, Rows::TH, true>, a, 1, 1, "fft_z_c2r_win", double(nrows) * ((N + 2) + wz) * sizeof(T),
                st, hook);
  }
  // r2c of nrows rows given as their points [z0, z0 + wz) (mod N)
  static void r2c_z_window(const T *win, T *out, long nrows, int z0, int wz, hipStream_t st, TimingHook *hook) {
    ZFwdArgs<T> a{};
    a.job[0] = {win, out, 0};
    a.nrows = nrows;
    a.iters = Rows::iters(nrows, 1);
    a.z0 = z0;
    a.wz = wz;
    rows_launch(k_fft_z_r2c<T, N, Rows::TH, true>, a, 1, 1, "fft_z_r2c_win", double(nrows) * ((N + 2) + wz) * sizeof(T),
                st, hook);
  }
  // the z and y passes of r2c_window: bufA <- wl[0] planes
  static void r2c_window_zy(const T *win, const int *w0, const int *wl, T *bufB, T *bufA, hipStream_t st,
                            TimingHook *hook) {
    r2c_z_window(win, bufB, long(wl[0]) * wl[1], w0[2], wl[2], st, hook);
    // y pass: tiles (x_local, kz block), lines over ky from the wl[1] window rows
    StridedArgs<T> ay{};
    ay.in = reinterpret_cast<const cx<T> *>(bufB);
    ay.out = reinterpret_cast<cx<T> *>(bufA);
    ay.in_ls = NZ;
    ay.in_os = long(wl[1]) * NZ;
    ay.out_ls = NZ;
    ay.out_os = long(N) * NZ;
    ay.win0 = 0;
    ay.wlen = N;
    ay.in_win0 = w0[1];
    ay.in_wlen = wl[1];
    ay.scale = T(1);
    strided<-1, PRE_NONE, POST_NONE, 5>(ay, wl[0], st, hook, "fft_y_fwd_win");
  }
  // spectrum of a field that is zero outside the real-space window
  // [w0, w0+wl) (per axis, mod N), given as the dense window `win`
  // (wl[0]*wl[1]*wl[2] reals): pruned z and y passes, a full x pass whose
  // output is scaled by post[|k|^2] (if given) and stored or added into spec.
  // bufB holds wl[0]*wl[1] padded rows, bufA wl[0]*N*(N/2+1) complex.
  static void r2c_window(const T *win, const int *w0, const int *wl, T *bufB, T *bufA, T *spec, const T *post,
                         bool accum, hipStream_t st, TimingHook *hook, const T *aux = nullptr, const FilterInline *fil = nullptr,
                         double kmin = 0) {
    r2c_window_zy(win, w0, wl, bufB, bufA, st, hook);
    // x pass: tiles (ky, kz block), lines over kx from the wl[0] window planes
    StridedArgs<T> ax{};
    ax.in = reinterpret_cast<const cx<T> *>(bufA);
    ax.out = reinterpret_cast<cx<T> *>(spec);
    ax.in_ls = long(N) * NZ;
    ax.in_os = NZ;
    ax.out_ls = long(N) * NZ;
    ax.out_os = NZ;
    ax.win0 = 0;
    ax.wlen = N;
    ax.in_win0 = w0[0];
    ax.in_wlen = wl[0];
    ax.scale = norm();
    ax.tab = post;
    ax.accum = accum ? 1 : 0;
    ax.aux = reinterpret_cast<const cx<T> *>(aux);
    if (fil) ax.fil = *fil;
    ax.kmin_d = kmin;
    if (aux) strided<-1, PRE_NONE, POST_AUX, 4>(ax, N, st, hook, "fft_x_fwd_win");
    else if (post) strided<-1, PRE_NONE, POST_TABLE, 4>(ax, N, st, hook, "fft_x_fwd_win");
    else strided<-1, PRE_NONE, POST_NONE, 4>(ax, N, st, hook, "fft_x_fwd_win");
  }
};

}  // namespace gic
