// Displacement map w -> psi as an explicit linear operator, and its transpose.
//
// The forward map is the Zel'dovich path of the context (ICGenerator::done ->
// MultiLevelField / ZeldovichParticleGenerator, ic.hpp:1633-1648,
// zeldovich.hpp:152-253, level combination field.hpp:816-849): per level l
//   delta_l = sqrtP_l * r2c(w_l),
//   psi_{l,a} = c2r(i k_a F_l / k^2 * delta_l)        (F_0 = 1, F_l = HP_l)
// and for a zoom level psi_l += I_l [ LP_{l-1} psi_{l-1} ] with I_l the
// tricubic interpolation onto the fine cells.  Every step is linear in w, so
// the gradient of a scalar loss of psi is the transposed chain (no
// counterpart in the reference):
//   g_l = psibar_l + LP_l c2r r2c [ I_{l+1}^T g_{l+1} ]         (finest first)
//   wbar_l = c2r( sum_a conj(i k_a F_l sqrtP_l / k^2) r2c(g_{l,a}) )
// With the unitary FFT (N^-1.5 both ways) r2c^T = c2r on real fields, so the
// transpose of c2r diag(D) r2c is c2r diag(conj D) r2c.
#include "context.h"

namespace gic {

namespace {

template <typename T> __global__ void k_tab_mul(T *__restrict__ out, const T *__restrict__ a, long n) {
  long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) out[i] *= a[i];
}

// g[padded] += src[dense]
template <typename T> __global__ void k_add_dense(T *__restrict__ g, const T *__restrict__ src, int n) {
  size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  size_t n3 = size_t(n) * n * n;
  if (i >= n3) return;
  size_t row = i / n, z = i - row * n;
  g[row * (n + 2) + z] += src[i];
}

// per axis, the indices with a cell of the mask; words of W cells (4 where
// rows are aligned to them: 16.8 MB of 256^3 cells in 8.5 us, by single bytes 20)
template <typename W> __global__ void k_mask_axes(const W *__restrict__ mask, int n, uint8_t *__restrict__ used) {
  // one row of cells (fixed x, y) a wavefront
  const int row = int(blockIdx.x) * (blockDim.x / 64) + int(threadIdx.x) / 64, lane = int(threadIdx.x) % 64;
  if (row >= n * n) return;
  const int nw = n / int(sizeof(W));
  const W *m = mask + size_t(row) * nw;
  bool any = false;
  for (int w = lane; w < nw; w += 64) {
    const W v = m[w];
    if (v == 0) continue;
    any = true;
    for (int b = 0; b < int(sizeof(W)); ++b)
      if ((v >> (8 * b)) & 0xff) used[2 * n + w * int(sizeof(W)) + b] = 1;
  }
  if (any) {
    used[row / n] = 1;
    used[n + row % n] = 1;
  }
}

// v (nc components of a box of cells) times the mask's cells there, and the
// sums of squares of each block
constexpr int MASK_BLOCKS = 512;
template <typename T>
__global__ __launch_bounds__(256) void k_mask_square(T *__restrict__ v, const uint8_t *__restrict__ mask, int n, int x0,
                                                     int y0, int z0, int wx, int wy, int wz,
                                                     double *__restrict__ part) {
  const unsigned nb = unsigned(wx) * wy * wz;
  double acc = 0;
  for (unsigned i = blockIdx.x * 256u + threadIdx.x; i < nb; i += gridDim.x * 256u) {
    const unsigned r = i / unsigned(wz);
    int z = int(i - r * wz) + z0, x = int(r / unsigned(wy)), y = int(r - unsigned(x) * wy) + y0;
    x += x0;
    x -= x >= n ? n : 0;
    y -= y >= n ? n : 0;
    z -= z >= n ? n : 0;
    const T m = mask[(size_t(x) * n + y) * n + z] ? T(1) : T(0);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const T q = v[size_t(c) * nb + i] * m;
      v[size_t(c) * nb + i] = q;
      acc += double(q) * double(q);
    }
  }
  __shared__ double red[256];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (int(threadIdx.x) < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

long table_entries(const LevelGeom &g) {
  long h = g.n / 2;
  return 3 * h * h + 1;
}

// out[|k|^2] = sqrtP(k) filter(k) / k^2 with the filter of kind (0 low, 1
// high, 2 unity) at kc, on level L; kept while the spectrum's settings are
template <typename T> void adjoint_table(gic_context *c, Level &L, int kind, double kc, DevBuf &out, TabKey &key) {
  const TabKey want{c->spectrum, kind, L.g.n, kc, L.g.box};
  if (key == want) return;
  key = TabKey{};
  long nent = table_entries(L.g);
  out.ensure(nent * sizeof(T));
  filter_table<T>(kind, kc, L.g.kmin(), nent, (T *)out.p, c->st, true);
  hipLaunchKernelGGL(k_tab_mul<T>, dim3((nent + 255) / 256), dim3(256), 0, c->st, (T *)out.p, (const T *)L.sqrtp.p,
                     nent);
  GIC_HIP(hipGetLastError());
  key = want;
}

void check_ready(gic_context *c) {
  if (c->levels.empty()) throw std::runtime_error("No grid has yet been initialised");
  if (!c->have_camb) throw std::runtime_error("No power spectrum has been set (use the camb command)");
}

// The context's noise while a caller's takes its place: from the construction
// on there is none, until done() says that the overdensity is the new one.  An
// exception in between (no memory for a scratch array, say) leaves a context
// that has to draw again, not one whose half-made field passes for a spectrum.
class Replacing {
 public:
  explicit Replacing(gic_context *c) : c_(c) { none(); }
  Replacing(const Replacing &) = delete;
  Replacing &operator=(const Replacing &) = delete;
  ~Replacing() {
    if (!done_) none();
  }
  void done(bool zeldovich) {
    done_ = true;
    c_->seeded = c_->drawn = c_->power_applied = true;
    c_->zeldovich_done = zeldovich;
  }

 private:
  void none() {
    c_->drawn = c_->power_applied = c_->zeldovich_done = false;
    for (auto &L : c_->levels) L->noise_fourier = L->dc_pending = L->psi_fourier = L->have_psi = L->have_psi2 = false;
  }
  gic_context *c_;
  bool done_ = false;
};

// L.noise <- the dense white noise transformed along z and y
template <typename T> void load_noise_zy(gic_context *c, Level &L, const T *noise) {
  alloc_field(c, L.noise, L.g);
  build_sqrtp<T>(c, L);
  FftZFwd<T> z;
  z.add(noise, (T *)L.noise.p, true);
  fft_z_forward<T>(z, L.g.n, c->st, c->hook());
  FftYFwd<T> y;
  y.add((const T *)L.noise.p, nullptr, (T *)L.noise.p);
  fft_y_forward<T>(y, L.g.n, c->st, c->hook());
}

}  // namespace

template <typename T> void do_displacement_forward(gic_context *c, const T *const *noise, T *const *psi) {
  check_ready(c);
  size_t nl = c->levels.size();
  for (size_t l = 0; l < nl; ++l)
    if (!noise[l] || !psi[3 * l] || !psi[3 * l + 1] || !psi[3 * l + 2])
      throw std::runtime_error("displacement forward: null device pointer");
  // the noise along z and y, read straight from the caller's dense arrays;
  // the x pass of do_zeldovich makes delta_l = sqrtP r2c(w_l) and what the
  // displacements need of it
  Replacing field(c);
  for (size_t l = 0; l < nl; ++l) load_noise_zy<T>(c, *c->levels[l], noise[l]);
  c->drawn = c->power_applied = true;
  int order = c->lpt_order;
  c->lpt_order = 1;
  try {
    do_zeldovich<T>(c, psi);
  } catch (...) {
    c->lpt_order = order;
    throw;
  }
  c->lpt_order = order;
  field.done(nl > 1);
  for (size_t l = 1; l < nl; ++l) {
    Level &L = *c->levels[l];
    for (int a = 0; a < 3; ++a) unpad<T, T>((const T *)L.psi[a].p, L.g.n, psi[3 * l + a], c->st);
  }
  GIC_HIP(hipStreamSynchronize(c->st));
}

template <typename T> void do_displacement_adjoint(gic_context *c, const T *const *psi_bar, T *const *noise_bar) {
  check_ready(c);
  size_t nl = c->levels.size();
  for (size_t l = 0; l < nl; ++l)
    if (!noise_bar[l] || !psi_bar[3 * l] || !psi_bar[3 * l + 1] || !psi_bar[3 * l + 2])
      throw std::runtime_error("displacement adjoint: null device pointer");
  size_t maxreals = 0;
  for (size_t l = 0; l < nl; ++l) {
    Level &L = *c->levels[l];
    build_sqrtp<T>(c, L);
    if (l + 1 < nl)
      for (auto &u : L.adj_u) alloc_field(c, u, L.g);
    maxreals = std::max(maxreals, L.g.padded_reals());
  }
  c->xhalf.ensure(3 * maxreals * sizeof(T));
  // per level: the Zel'dovich operator's table sqrtP F_l / k^2, and the low
  // pass towards the next finer level (for level 0 with sqrtP / k^2 folded in)
  for (size_t l = 0; l < nl; ++l) {
    Level &L = *c->levels[l];
    adjoint_table<T>(c, L, l >= 1 ? 1 : 2, l >= 1 ? kcut_for_level(c, int(l) - 1) : 0.0, L.adj_tab,
                     L.adj_tab_key);
    if (l + 1 < nl) {
      if (l == 0) {
        adjoint_table<T>(c, L, 0, kcut_for_level(c, 0), L.adj_lp, L.adj_lp_key);
      } else {
        L.adj_lp.ensure(table_entries(L.g) * sizeof(T));
        filter_table<T>(0, kcut_for_level(c, int(l)), L.g.kmin(), table_entries(L.g), (T *)L.adj_lp.p, c->st);
      }
    }
  }
  for (size_t li = nl; li-- > 0;) {
    Level &L = *c->levels[li];
    const int n = L.g.n;
    const size_t reals = L.g.padded_reals();
    const bool finer = li + 1 < nl;
    // the level's gradient g: psibar alone (dense) on the finest level, on a
    // middle one psibar + LP c2r r2c (I^T g_finer), held in adj_u (padded);
    // on the base level the second term enters through adj_lp below
    const bool mid = finer && li >= 1;
    T *u[3] = {(T *)L.adj_u[0].p, (T *)L.adj_u[1].p, (T *)L.adj_u[2].p};
    if (mid) {
      for (int a = 0; a < 3; ++a) {
        fft_r2c_post<T>(u[a], n, (const T *)L.adj_lp.p, c->st, c->hook());
        fft3d<T>(u[a], n, +1, c->st, c->hook());
        hipLaunchKernelGGL(k_add_dense<T>, dim3((L.g.n3() + 255) / 256), dim3(256), 0, c->st, u[a],
                           psi_bar[3 * li + a], n);
        GIC_HIP(hipGetLastError());
      }
    }
    if (li >= 1) {
      // push g to the coarser level through the transposed interpolation
      Level &C = *c->levels[li - 1];
      InterpGeom ig = interp_geom(L.g, C.g);
      c->adj_fold.ensure(interp_adjoint_bytes<T>(n, ig));
      for (int a = 0; a < 3; ++a) {
        T *cu = (T *)C.adj_u[a].p;
        fill<T>(cu, C.g.padded_reals(), T(0), c->st);
        interp_adjoint<T>(mid ? u[a] : psi_bar[3 * li + a], n, mid ? n + 2 : n, cu, ig, (T *)c->adj_fold.p, c->st);
      }
    }
    // the transposed displacement: the gradients of psi_y and psi_z meet in
    // the y pass, those of psi_x and of both in the x pass
    T *h[3] = {(T *)c->xhalf.p, (T *)c->xhalf.p + reals, (T *)c->xhalf.p + 2 * reals};
    const bool low = finer && li == 0;
    FftZFwd<T> z;
    for (int a = 0; a < 3; ++a) z.add(mid ? u[a] : psi_bar[3 * li + a], h[a], !mid);
    if (low)
      for (int a = 0; a < 3; ++a) z.add(u[a], u[a], false);
    fft_z_forward<T>(z, n, c->st, c->hook());
    FftYFwd<T> y;
    y.kmin = L.g.kmin();
    y.add(h[0], nullptr, h[0]);
    y.add(h[1], h[2], h[1]);
    if (low) {
      y.add(u[0], nullptr, u[0]);
      y.add(u[1], u[2], u[1]);
    }
    fft_y_forward<T>(y, n, c->st, c->hook());
    FftXAdj<T> x;
    x.out = h[0];
    x.h1 = h[0];
    x.h0 = h[1];
    x.tab = (const T *)L.adj_tab.p;
    if (low) {
      x.g1 = u[0];
      x.g0 = u[1];
      x.gtab = (const T *)L.adj_lp.p;
    }
    x.kmin = L.g.kmin();
    fft_x_adjoint<T>(x, n, c->st, c->hook());
    FftY<T> yb;
    yb.add(h[0], h[0], FFT_YZ_ONE);
    fft_y<T>(yb, n, c->st, c->hook());
    FftZ<T> zb;
    zb.add(h[0], nullptr, noise_bar[li], FFT_YZ_ONE);
    fft_z<T>(zb, n, c->st, c->hook());
  }
  GIC_HIP(hipStreamSynchronize(c->st));
}

// The sum of |psi|^2 over the cells of a mask, and its gradient 2 Psi^T m Psi w:
// displacements are needed at the mask's cells only, so the passes after the
// forward ones are cut to the box around them (a box that spans the level
// takes them whole).  256^3 FP32, a sphere of 31 cells, value and gradient:
// 0.33 ms of kernels, against 0.75 for the full displacements and their
// transpose and 0.75 for the products and sums of full fields between them.
template <typename T>
double do_masked_displacement(gic_context *c, const T *noise, const uint8_t *mask, T *grad) {
  check_ready(c);
  if (c->levels.size() != 1) throw std::runtime_error("masked displacement: one level expected");
  if (!noise || !mask) throw std::runtime_error("masked displacement: null device pointer");
  Level &L = *c->levels[0];
  const int n = L.g.n;
  const size_t nz = size_t(n / 2 + 1);
  int w0[3], wl[3];
  {
    std::vector<uint8_t> used(3 * size_t(n));
    c->stage.ensure(used.size());
    fill<uint8_t>((uint8_t *)c->stage.p, used.size(), 0, c->st);
    if (n % 4 == 0 && reinterpret_cast<uintptr_t>(mask) % 4 == 0)
      hipLaunchKernelGGL(k_mask_axes<uint32_t>, dim3((n * n + 3) / 4), dim3(256), 0, c->st,
                         reinterpret_cast<const uint32_t *>(mask), n, (uint8_t *)c->stage.p);
    else
      hipLaunchKernelGGL(k_mask_axes<uint8_t>, dim3((n * n + 3) / 4), dim3(256), 0, c->st, mask, n,
                         (uint8_t *)c->stage.p);
    GIC_HIP(hipGetLastError());
    GIC_HIP(hipMemcpyAsync(used.data(), c->stage.p, used.size(), hipMemcpyDeviceToHost, c->st));
    GIC_HIP(hipStreamSynchronize(c->st));
    for (int d = 0; d < 3; ++d) {
      cyclic_hull(used.data() + size_t(d) * n, n, w0[d], wl[d]);
      if (wl[d] == 0) wl[d] = 1;   // an empty mask: one cell, of weight 0
    }
  }
  Replacing field(c);
  load_noise_zy<T>(c, L, noise);
  // planes: f m and i k_x f m of the box's x; rows: of its x and y; the box
  const size_t planes = size_t(wl[0]) * n * nz * 2, rows = size_t(wl[0]) * wl[1] * nz * 2;
  const size_t nb = size_t(wl[0]) * wl[1] * wl[2];
  c->stage.ensure(MASK_BLOCKS * sizeof(double) + (2 * planes + 3 * rows + 3 * nb) * sizeof(T));
  double *part = (double *)c->stage.p;
  T *A = (T *)(part + MASK_BLOCKS), *B = A + 2 * planes, *O = B + 3 * rows;
  FftX<T> x;
  x.in = x.spec = (T *)L.noise.p;
  x.forward = true;
  x.post = (const T *)L.sqrtp.p;
  x.out[1] = A;
  x.out[2] = A + planes;
  x.inv_k2 = 1.0;
  x.kmin = L.g.kmin();
  x.win0 = w0[0];
  x.wlen = wl[0];
  fft_x<T>(x, n, c->st, c->hook());
  L.noise_fourier = true;
  field.done(false);
  FftY<T> y;
  y.kmin = L.g.kmin();
  y.nouter = wl[0];
  y.win0 = w0[1];
  y.wlen = wl[1];
  y.add(A + planes, B, FFT_YZ_ONE);
  y.add(A, B + rows, FFT_YZ_IKY, B + 2 * rows, FFT_YZ_IKZ);
  fft_y<T>(y, n, c->st, c->hook());
  fft_z_window<T>(B, O, 3 * long(wl[0]) * wl[1], w0[2], wl[2], n, c->st, c->hook());
  hipLaunchKernelGGL(k_mask_square<T>, dim3(MASK_BLOCKS), dim3(256), 0, c->st, O, mask, n, w0[0], w0[1], w0[2], wl[0],
                     wl[1], wl[2], part);
  GIC_HIP(hipGetLastError());
  if (grad) {
    adjoint_table<T>(c, L, 2, 0.0, L.adj_tab, L.adj_tab_key);
    fft_r2c_z_window<T>(O, B, 3 * long(wl[0]) * wl[1], w0[2], wl[2], n, c->st, c->hook());
    FftYFwd<T> yf;
    yf.kmin = L.g.kmin();
    yf.nouter = wl[0];
    yf.iwin0 = w0[1];
    yf.iwlen = wl[1];
    yf.add(B, nullptr, A + planes);
    yf.add(B + rows, B + 2 * rows, A);
    fft_y_forward<T>(yf, n, c->st, c->hook());
    c->xhalf.ensure(L.g.padded_reals() * sizeof(T));
    T *h = (T *)c->xhalf.p;
    FftXAdj<T> xa;
    xa.out = h;
    xa.h1 = A + planes;
    xa.h0 = A;
    xa.tab = (const T *)L.adj_tab.p;
    xa.kmin = L.g.kmin();
    xa.iwin0 = w0[0];
    xa.iwlen = wl[0];
    fft_x_adjoint<T>(xa, n, c->st, c->hook());
    FftY<T> yb;
    yb.add(h, h, FFT_YZ_ONE);
    fft_y<T>(yb, n, c->st, c->hook());
    FftZ<T> zb;
    zb.scale = 2;
    zb.add(h, nullptr, grad, FFT_YZ_ONE);
    fft_z<T>(zb, n, c->st, c->hook());
  }
  std::vector<double> sums(MASK_BLOCKS);
  GIC_HIP(hipMemcpyAsync(sums.data(), part, MASK_BLOCKS * sizeof(double), hipMemcpyDeviceToHost, c->st));
  GIC_HIP(hipStreamSynchronize(c->st));
  double v = 0;
  for (double s : sums) v += s;
  return v;
}

template double do_masked_displacement<float>(gic_context *, const float *, const uint8_t *, float *);
template double do_masked_displacement<double>(gic_context *, const double *, const uint8_t *, double *);
template void do_displacement_forward<float>(gic_context *, const float *const *, float *const *);
template void do_displacement_forward<double>(gic_context *, const double *const *, double *const *);
template void do_displacement_adjoint<float>(gic_context *, const float *const *, float *const *);
template void do_displacement_adjoint<double>(gic_context *, const double *const *, double *const *);

}  // namespace gic
