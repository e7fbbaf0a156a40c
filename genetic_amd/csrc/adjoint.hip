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

long table_entries(const LevelGeom &g) {
  long h = g.n / 2;
  return 3 * h * h + 1;
}

// out[|k|^2] = sqrtP(k) filter(k) / k^2 with the filter of kind (0 low, 1
// high, 2 unity) at kc, on level L
template <typename T> void adjoint_table(gic_context *c, Level &L, int kind, double kc, DevBuf &out) {
  long nent = table_entries(L.g);
  out.ensure(nent * sizeof(T));
  filter_table<T>(kind, kc, L.g.kmin(), nent, (T *)out.p, c->st, true);
  hipLaunchKernelGGL(k_tab_mul<T>, dim3((nent + 255) / 256), dim3(256), 0, c->st, (T *)out.p, (const T *)L.sqrtp.p,
                     nent);
  GIC_HIP(hipGetLastError());
}

void check_ready(gic_context *c) {
  if (c->levels.empty()) throw std::runtime_error("No grid has yet been initialised");
  if (!c->have_camb) throw std::runtime_error("No power spectrum has been set (use the camb command)");
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
  for (size_t l = 0; l < nl; ++l) {
    Level &L = *c->levels[l];
    alloc_field(c, L.noise, L.g);
    build_sqrtp<T>(c, L);
    FftZFwd<T> z;
    z.add(noise[l], (T *)L.noise.p, true);
    fft_z_forward<T>(z, L.g.n, c->st, c->hook());
    FftYFwd<T> y;
    y.add((const T *)L.noise.p, nullptr, (T *)L.noise.p);
    fft_y_forward<T>(y, L.g.n, c->st, c->hook());
    L.have_psi = L.have_psi2 = false;
  }
  c->seeded = c->drawn = c->power_applied = true;
  int order = c->lpt_order;
  c->lpt_order = 1;
  try {
    do_zeldovich<T>(c, psi);
  } catch (...) {
    c->lpt_order = order;
    throw;
  }
  c->lpt_order = order;
  c->zeldovich_done = nl > 1;
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
    adjoint_table<T>(c, L, l >= 1 ? 1 : 2, l >= 1 ? kcut_for_level(c, int(l) - 1) : 0.0, L.adj_tab);
    if (l + 1 < nl) {
      if (l == 0) {
        adjoint_table<T>(c, L, 0, kcut_for_level(c, 0), L.adj_lp);
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
    fft_x_adjoint<T>(h[0], h[1], (const T *)L.adj_tab.p, low ? u[0] : nullptr, low ? u[1] : nullptr,
                     low ? (const T *)L.adj_lp.p : nullptr, n, L.g.kmin(), c->st, c->hook());
    FftY<T> yb;
    yb.add(h[0], h[0], FFT_YZ_ONE);
    fft_y<T>(yb, n, c->st, c->hook());
    FftZ<T> zb;
    zb.add(h[0], nullptr, noise_bar[li], FFT_YZ_ONE);
    fft_z<T>(zb, n, c->st, c->hook());
  }
  GIC_HIP(hipStreamSynchronize(c->st));
}

template void do_displacement_forward<float>(gic_context *, const float *const *, float *const *);
template void do_displacement_forward<double>(gic_context *, const double *const *, double *const *);
template void do_displacement_adjoint<float>(gic_context *, const float *const *, float *const *);
template void do_displacement_adjoint<double>(gic_context *, const double *const *, double *const *);

}  // namespace gic
