// C-ABI implementation: the ICGenerator field path on one GPU.
//
// The orchestration follows the reference's ICGenerator (genetIC/src/ic.hpp)
// and MultiLevelParticleGenerator (particles/multilevelgenerator.hpp:78-128);
// the arithmetic runs in the kernels of fft.hip, rng.hip and kspace.hip.
#include "context.h"

using namespace gic;

namespace gic {

size_t total_bytes(gic_context *c) {
  size_t b = c->work.bytes + c->stage.bytes + c->tab_a.bytes + c->tab_b.bytes + c->tab_c.bytes + c->spl_x.bytes * 3;
  for (auto &l : c->levels) {
    b += l->noise.bytes + l->sqrtp.bytes;
    for (auto &p : l->psi) b += p.bytes;
  }
  return b;
}

Level &level_at(gic_context *c, int level) {
  if (level < 0 || level >= (int)c->levels.size()) throw std::runtime_error("Specified level does not exist.");
  return *c->levels[level];
}


void alloc_field(gic_context *c, DevBuf &b, const LevelGeom &g) {
  b.ensure(g.padded_reals() * c->tsize());
}

// camb.hpp:300-328: sigma(R) by a 50000-step rectangle rule with accumulated k
double variance_in_sphere(gic_context *c, double radius) {
  double s = 0., k, t;
  double amp = 9. / 2. / M_PI / M_PI;
  double kmax = std::min(c->kpts.back(), 200.0 / radius) * 0.999999;
  double kmin = c->kpts[0] * 1.000001;
  double dk = (kmax - kmin) / 50000.;
  for (k = kmin; k < kmax; k += dk) {
    t = c->tf_all(k);
    double kr = k * radius;
    double w = (sin(kr) - kr * cos(kr)) / (kr * kr * kr);
    s += pow(k, c->ns_frozen + 2.) * w * w * t * t;
  }
  return sqrt(s * amp * dk);
}

// (The table depends on the spectrum's settings and the level alone, and is
// kept while they are: evaluating the spline takes 5 us at n = 64, a twelfth
// of a whole displacement there, and 7 us at 256.)
template <typename T>
static void sqrtp_of(gic_context *c, Level &L, const SplineHost &spline, DevBuf &tab, TabKey &key) {
  if (!c->have_camb) throw std::runtime_error("No power spectrum has been set (use the camb command)");
  const TabKey want{c->spectrum, 0, L.g.n, 0.0, L.g.box};
  if (key == want) return;
  key = TabKey{};
  long h = L.g.n / 2;
  long nent = 3 * h * h + 1;
  tab.ensure(nent * sizeof(T));
  double kw = 2. * M_PI / L.g.box;
  double norm = kw * kw * kw / pow(2.f * M_PI, 3.f) * double(L.g.n3());
  sqrtp_table<T>(spline, c->amplitude, c->ns_frozen, L.g.kmin(), norm, nent, (T *)tab.p, c->st);
  key = want;
}

template <typename T> void build_sqrtp(gic_context *c, Level &L) { sqrtp_of<T>(c, L, c->spline_dev, L.sqrtp, L.sqrtp_key); }

// the dark-matter column of the transfer table (camb.hpp:181-185): the
// covectors of the modifications carry this spectrum
template <typename T> void build_sqrtp_dm(gic_context *c, Level &L) {
  sqrtp_of<T>(c, L, c->spline_dm_dev, L.sqrtp_dm, L.sqrtp_dm_key);
}

// The white noise stays in real space after the draw; the first transform
// to Fourier space zeroes Re(w_0) (randomfieldgenerator.hpp:194-195).  When
// the power spectrum is applied to noise that is still real, the r2c and the
// sqrt P multiply share one pass.
template <typename T> void noise_to_fourier(gic_context *c, Level &L, const T *post) {
  if (L.noise_fourier) {
    if (post) mul_table<T>((T *)L.noise.p, L.g.n, post, c->st);
    return;
  }
  fft_r2c_post<T>((T *)L.noise.p, L.g.n, post, c->st, c->hook());
  L.noise_fourier = true;
  if (L.dc_pending) {
    if (!post) fill<T>((T *)L.noise.p, 1, T(0), c->st);   // with sqrt P applied the k=0 mode is already 0
    L.dc_pending = false;
  }
}

template <typename T> void do_draw(gic_context *c) {
  if (!c->seeded) throw std::runtime_error("The random number generator has not been seeded");
  if (c->drawn) throw std::runtime_error("Trying to re-draw the random field after it was already initialised");
  if (c->levels.empty()) throw std::runtime_error("Cannot draw a random field before the base grid is initialised");
  Phase ph(c, "phase:draw");
  for (auto &L : c->levels) alloc_field(c, L->noise, L->g);
  if (c->seed_mode == GIC_SEED_REAL_SPACE) {
    std::vector<RngLevelOut> outs;
    size_t total = 0;
    for (auto &L : c->levels) {
      outs.push_back({L->noise.p, L->g.n, L->g.n3()});
      total += L->g.n3();
    }
    RngPlan plan;
    rng_plan(c->seed, total, plan);
    c->work.ensure(rng_workspace_bytes(plan));
    rng_draw_real<T>(plan, outs, c->work.p, c->work.bytes, c->st, c->hook());
    for (auto &L : c->levels) {
      L->noise_fourier = false;
      L->dc_pending = true;
    }
  } else {
    // Fourier-space draws: the Gaussians of every level in draw order into a
    // dense buffer (one stream continued across levels, or in parallel mode a
    // stream seeded seed+ks per shell and level), then placed mode by mode.
    const double sigma = double(T(1.0 / sqrt(2.0)));
    bool parallel = c->seed_mode == GIC_SEED_FOURIER_PARALLEL;
    int reverse = c->seed_mode == GIC_SEED_FOURIER_REVERSE ? 1 : 0;
    std::vector<size_t> off;
    size_t total = 0, maxslots = 0;
    for (auto &L : c->levels) {
      off.push_back(total);
      total += 2 * size_t(fourier_draw_count(L->g.n));
      maxslots = std::max(maxslots, size_t(L->g.n) * L->g.n * (L->g.n / 2 + 1));
    }
    size_t gbytes = (total * sizeof(T) + 255) / 256 * 256;
    c->stage.ensure(gbytes + maxslots * 4);
    T *gauss = (T *)c->stage.p;
    uint32_t *owner = (uint32_t *)((char *)c->stage.p + gbytes);
    if (total) {
      // one stream, or all shells' streams in one draw
      std::vector<RngStream> streams;
      if (!parallel) {
        streams.push_back({c->seed, total, 0});
      } else {
        for (size_t l = 0; l < c->levels.size(); ++l) {
          size_t pos = off[l];
          for (int ks = 1; ks < c->levels[l]->g.n / 2; ++ks) {
            size_t cnt = 24 * size_t(ks) * ks;
            streams.push_back({c->seed + ks, cnt, pos});
            pos += cnt;
          }
        }
      }
      RngPlan plan;
      rng_plan(streams, plan);
      c->work.ensure(rng_workspace_bytes(plan));
      std::vector<RngLevelOut> outs{{gauss, 0, total}};
      rng_draw_real<T>(plan, outs, c->work.p, c->work.bytes, c->st, c->hook(), sigma);
    }
    for (size_t l = 0; l < c->levels.size(); ++l) {
      Level &L = *c->levels[l];
      fourier_draw_scatter<T>(gauss + off[l], L.g.n, (T *)L.noise.p, owner, reverse, c->st);
      L.noise_fourier = true;
      L.dc_pending = false;
    }
  }
  c->drawn = true;
  if (c->fix_power) {
    // enforceUnitVariance (multilevelfield.hpp:395-407), right after the draw (ic.hpp:1343-1344)
    for (auto &Lp : c->levels) {
      ensure_noise_fourier<T>(c, *Lp);
      unit_modulus<T>((T *)Lp->noise.p, Lp->g.n, c->st);
    }
  }
}

template <typename T> void ensure_noise_fourier(gic_context *c, Level &L) { noise_to_fourier<T>(c, L, nullptr); }

template <typename T> void do_apply_ps(gic_context *c) {
  if (!c->drawn) do_draw<T>(c);
  for (auto &Lp : c->levels) {
    Level &L = *Lp;
    build_sqrtp<T>(c, L);
    if (c->hook()) c->hook()->begin("apply_sqrtp", c->st);
    noise_to_fourier<T>(c, L, (const T *)L.sqrtp.p);
    if (c->hook()) c->hook()->end("apply_sqrtp", c->st);
  }
  c->power_applied = true;
}

double kcut_for_level(gic_context *c, int level) {
  const LevelGeom &g = c->levels[level]->g;
  return 0.3 * (double(g.n) * g.kmin());   // FRACTIONAL_K_SPLIT * k_pixel (filterfamily.hpp:110-118)
}

InterpGeom interp_geom(const LevelGeom &gf, const LevelGeom &gc) {
  InterpGeom ig;
  int ratio = (int)llround(gc.dx / gf.dx);
  double dxs = gc.dx / ratio;
  ig.off[0] = (int)llround((gf.ox - gc.ox) / dxs);
  ig.off[1] = (int)llround((gf.oy - gc.oy) / dxs);
  ig.off[2] = (int)llround((gf.oz - gc.oz) / dxs);
  ig.sim = (int)llround(gf.periodic / dxs);
  ig.nsup = gc.n * ratio;
  ig.nc = gc.n;
  ig.wrap = gc.n == (int)llround(gc.periodic / gc.dx) ? 1 : 0;
  return ig;
}

// Low-passed real-space copy of a coarse level for the interpolation onto the
// next level (addFieldFromDifferentGridWithFilter, FILTER_ON_COARSE_GRID
// branch, field.hpp:816-830): copy the field, filter in Fourier space,
// transform back.  For a zoom level the coarse fields are combined real
// fields; the copy is transformed forward with the filter fused into its
// last pass.
template <typename T> CoarseView lowpass_full(gic_context *c, const DevBuf &src, const LevelGeom &g, const T *lp) {
  size_t bytes = g.padded_reals() * sizeof(T);
  c->stage.ensure(bytes);
  GIC_HIP(hipMemcpyAsync(c->stage.p, src.p, bytes, hipMemcpyDeviceToDevice, c->st));
  fft_r2c_post<T>((T *)c->stage.p, g.n, lp, c->st, c->hook());
  fft3d<T>((T *)c->stage.p, g.n, +1, c->st, c->hook());
  CoarseView v;
  v.p = c->stage.p;
  for (int a = 0; a < 3; ++a) {
    v.org[a] = 0;
    v.len[a] = g.n;
  }
  v.sx = long(g.n) * (g.n + 2);
  v.sy = g.n + 2;
  return v;
}

// Coarse cells the tricubic stencils of a fine level touch: the fine grid
// spans coarse cells [o, o + nf/r); the stencil reaches 2 cells below and
// 2 above, plus one cell of slack for rounding in floor().
void coarse_window(const LevelGeom &gf, const LevelGeom &gc, int *w0, int *wl) {
  int r = (int)llround(gc.dx / gf.dx);
  double off[3] = {gf.ox - gc.ox, gf.oy - gc.oy, gf.oz - gc.oz};
  for (int a = 0; a < 3; ++a) {
    int o = (int)llround(off[a] / gc.dx);
    int start = o - 3;
    int len = gf.n / r + 6;
    start %= gc.n;
    if (start < 0) start += gc.n;
    w0[a] = start;
    wl[a] = len;
  }
}

// What a fine level takes of the base level's spectrum m (already multiplied
// by its own factor where it has one): the low-passed displacement LP/k^2 i k m
// scale and with delta the low-passed m itself, in the coarse window only --
// one x pass, one y pass, then the rows.  view[0..2] receive the
// displacements, view[3] the low-passed m; they lie in buf.
template <typename T>
void coarse_parts(gic_context *c, const T *m, const LevelGeom &g, double kc, double scale, bool delta, const int *w0,
                  const int *wl, DevBuf &buf, CoarseView *view) {
  const int n = g.n, nz = n / 2 + 1, nv = delta ? 4 : 3;
  const size_t a_n = size_t(wl[0]) * n * nz * 2, b_n = size_t(wl[0]) * wl[1] * nz * 2;
  const size_t o_n = size_t(wl[0]) * wl[1] * wl[2];
  buf.ensure(((nv - 1) * a_n + nv * (b_n + o_n)) * sizeof(T));
  T *A = (T *)buf.p, *B = A + (nv - 1) * a_n, *O = B + nv * b_n;
  long h = n / 2, nent = 3 * h * h + 1;
  c->tab_b.ensure(nent * sizeof(T));
  c->tab_c.ensure(nent * sizeof(T));
  filter_table<T>(0, kc, g.kmin(), nent, (T *)c->tab_b.p, c->st);
  filter_table<T>(0, kc, g.kmin(), nent, (T *)c->tab_c.p, c->st, true, scale);
  FilterInline fil;   // the same low pass over k^2, formed in the pass (FP32)
  fil.nf = 1;
  fil.kind[0] = 0;
  fil.kc[0] = kc;
  fil.scale = scale;
  fil.over_k2 = 1;
  FftX<T> x;
  x.in = m;
  x.out[1] = A;
  x.out[2] = A + a_n;
  if (delta) {
    x.out[0] = A + 2 * a_n;
    x.plain0 = true;
  }
  x.fil = &fil;
  x.tab = (const T *)c->tab_c.p;
  x.tab0 = (const T *)c->tab_b.p;
  x.kmin = g.kmin();
  x.win0 = w0[0];
  x.wlen = wl[0];
  fft_x<T>(x, n, c->st, c->hook());
  FftY<T> y;
  y.kmin = g.kmin();
  y.nouter = wl[0];
  y.win0 = w0[1];
  y.wlen = wl[1];
  y.add(A + a_n, B, FFT_YZ_ONE);
  y.add(A, B + b_n, FFT_YZ_IKY, B + 2 * b_n, FFT_YZ_IKZ);
  if (delta) y.add(A + 2 * a_n, B + 3 * b_n, FFT_YZ_ONE);
  fft_y<T>(y, n, c->st, c->hook());
  for (int f = 0; f < nv; ++f) {
    fft_z_window<T>(B + f * b_n, O + f * o_n, long(wl[0]) * wl[1], w0[2], wl[2], n, c->st, c->hook());
    view[f].p = O + f * o_n;
    for (int a = 0; a < 3; ++a) {
      view[f].org[a] = w0[a];
      view[f].len[a] = wl[a];
    }
    view[f].sx = long(wl[1]) * wl[2];
    view[f].sy = wl[2];
  }
}

// out[a] (padded) and, if given, dense[a] <- the displacement of x passes X0
// (of f m) and X1 (of i k_x f m): psi_y and psi_z share X0's y pass, psi_z's
// factor k_z rides on its z pass.  X0 and X1 may be outputs.
template <typename T>
void displacement_yz(gic_context *c, const T *X0, const T *X1, T *const *out, T *const *dense, bool padded,
                     const LevelGeom &g) {
  FftY<T> y;
  y.kmin = g.kmin();
  y.add(X1, out[0], FFT_YZ_ONE);
  y.add(X0, out[1], FFT_YZ_IKY, out[2], FFT_YZ_ONE);
  fft_y<T>(y, g.n, c->st, c->hook());
  FftZ<T> z;
  z.kmin = g.kmin();
  for (int a = 0; a < 3; ++a)
    z.add(out[a], padded ? out[a] : nullptr, dense ? dense[a] : nullptr, a == 2 ? FFT_YZ_IKZ : FFT_YZ_ONE);
  fft_z<T>(z, g.n, c->st, c->hook());
}

// Second-order LPT (no counterpart in the reference, which stops at
// Zel'dovich, zeldovich.hpp:152-253).  With phi_ij = k_i k_j delta / k^2 the
// source is S = sum_{i<j} (phi_ii phi_jj - phi_ij^2) and
// psi2 = (3/7) i k S / k^2, i.e. D2 = -3/7 D1^2 with delta at the output
// redshift; the velocity uses f2 = 2 f1.  Each level is built from its
// combined overdensity; a zoom level keeps the high-pass part of its own
// psi2 and takes the low-pass part from the level above, as for psi.  The
// base level's source comes from its Zel'dovich passes, in the first field
// of xhalf.
template <typename T> void do_second_order(gic_context *c) {
  size_t nl = c->levels.size();
  CoarseView win_view[3];
  bool win_ready = false;
  for (size_t l = 0; l < nl; ++l) {
    Level &L = *c->levels[l];
    const LevelGeom &g = L.g;
    int n = g.n;
    size_t reals = g.padded_reals(), bytes = reals * sizeof(T);
    for (auto &p : L.psi2) alloc_field(c, p, g);
    long h = n / 2, nent = 3 * h * h + 1;
    c->tab_c.ensure(nent * sizeof(T));
    T *q[3] = {(T *)L.psi2[0].p, (T *)L.psi2[1].p, (T *)L.psi2[2].p};
    c->xhalf.ensure(3 * bytes);
    T *X[3] = {(T *)c->xhalf.p, (T *)c->xhalf.p + reals, (T *)c->xhalf.p + 2 * reals};
    T *S = X[0];
    if (c->hook()) c->hook()->begin("lpt_source", c->st);
    if (l > 0) {
      // the x passes of (1/k^2) delta, i k_x (1/k^2) delta and k_x^2 (1/k^2) delta
      c->stage.ensure(2 * bytes);
      T *D = (T *)c->stage.p;
      S = D + reals;
      FftX<T> x;
      if (L.noise_fourier) {
        x.in = (const T *)L.noise.p;
      } else {
        FftZFwd<T> zf;
        zf.add((const T *)L.noise.p, D, false);
        fft_z_forward<T>(zf, n, c->st, c->hook());
        FftYFwd<T> yf;
        yf.add(D, nullptr, D);
        fft_y_forward<T>(yf, n, c->st, c->hook());
        x.in = D;
        x.forward = true;
      }
      for (int i = 0; i < 3; ++i) x.out[i + 1] = X[i];
      x.inv_k2 = 1.0;
      x.kmin = g.kmin();
      fft_x<T>(x, n, c->st, c->hook());
      FftY<T> y;
      y.kmin = g.kmin();
      y.add(X[2], q[0], FFT_YZ_ONE);
      y.add(X[1], X[1], FFT_YZ_ONE, q[2], FFT_YZ_MIKY);
      y.add(X[0], X[0], FFT_YZ_ONE, D, FFT_YZ_KY, q[1], FFT_YZ_KYKY);
      fft_y<T>(y, n, c->st, c->hook());
      fft_z_lpt<T>(X[1], D, X[0], q[0], q[1], q[2], S, false, n, g.kmin(), c->st, c->hook());
    }
    if (c->hook()) c->hook()->end("lpt_source", c->st);
    // the level whose low-pass part level 1 takes straight from the base
    // source spectrum (a pruned c2r into the coarse window)
    int w0[3], wl[3];
    bool window = l == 0 && nl >= 2 && g.covers_full();
    if (window) {
      coarse_window(c->levels[1]->g, g, w0, wl);
      window = wl[0] < n && wl[1] < n && wl[2] < n;
    }
    {
      // S transformed, its x pass making f S and i k_x f S, f the level's
      // filter (3/7)/k^2 (unit filter on the base level, formed in the pass)
      FftZFwd<T> zf;
      zf.add(S, S, false);
      fft_z_forward<T>(zf, n, c->st, c->hook());
      FftYFwd<T> yf;
      yf.add(S, nullptr, S);
      fft_y_forward<T>(yf, n, c->st, c->hook());
      FftX<T> x;
      x.in = S;
      x.forward = true;
      if (window) x.spec = S;
      x.out[1] = X[1];
      x.out[2] = X[2];
      if (l >= 1) {
        filter_table<T>(1, kcut_for_level(c, int(l) - 1), g.kmin(), nent, (T *)c->tab_c.p, c->st, true, 3.0 / 7.0);
        x.tab = (const T *)c->tab_c.p;
      } else {
        x.inv_k2 = 3.0 / 7.0;
      }
      x.kmin = g.kmin();
      fft_x<T>(x, n, c->st, c->hook());
      displacement_yz<T>(c, X[1], X[2], q, nullptr, true, g);
    }
    if (l >= 1) {
      Level &C = *c->levels[l - 1];
      InterpGeom ig = interp_geom(g, C.g);
      if (l == 1 && win_ready) {
        for (int a = 0; a < 3; ++a) interp_add<T>(q[a], n, win_view[a], ig, c->st);
      } else {
        long hc = C.g.n / 2, nc_ent = 3 * hc * hc + 1;
        c->tab_b.ensure(nc_ent * sizeof(T));
        filter_table<T>(0, kcut_for_level(c, int(l) - 1), C.g.kmin(), nc_ent, (T *)c->tab_b.p, c->st);
        for (int a = 0; a < 3; ++a) {
          CoarseView v = lowpass_full<T>(c, C.psi2[a], C.g, (const T *)c->tab_b.p);
          interp_add<T>(q[a], n, v, ig, c->st);
        }
      }
    }
    if (window) {
      coarse_parts<T>(c, S, g, kcut_for_level(c, 0), 3.0 / 7.0, false, w0, wl, c->lpt_win, win_view);
      win_ready = true;
    }
    L.have_psi2 = true;
  }
}

// The displacements of level l from its spectrum (L.noise), or with forward
// from noise transformed along z and y there, whose spectrum times sqrt P is
// left in its place.  A zoom level carries its high-pass filter (the cut of
// the level above).  The base level of a second-order run also gets its
// source, into the first field of xhalf, from the same y passes.
template <typename T> void level_displacements(gic_context *c, size_t l, bool forward, T *const *dense) {
  Level &L = *c->levels[l];
  const LevelGeom &g = L.g;
  const bool lpt = l == 0 && c->lpt_order == 2;
  const bool padded = !(dense && c->levels.size() == 1);   // a lone level's go to the caller only
  size_t reals = g.padded_reals();
  if (padded)
    for (auto &p : L.psi) alloc_field(c, p, g);
  c->xhalf.ensure(3 * reals * sizeof(T));
  T *X0 = (T *)c->xhalf.p, *X1 = X0 + reals, *X2 = X1 + reals;
  T *psi[3] = {padded ? (T *)L.psi[0].p : X1, padded ? (T *)L.psi[1].p : X0, padded ? (T *)L.psi[2].p : X2};
  FftX<T> x;
  x.in = (const T *)L.noise.p;
  if (forward) {
    x.forward = true;
    x.spec = (T *)L.noise.p;
    x.post = (const T *)L.sqrtp.p;
  }
  x.out[1] = X0;
  x.out[2] = X1;
  if (lpt) x.out[3] = X2;
  if (l >= 1) {
    long h = g.n / 2, nent = 3 * h * h + 1;
    c->tab_c.ensure(nent * sizeof(T));
    filter_table<T>(1, kcut_for_level(c, int(l) - 1), g.kmin(), nent, (T *)c->tab_c.p, c->st, true);
    x.tab = (const T *)c->tab_c.p;
  } else {
    x.inv_k2 = 1.0;
  }
  x.kmin = g.kmin();
  fft_x<T>(x, g.n, c->st, c->hook());
  if (!lpt) {
    displacement_yz<T>(c, X0, X1, psi, dense, padded, g);
    return;
  }
  for (auto &p : L.psi2) alloc_field(c, p, g);
  T *q[3] = {(T *)L.psi2[0].p, (T *)L.psi2[1].p, (T *)L.psi2[2].p};
  FftY<T> y;
  y.kmin = g.kmin();
  y.add(X2, q[0], FFT_YZ_ONE);
  y.add(X1, psi[0], FFT_YZ_ONE, q[2], FFT_YZ_MIKY);
  y.add(X0, psi[2], FFT_YZ_ONE, psi[1], FFT_YZ_KY, q[1], FFT_YZ_KYKY);
  fft_y<T>(y, g.n, c->st, c->hook());
  fft_z_lpt<T>(psi[0], psi[1], psi[2], q[0], q[1], q[2], X0, true, g.n, g.kmin(), c->st, c->hook());
}

// dense: the differentiable forward map, whose noise has been transformed
// along z and y into the levels' fields; the base level's displacements also
// go to its first three arrays
template <typename T> void do_zeldovich(gic_context *c, T *const *dense) {
  if (!c->power_applied) do_apply_ps<T>(c);
  Phase ph(c, "phase:zeldovich");
  size_t nl = c->levels.size();
  // the levels are independent here; the base level goes last so that its
  // second-order source stays in xhalf
  for (size_t li = nl; li-- > 0;) {
    size_t l = li;
    Level &L = *c->levels[l];
    if (!dense) ensure_noise_fourier<T>(c, L);
    level_displacements<T>(c, l, dense != nullptr, dense && l == 0 ? dense : nullptr);
    if (dense) {
      L.noise_fourier = true;
      L.dc_pending = false;
    }
    if (l >= 1) {
      long h = L.g.n / 2, nent = 3 * h * h + 1;
      c->tab_a.ensure(nent * sizeof(T));
      filter_table<T>(1, kcut_for_level(c, int(l) - 1), L.g.kmin(), nent, (T *)c->tab_a.p, c->st);
      mul_table<T>((T *)L.noise.p, L.g.n, (const T *)c->tab_a.p, c->st);
      to_real<T>(c, L.noise, L.g.n, L.noise_fourier);
    }
    L.psi_fourier = false;
    L.have_psi = !dense || nl > 1;
  }
  // fine <- HP(fine) + interpolate(LP(coarse)), coarse already combined
  for (size_t l = 1; l < nl; ++l) {
    Level &F = *c->levels[l];
    Level &C = *c->levels[l - 1];
    double kc = kcut_for_level(c, int(l) - 1);
    InterpGeom ig = interp_geom(F.g, C.g);
    int w0[3], wl[3];
    coarse_window(F.g, C.g, w0, wl);
    bool pruned = l == 1 && C.noise_fourier && C.g.covers_full() && wl[0] < C.g.n && wl[1] < C.g.n && wl[2] < C.g.n;
    CoarseView view[4];
    const T *lp = nullptr;
    if (pruned) {
      // the base level's delta spectrum is intact: low-pass it (and form
      // psi from it) straight into the coarse window only
      coarse_parts<T>(c, (const T *)C.noise.p, C.g, kc, 1.0, true, w0, wl, c->stage, view);
    } else {
      long h = C.g.n / 2, nent = 3 * h * h + 1;
      c->tab_b.ensure(nent * sizeof(T));
      filter_table<T>(0, kc, C.g.kmin(), nent, (T *)c->tab_b.p, c->st);
      lp = (const T *)c->tab_b.p;
    }
    to_real<T>(c, F.noise, F.g.n, F.noise_fourier);
    for (int f = 0; f < 4; ++f) {   // psi, then delta
      DevBuf &target = f == 3 ? F.noise : F.psi[f];
      if (!pruned) {
        if (f == 3) to_real<T>(c, C.noise, C.g.n, C.noise_fourier);
        view[f] = lowpass_full<T>(c, f == 3 ? C.noise : C.psi[f], C.g, lp);
      }
      // the fine field read and written, the coarse window read once
      double coarse = double(view[f].len[0]) * view[f].len[1] * view[f].len[2];
      Timed t(c, "interp_add", (2.0 * F.g.n3() + coarse) * sizeof(T));
      interp_add<T>((T *)target.p, F.g.n, view[f], ig, c->st);
    }
  }
  if (c->lpt_order == 2) {
    Phase ph2(c, "phase:2lpt");
    do_second_order<T>(c);
  }
  c->zeldovich_done = true;
}

template <typename T> void do_copy_field(gic_context *c, int field, int level, int space, void *host, int dtype) {
  Level &L = level_at(c, level);
  DevBuf *b;
  bool *flag;
  if (field == GIC_FIELD_OVERDENSITY) {
    if (!c->drawn) do_draw<T>(c);
    b = &L.noise;
    flag = &L.noise_fourier;
  } else if (field >= 1 && field <= 3) {
    if (!L.have_psi) throw std::runtime_error("Attempt to generate particles before they have been calculated");
    b = &L.psi[field - 1];
    flag = &L.psi_fourier;
  } else if (field >= 4 && field <= 6) {
    if (!L.have_psi2) throw std::runtime_error("Second-order displacements have not been calculated (lpt_order 2)");
    if (space != GIC_REAL_SPACE) throw std::runtime_error("second-order displacements are held in real space");
    b = &L.psi2[field - 4];
    static bool real_flag;
    real_flag = false;
    flag = &real_flag;
  } else {
    throw std::runtime_error("unknown field");
  }
  int n = L.g.n;
  if (space == GIC_REAL_SPACE) {
    if (field == GIC_FIELD_OVERDENSITY) {
      if (L.dc_pending) ensure_noise_fourier<T>(c, L);
      to_real<T>(c, *b, n, *flag);
    }
    else if (*flag) {
      for (int a = 0; a < 3; ++a) {
        bool f = true;
        to_real<T>(c, L.psi[a], n, f);
      }
      *flag = false;
    }
    size_t n3 = L.g.n3();
    size_t ob = n3 * (dtype == GIC_DTYPE_F32 ? 4 : 8);
    c->stage.ensure(ob);
    if (dtype == GIC_DTYPE_F32) unpad<T, float>((const T *)b->p, n, (float *)c->stage.p, c->st);
    else unpad<T, double>((const T *)b->p, n, (double *)c->stage.p, c->st);
    c->to_host.run({{host, c->stage.p, ob}}, c->st);
  } else {
    if (field == GIC_FIELD_OVERDENSITY) ensure_noise_fourier<T>(c, L);
    else if (!*flag) {
      for (int a = 0; a < 3; ++a) {
        bool f = false;
        to_fourier<T>(c, L.psi[a], n, f);
      }
      *flag = true;
    }
    size_t nreal = L.g.padded_reals();
    size_t ob = nreal * (dtype == GIC_DTYPE_F32 ? 4 : 8);
    c->stage.ensure(ob);
    if (dtype == GIC_DTYPE_F32) convert<T, float>((const T *)b->p, nreal, (float *)c->stage.p, c->st);
    else convert<T, double>((const T *)b->p, nreal, (double *)c->stage.p, c->st);
    c->to_host.run({{host, c->stage.p, ob}}, c->st);
  }
  GIC_HIP(hipStreamSynchronize(c->st));
}

template <typename T> void do_set_field(gic_context *c, int field, int level, int space, const void *host, int dtype) {
  Level &L = level_at(c, level);
  if (field != GIC_FIELD_OVERDENSITY) throw std::runtime_error("only the overdensity / noise field can be set");
  alloc_field(c, L.noise, L.g);
  int n = L.g.n;
  size_t es = dtype == GIC_DTYPE_F32 ? 4 : 8;
  if (space == GIC_REAL_SPACE) {
    size_t ob = L.g.n3() * es;
    c->stage.ensure(ob);
    GIC_HIP(hipMemcpyAsync(c->stage.p, host, ob, hipMemcpyHostToDevice, c->st));
    if (dtype == GIC_DTYPE_F32) pad<float, T>((const float *)c->stage.p, n, (T *)L.noise.p, c->st);
    else pad<double, T>((const double *)c->stage.p, n, (T *)L.noise.p, c->st);
    L.noise_fourier = false;
    L.dc_pending = false;
  } else {
    size_t nreal = L.g.padded_reals();
    c->stage.ensure(nreal * es);
    GIC_HIP(hipMemcpyAsync(c->stage.p, host, nreal * es, hipMemcpyHostToDevice, c->st));
    if (dtype == GIC_DTYPE_F32) convert<float, T>((const float *)c->stage.p, nreal, (T *)L.noise.p, c->st);
    else convert<double, T>((const double *)c->stage.p, nreal, (T *)L.noise.p, c->st);
    L.noise_fourier = true;
    L.dc_pending = false;
  }
  GIC_HIP(hipStreamSynchronize(c->st));
}

// Per-|k|^2 histogram of the overdensity's power and the theory covariance
// P(k) N^3/V for dumpPowerSpectrum (cosmology/parameters.hpp:112-205).  The
// overdensity is transformed on a copy, so the field keeps its space.
template <typename T>
void do_mode_power(gic_context *c, int level, double *sum, double *cnt, double *theory, size_t nm) {
  Level &L = level_at(c, level);
  long h = L.g.n / 2;
  if (nm != size_t(3 * h * h + 1)) throw std::runtime_error("histogram length must be 3(n/2)^2+1");
  if (!c->drawn) do_draw<T>(c);
  if (!c->power_applied) do_apply_ps<T>(c);
  if (L.dc_pending) ensure_noise_fourier<T>(c, L);
  size_t bytes = L.g.padded_reals() * sizeof(T);
  size_t hb = nm * sizeof(double);
  c->stage.ensure(bytes + 2 * hb);
  T *spec = (T *)L.noise.p;
  if (!L.noise_fourier) {
    GIC_HIP(hipMemcpyAsync(c->stage.p, L.noise.p, bytes, hipMemcpyDeviceToDevice, c->st));
    spec = (T *)c->stage.p;
    fft3d<T>(spec, L.g.n, -1, c->st, c->hook());
  }
  double *dsum = (double *)((char *)c->stage.p + bytes);
  double *dcnt = dsum + nm;
  fill<double>(dsum, 2 * nm, 0.0, c->st);
  mode_power<T>(spec, L.g.n, dsum, dcnt, c->st);
  GIC_HIP(hipMemcpyAsync(sum, dsum, hb, hipMemcpyDeviceToHost, c->st));
  GIC_HIP(hipMemcpyAsync(cnt, dcnt, hb, hipMemcpyDeviceToHost, c->st));
  std::vector<T> tab(nm);
  build_sqrtp<T>(c, L);
  GIC_HIP(hipMemcpyAsync(tab.data(), L.sqrtp.p, nm * sizeof(T), hipMemcpyDeviceToHost, c->st));
  GIC_HIP(hipStreamSynchronize(c->st));
  for (size_t m = 0; m < nm; ++m) theory[m] = double(tab[m]) * double(tab[m]);
}

double velocity_ratio(const Cosmo &c) {
  double f = 1.0;
  return f * 100. * sqrt(c.Om / (c.a * c.a * c.a) + c.Ol) * sqrt(c.a);
}

template <typename T>
void do_particles(gic_context *c, int level, const uint64_t *cells, size_t start, size_t count, float *pos,
                  float *vel) {
  Level &L = level_at(c, level);
  if (!L.have_psi) throw std::runtime_error("Attempt to generate particles before they have been calculated");
  if (L.psi_fourier) {
    for (int a = 0; a < 3; ++a) {
      bool f = true;
      to_real<T>(c, L.psi[a], L.g.n, f);
    }
    L.psi_fourier = false;
  }
  size_t n3 = L.g.n3();
  if (cells) {
    for (size_t i = 0; i < count; ++i)
      if (cells[i] >= n3) throw std::out_of_range("particle cell index out of range for the level");
  } else if (start > n3 || count > n3 - start) {
    throw std::out_of_range("particle range exceeds the level's cells");
  }
  ParticleGeom pg;
  pg.dx = L.g.dx;
  pg.o[0] = L.g.ox;
  pg.o[1] = L.g.oy;
  pg.o[2] = L.g.oz;
  pg.periodic = L.g.periodic;
  pg.vratio = velocity_ratio(c->cosmo);
  pg.vratio2 = 2.0 * pg.vratio;   // f2 = 2 f1 (f1 = 1, as zeldovichVelocityToOffsetRatio)
  // device staging: cell list + outputs, processed in slices
  const size_t slice = size_t(1) << 24;
  for (size_t s0 = 0; s0 < count; s0 += slice) {
    size_t m = std::min(slice, count - s0);
    size_t need = m * 24 + (cells ? m * 8 : 0);
    c->stage.ensure(need);
    float *dpos = (float *)c->stage.p;
    float *dvel = dpos + 3 * m;
    uint64_t *dcells = nullptr;
    if (cells) {
      dcells = (uint64_t *)(dvel + 3 * m);
      GIC_HIP(hipMemcpyAsync(dcells, cells + s0, m * 8, hipMemcpyHostToDevice, c->st));
    }
    const T *q2[3] = {(const T *)L.psi2[0].p, (const T *)L.psi2[1].p, (const T *)L.psi2[2].p};
    particles<T>((const T *)L.psi[0].p, (const T *)L.psi[1].p, (const T *)L.psi[2].p, L.have_psi2 ? q2 : nullptr,
                 L.g.n, pg, dcells, start + s0, m,
                 dpos, dvel, c->st);
    c->to_host.run({{pos + 3 * s0, dpos, m * 12}, {vel + 3 * s0, dvel, m * 12}}, c->st);
  }
}

template <typename F> int guarded(gic_context *c, F &&f) {
  if (!c) return 2;
  try {
    GIC_HIP(hipSetDevice(c->device));
    f();
    return 0;
  } catch (std::exception &e) {
    c->err = e.what();
    return 1;
  }
}

#define DISPATCH(c, fn, ...)                  \
  do {                                        \
    if ((c)->prec == 32) fn<float>(__VA_ARGS__); \
    else fn<double>(__VA_ARGS__);             \
  } while (0)

template void build_sqrtp<float>(gic_context *, Level &);
template void build_sqrtp<double>(gic_context *, Level &);
template void build_sqrtp_dm<float>(gic_context *, Level &);
template void build_sqrtp_dm<double>(gic_context *, Level &);
template void do_draw<float>(gic_context *);
template void do_draw<double>(gic_context *);
template void ensure_noise_fourier<float>(gic_context *, Level &);
template void ensure_noise_fourier<double>(gic_context *, Level &);
template void do_zeldovich<float>(gic_context *, float *const *);
template void do_zeldovich<double>(gic_context *, double *const *);

template <typename T> void do_import_level(gic_context *c, int level, const double *host) {
  if (!c->drawn) do_draw<T>(c);
  if (c->power_applied) throw std::runtime_error("import_level acts on the white noise, before the output is generated");
  Level &L = level_at(c, level);
  int n = L.g.n;
  size_t n3 = L.g.n3();
  c->stage.ensure(n3 * sizeof(double));
  GIC_HIP(hipMemcpyAsync(c->stage.p, host, n3 * sizeof(double), hipMemcpyHostToDevice, c->st));
  pad<double, T>((const double *)c->stage.p, n, (T *)L.noise.p, c->st);
  // the file holds a dark-matter overdensity: back to white noise with P_dm^-1/2
  build_sqrtp_dm<T>(c, L);
  long h = n / 2, nent = 3 * h * h + 1;
  c->tab_a.ensure(nent * sizeof(T));
  inverse_table<T>((const T *)L.sqrtp_dm.p, nent, (T *)c->tab_a.p, c->st);
  fft_r2c_post<T>((T *)L.noise.p, n, (const T *)c->tab_a.p, c->st, c->hook());
  L.noise_fourier = true;
  L.dc_pending = false;
  GIC_HIP(hipStreamSynchronize(c->st));
}

}  // namespace gic

extern "C" {

int gic_create(gic_context **out, int device, int precision) {
  if (!out) return 2;
  *out = nullptr;
  if (precision != 32 && precision != 64) return 3;
  auto *c = new gic_context();
  c->device = device;
  c->prec = precision;
  try {
    int ndev = 0;
    GIC_HIP(hipGetDeviceCount(&ndev));
    if (device < 0 || device >= ndev) throw std::runtime_error("no such HIP device");
    GIC_HIP(hipSetDevice(device));
    GIC_HIP(hipStreamCreateWithFlags(&c->st, hipStreamNonBlocking));
    rng_scratch_setup(device);   // the fixed workspace of gic_gaussian_stream_noalloc on this device
  } catch (std::exception &e) {
    delete c;
    return 4;
  }
  *out = c;
  return 0;
}

void gic_destroy(gic_context *c) {
  if (!c) return;
  (void)hipSetDevice(c->device);
  if (c->st) (void)hipStreamSynchronize(c->st);
  c->timer.reset();
  c->levels.clear();
  if (c->st) (void)hipStreamDestroy(c->st);
  delete c;
}

const char *gic_last_error(const gic_context *c) { return c ? c->err.c_str() : "null context"; }

int gic_set_cosmology(gic_context *c, double Om, double Ol, double Ob, double hubble, double s8, double ns, double z) {
  return guarded(c, [&] {
    c->cosmo.Om = Om;
    c->cosmo.Ol = Ol;
    c->cosmo.Ob = Ob;
    c->cosmo.h = hubble;
    c->cosmo.s8 = s8;
    c->cosmo.ns = ns;
    c->cosmo.z = z;
    c->cosmo.a = 1. / (z + 1.);
  });
}

int gic_set_power_law(gic_context *c, double amplitude) {
  return guarded(c, [&] {
    if (!(amplitude > 0) || !std::isfinite(amplitude)) throw std::runtime_error("powerlaw_amplitude must be positive");
    ++c->spectrum;
    c->kpts.clear();
    c->ns_frozen = c->cosmo.ns;
    c->amplitude = amplitude;
    c->spline_dev = SplineHost{};       // n = 0: unit transfer function for every species
    c->spline_dm_dev = SplineHost{};
    c->have_camb = true;
    for (auto &Lp : c->levels) {
      Lp->sqrtp.release();
      Lp->sqrtp_dm.release();
    }
  });
}

int gic_set_camb_table(gic_context *c, const double *v, size_t nv, int ncols) {
  return guarded(c, [&] {
    if (ncols != 7 && ncols != 13) throw std::runtime_error("CAMB transfer file doesn't have a sensible number of columns");
    if (nv < size_t(ncols) * 2) throw std::runtime_error("CAMB transfer file is too short");
    double tnorm = v[1];
    std::vector<double> kp, tall;
    for (size_t j = 0; j < nv / ncols; ++j) {
      if (v[ncols * j] > 0) {
        kp.push_back(v[ncols * j]);
        tall.push_back(v[ncols * j + 6] / tnorm);
      }
    }
    std::vector<double> tdm;
    for (size_t j = 0; j < nv / ncols; ++j)
      if (v[ncols * j] > 0) tdm.push_back(v[ncols * j + 1] / tnorm);
    ++c->spectrum;
    c->kpts = kp;
    c->tf_all = LogSpline();
    c->tf_all.init(kp, tall);
    c->tf_dm = LogSpline();
    c->tf_dm.init(kp, tdm);
    c->ns_frozen = c->cosmo.ns;
    double gf = growth_factor(c->cosmo.a, c->cosmo.Om, c->cosmo.Ol) / growth_factor(1.0, c->cosmo.Om, c->cosmo.Ol);
    double s8pre = variance_in_sphere(c, 8.);
    double lr = (c->cosmo.s8 / s8pre) * gf;
    c->amplitude = lr * lr;
    const Spline &s = c->tf_all.s;
    int n = (int)s.x.size();
    c->spl_x.ensure(n * 8);
    c->spl_y.ensure(n * 8);
    c->spl_c.ensure(n * 8);
    GIC_HIP(hipMemcpy(c->spl_x.p, s.x.data(), n * 8, hipMemcpyHostToDevice));
    GIC_HIP(hipMemcpy(c->spl_y.p, s.y.data(), n * 8, hipMemcpyHostToDevice));
    GIC_HIP(hipMemcpy(c->spl_c.p, s.c.data(), n * 8, hipMemcpyHostToDevice));
    c->spline_dev = SplineHost{(double *)c->spl_x.p, (double *)c->spl_y.p, (double *)c->spl_c.p, n, c->tf_all.minx,
                               c->tf_all.maxx};
    const Spline &sd = c->tf_dm.s;
    int nd = (int)sd.x.size();
    c->spl_dm_x.ensure(nd * 8);
    c->spl_dm_y.ensure(nd * 8);
    c->spl_dm_c.ensure(nd * 8);
    GIC_HIP(hipMemcpy(c->spl_dm_x.p, sd.x.data(), nd * 8, hipMemcpyHostToDevice));
    GIC_HIP(hipMemcpy(c->spl_dm_y.p, sd.y.data(), nd * 8, hipMemcpyHostToDevice));
    GIC_HIP(hipMemcpy(c->spl_dm_c.p, sd.c.data(), nd * 8, hipMemcpyHostToDevice));
    c->spline_dm_dev = SplineHost{(double *)c->spl_dm_x.p, (double *)c->spl_dm_y.p, (double *)c->spl_dm_c.p, nd,
                                  c->tf_dm.minx, c->tf_dm.maxx};
    c->have_camb = true;
  });
}

int gic_init_base_grid(gic_context *c, double box, int n) {
  return guarded(c, [&] {
    if (!c->levels.empty()) throw std::runtime_error("Cannot re-initialize the base grid");
    if (c->drawn) throw std::runtime_error("Trying to initialize a grid after the random field was already drawn");
    if (box <= 0) throw std::runtime_error("Box size must be positive");
    if (n < 4 || (n & (n - 1))) throw std::runtime_error("Grid size must be a power of two >= 4");
    auto L = std::make_unique<Level>();
    L->g.n = n;
    L->g.periodic = box;
    L->g.dx = box / n;
    L->g.box = L->g.dx * n;
    c->levels.push_back(std::move(L));
  });
}

int gic_init_zoom_grid_with_origin_at(gic_context *c, int x0, int y0, int z0, int zoomfac, int n) {
  return guarded(c, [&] {
    if (c->drawn) throw std::runtime_error("Trying to initialize a grid after the random field was already drawn");
    if (c->levels.empty()) throw std::runtime_error("Cannot initialise a zoom grid before initialising the base grid");
    if (c->levels.size() >= 4) throw std::runtime_error("At most 4 levels are supported");
    if (n < 4 || (n & (n - 1))) throw std::runtime_error("Grid size must be a power of two >= 4");
    if (zoomfac < 1) throw std::runtime_error("Zoom factor must be positive");
    const LevelGeom &A = c->levels.back()->g;
    if (x0 < 0 || y0 < 0 || z0 < 0)
      throw std::runtime_error("The newly initialised zoom level is not fully contained within the previous level");
    int nc = A.n / zoomfac;
    if (!A.covers_full() && (x0 + nc > A.n || y0 + nc > A.n || z0 + nc > A.n))
      throw std::runtime_error("The newly initialised zoom level is not fully contained within the previous level");
    auto L = std::make_unique<Level>();
    double size = A.box / zoomfac;
    L->g.n = n;
    L->g.periodic = A.periodic;
    L->g.dx = size / n;
    L->g.box = L->g.dx * n;
    L->g.ox = A.ox + x0 * A.dx;
    L->g.oy = A.oy + y0 * A.dx;
    L->g.oz = A.oz + z0 * A.dx;
    double r = A.dx / L->g.dx;
    if (std::fabs(r - std::round(r)) > 1e-6 || std::round(r) < 1)
      throw std::runtime_error("Zoom cell size must divide the parent cell size");
    c->levels.push_back(std::move(L));
  });
}

int gic_num_levels(gic_context *c, int *out) {
  return guarded(c, [&] { *out = (int)c->levels.size(); });
}

int gic_level_geometry(gic_context *c, int level, int *n, double *box, double *off, double *dx) {
  return guarded(c, [&] {
    const LevelGeom &g = level_at(c, level).g;
    if (n) *n = g.n;
    if (box) *box = g.box;
    if (off) {
      off[0] = g.ox;
      off[1] = g.oy;
      off[2] = g.oz;
    }
    if (dx) *dx = g.dx;
  });
}

int gic_seed(gic_context *c, unsigned long seed, int mode) {
  return guarded(c, [&] {
    if (c->seeded) throw std::runtime_error("The random number generator has already been seeded");
    if (mode < 0 || mode > 3) throw std::runtime_error("unknown seeding mode");
    c->seed = seed;
    c->seed_mode = mode;
    c->seeded = true;
  });
}

int gic_reseed(gic_context *c, unsigned long seed, int mode) {
  return guarded(c, [&] {
    if (mode < 0 || mode > 3) throw std::runtime_error("unknown seeding mode");
    c->seed = seed;
    c->seed_mode = mode;
    c->seeded = true;
    c->drawn = c->power_applied = c->zeldovich_done = false;
    for (auto &L : c->levels) {
      L->noise_fourier = false;
      L->psi_fourier = false;
      L->have_psi = false;
    }
  });
}

int gic_draw(gic_context *c) {
  return guarded(c, [&] { DISPATCH(c, do_draw, c); });
}

int gic_zero_level(gic_context *c, int level) {
  return guarded(c, [&] {
    Level &L = level_at(c, level);
    if (!c->drawn) DISPATCH(c, do_draw, c);
    if (c->prec == 32) fill<float>((float *)L.noise.p, L.g.padded_reals(), 0.f, c->st);
    else fill<double>((double *)L.noise.p, L.g.padded_reals(), 0.0, c->st);
    GIC_HIP(hipStreamSynchronize(c->st));
  });
}

int gic_set_exact_power_spectrum(gic_context *c, int enable) {
  return guarded(c, [&] {
    if (c->drawn) throw std::runtime_error("fix_power must be set before the random field is drawn");
    c->fix_power = enable != 0;
  });
}

int gic_reverse(gic_context *c) {
  return guarded(c, [&] {
    if (!c->drawn) DISPATCH(c, do_draw, c);
    if (c->power_applied) throw std::runtime_error("reverse acts on the white noise, before the output is generated");
    for (auto &Lp : c->levels) {
      if (c->prec == 32) scale_all<float>((float *)Lp->noise.p, Lp->g.padded_reals(), -1.f, c->st);
      else scale_all<double>((double *)Lp->noise.p, Lp->g.padded_reals(), -1.0, c->st);
    }
    GIC_HIP(hipStreamSynchronize(c->st));
  });
}

int gic_reverse_small_k(gic_context *c, double kmax) {
  return guarded(c, [&] {
    if (!c->drawn) DISPATCH(c, do_draw, c);
    if (c->power_applied) throw std::runtime_error("reverse_small_k acts on the white noise, before the output is generated");
    for (auto &Lp : c->levels) {
      Level &L = *Lp;
      if (c->prec == 32) {
        ensure_noise_fourier<float>(c, L);
        reverse_small_k<float>((float *)L.noise.p, L.g.n, L.g.kmin(), kmax, c->st);
      } else {
        ensure_noise_fourier<double>(c, L);
        reverse_small_k<double>((double *)L.noise.p, L.g.n, L.g.kmin(), kmax, c->st);
      }
    }
    GIC_HIP(hipStreamSynchronize(c->st));
  });
}

int gic_import_level(gic_context *c, int level, const double *host, size_t n) {
  return guarded(c, [&] {
    Level &L = level_at(c, level);
    if (!host || n != L.g.n3()) throw std::runtime_error("import_level: the data must hold n^3 values of the level");
    DISPATCH(c, do_import_level, c, level, host);
  });
}

int gic_splice(gic_context *c, unsigned long new_seed, int *cg_iterations) {
  return guarded(c, [&] { DISPATCH(c, do_splice, c, new_seed, cg_iterations); });
}

int gic_apply_power_spectrum(gic_context *c) {
  return guarded(c, [&] {
    DISPATCH(c, do_apply_ps, c);
    GIC_HIP(hipStreamSynchronize(c->st));
  });
}

int gic_zeldovich(gic_context *c) {
  return guarded(c, [&] {
    DISPATCH(c, do_zeldovich, c, nullptr);
    GIC_HIP(hipStreamSynchronize(c->st));
  });
}

int gic_copy_field(gic_context *c, int field, int level, int space, void *host, int dtype) {
  return guarded(c, [&] { DISPATCH(c, do_copy_field, c, field, level, space, host, dtype); });
}

int gic_set_field(gic_context *c, int field, int level, int space, const void *host, int dtype) {
  return guarded(c, [&] {
    DISPATCH(c, do_set_field, c, field, level, space, host, dtype);
    c->drawn = true;
  });
}

int gic_particles(gic_context *c, int level, const uint64_t *cells, size_t start, size_t count, float *pos,
                  float *vel) {
  return guarded(c, [&] { DISPATCH(c, do_particles, c, level, cells, start, count, pos, vel); });
}

int gic_mode_power(gic_context *c, int level, double *sum_power, double *count, double *theory, size_t nm) {
  return guarded(c, [&] { DISPATCH(c, do_mode_power, c, level, sum_power, count, theory, nm); });
}

int gic_particle_mass_eps(gic_context *c, int level, double *mass, double *eps) {
  return guarded(c, [&] {
    const LevelGeom &g = level_at(c, level).g;
    double boxMass = 27.744948 * c->cosmo.Om * pow(g.periodic, 3.0);
    if (mass) *mass = boxMass * pow(g.dx / g.periodic, 3.0);
    if (eps) *eps = g.dx * 1.0 * 0.01075;
  });
}

int gic_set_lpt_order(gic_context *c, int order) {
  return guarded(c, [&] {
    if (order != 1 && order != 2) throw std::runtime_error("LPT order must be 1 or 2");
    c->lpt_order = order;
  });
}

int gic_set_flags(gic_context *c, int level, const uint64_t *cells, size_t n) {
  return guarded(c, [&] {
    Level &L = level_at(c, level);
    c->flags.resize(c->levels.size());
    std::vector<uint64_t> f(cells, cells + n);
    for (uint64_t v : f)
      if (v >= L.g.n3()) throw std::out_of_range("flagged cell index out of range for the level");
    std::sort(f.begin(), f.end());
    f.erase(std::unique(f.begin(), f.end()), f.end());
    c->flags[level] = f;
  });
}

int gic_set_variance_filter_scale(gic_context *c, double scale) {
  return guarded(c, [&] { c->variance_scale = scale; });
}

int gic_calculate(gic_context *c, const char *name, double *out) {
  return guarded(c, [&] {
    if (c->prec == 32) *out = mod_calculate<float>(c, name);
    else *out = mod_calculate<double>(c, name);
  });
}

int gic_add_modification(gic_context *c, const char *name, int relative, double target, int init_steps,
                         double precision) {
  return guarded(c, [&] {
    if (c->prec == 32) mod_add<float>(c, name, relative != 0, target, init_steps, precision);
    else mod_add<double>(c, name, relative != 0, target, init_steps, precision);
  });
}

int gic_apply_modifications(gic_context *c, double *pre_chi2, double *post_chi2) {
  return guarded(c, [&] {
    Phase ph(c, "phase:modifications");
    DISPATCH(c, mod_apply, c, pre_chi2, post_chi2);
  });
}

int gic_clear_modifications(gic_context *c) {
  return guarded(c, [&] { mod_clear(c); });
}

int gic_chi2(gic_context *c, double *chi2, uint64_t *dof) {
  return guarded(c, [&] {
    if (c->prec == 32) *chi2 = mod_chi2<float>(c);
    else *chi2 = mod_chi2<double>(c);
    if (dof) *dof = num_dof(c);
  });
}

int gic_displacement_forward(gic_context *c, const void *const *noise, void *const *psi) {
  return guarded(c, [&] {
    if (!noise || !psi) throw std::runtime_error("displacement forward: null pointer array");
    if (c->prec == 32) do_displacement_forward<float>(c, (const float *const *)noise, (float *const *)psi);
    else do_displacement_forward<double>(c, (const double *const *)noise, (double *const *)psi);
  });
}

int gic_batch_constrained(gic_context *c, int nreal, const uint64_t *seeds, int ncons, const double *cons,
                          void *out, int lanes, int /*use_graph*/, double *elapsed_ms) {
  return guarded(c, [&] {
    if (c->prec == 32) do_batch<float>(c, nreal, seeds, ncons, cons, (float *)out, lanes, elapsed_ms);
    else do_batch<double>(c, nreal, seeds, ncons, cons, (double *)out, lanes, elapsed_ms);
  });
}

int gic_displacement_adjoint(gic_context *c, const void *const *psi_bar, void *const *noise_bar) {
  return guarded(c, [&] {
    if (!psi_bar || !noise_bar) throw std::runtime_error("displacement adjoint: null pointer array");
    if (c->prec == 32) do_displacement_adjoint<float>(c, (const float *const *)psi_bar, (float *const *)noise_bar);
    else do_displacement_adjoint<double>(c, (const double *const *)psi_bar, (double *const *)noise_bar);
  });
}

int gic_masked_displacement(gic_context *c, const void *noise, const uint8_t *mask, double *value, void *grad) {
  return guarded(c, [&] {
    if (!value) throw std::runtime_error("masked displacement: null pointer");
    if (c->prec == 32) *value = do_masked_displacement<float>(c, (const float *)noise, mask, (float *)grad);
    else *value = do_masked_displacement<double>(c, (const double *)noise, mask, (double *)grad);
  });
}

int gic_variance_gradient(gic_context *c, const void *const *noise, double *value, void *const *grad) {
  return guarded(c, [&] {
    if (!noise || !value) throw std::runtime_error("variance gradient: null pointer");
    if (c->prec == 32) *value = mod_variance_gradient<float>(c, (const float *const *)noise, (float *const *)grad);
    else *value = mod_variance_gradient<double>(c, (const double *const *)noise, (double *const *)grad);
  });
}

int gic_set_quadratic_line_search(gic_context *c, int enable) {
  return guarded(c, [&] { mod_set_line_search(c, enable != 0); });
}

int gic_velocity_ratio(gic_context *c, double *out) {
  return guarded(c, [&] { *out = velocity_ratio(c->cosmo); });
}

int gic_fft_inplace(gic_context *c, void *dev, int n, int direction) {
  return guarded(c, [&] {
    if (direction != -1 && direction != 1) throw std::runtime_error("direction must be -1 or +1");
    if (c->prec == 32) fft3d<float>((float *)dev, n, direction, c->st, c->hook());
    else fft3d<double>((double *)dev, n, direction, c->st, c->hook());
    GIC_HIP(hipStreamSynchronize(c->st));
  });
}

int gic_raw_stream(gic_context *c, unsigned long seed, uint32_t *host_out, size_t n) {
  return guarded(c, [&] {
    RngPlan plan;
    rng_plan(seed, n / 2 + 1, plan);
    DevBuf out;
    out.ensure(n * 4);
    rng_raw(plan, (uint32_t *)out.p, n, c->st);
    GIC_HIP(hipMemcpyAsync(host_out, out.p, n * 4, hipMemcpyDeviceToHost, c->st));
    GIC_HIP(hipStreamSynchronize(c->st));
  });
}

int gic_gaussian_stream(gic_context *c, unsigned long seed, double *host_out, size_t n) {
  return guarded(c, [&] {
    if (n == 0) return;
    RngPlan plan;
    rng_plan(seed, n, plan);
    c->work.ensure(rng_workspace_bytes(plan));
    DevBuf dense;
    dense.ensure(n * 8);
    std::vector<RngLevelOut> outs{{dense.p, 0, n}};
    rng_draw_real<double>(plan, outs, c->work.p, c->work.bytes, c->st, c->hook());
    GIC_HIP(hipMemcpyAsync(host_out, dense.p, n * 8, hipMemcpyDeviceToHost, c->st));
    GIC_HIP(hipStreamSynchronize(c->st));
  });
}

int gic_gaussian_stream_noalloc(gic_context *c, unsigned long seed, double *device_out, size_t n) {
  return guarded(c, [&] {
    if (n == 0) return;
    if (!device_out) throw std::runtime_error("gic_gaussian_stream_noalloc: no output array");
    rng_gaussians_noalloc(c->device, seed, device_out, n, c->st);
    GIC_HIP(hipStreamSynchronize(c->st));
  });
}

int gic_synchronize(gic_context *c) {
  return guarded(c, [&] { GIC_HIP(hipStreamSynchronize(c->st)); });
}

int gic_set_event_timing(gic_context *c, int enable) {
  return guarded(c, [&] {
    if (enable && !c->timer) c->timer = std::make_unique<EventTimer>();
    if (!enable) c->timer.reset();
  });
}

int gic_get_event_timing(gic_context *c, const char *kernel, double *total_ms, long *count) {
  return guarded(c, [&] {
    if (!c->timer) throw std::runtime_error("event timing is not enabled");
    c->timer->collect();
    auto it = c->timer->totals.find(kernel);
    *total_ms = it == c->timer->totals.end() ? 0.0 : it->second.first;
    *count = it == c->timer->totals.end() ? 0 : it->second.second;
  });
}

int gic_reset_event_timing(gic_context *c) {
  return guarded(c, [&] {
    if (c->timer) {
      c->timer->collect();
      c->timer->totals.clear();
      c->timer->algo_bytes.clear();
    }
  });
}

int gic_list_event_timing(gic_context *c, char *buf, size_t buflen, size_t *needed) {
  return guarded(c, [&] {
    if (!c->timer) throw std::runtime_error("event timing is not enabled");
    c->timer->collect();
    std::string s;
    char line[256];
    for (auto &kv : c->timer->totals) {
      auto ab = c->timer->algo_bytes.find(kv.first);
      double b = ab == c->timer->algo_bytes.end() ? 0.0 : ab->second;
      snprintf(line, sizeof line, "%s\t%.6f\t%ld\t%.0f\n", kv.first.c_str(), kv.second.first, kv.second.second, b);
      s += line;
    }
    if (needed) *needed = s.size() + 1;
    if (buf && buflen) {
      size_t m = std::min(buflen - 1, s.size());
      memcpy(buf, s.data(), m);
      buf[m] = 0;
    }
  });
}

int gic_device_bytes(gic_context *c, size_t *out) {
  return guarded(c, [&] { *out = total_bytes(c); });
}

}  // extern "C"
