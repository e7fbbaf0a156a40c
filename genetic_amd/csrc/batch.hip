// Batches of independent constrained realisations of one single-level grid.
//
// The reference makes one realisation per run: the draw
// (randomfieldgenerator.hpp:122-139, 181-197), linear modifications
// (linearmodification.hpp, modificationmanager.hpp:160-312), the transfer
// function (field.hpp:394-412) and the Zel'dovich displacement
// (zeldovich.hpp:152-253).  Here many seeds, each with its own set of top-hat
// overdensity constraints, run as one sequence of device work with no host
// synchronisation inside; every launch works on several realisations:
//   w      = draw(seed)                          (the stream of gic_draw)
//   c_i    = sqrtP_dm r2c(1_{S_i})               (the realisation's constraints in one batched r2c)
//   G_ij   = <c_i, c_j>,  d_i = <c_i, w>         (FP64 sums, one pass over all vectors)
//   x      = (G_ij / N_i N_j)^-1 (t_i - d_i / N_i)  (FP64 Cholesky on the device, N_i = |S_i|)
//   delta  = sqrtP (w + sum_i x_i c_i / N_i)
//   out    = c2r(delta), c2r(i k_a delta / k^2)   (dense n^3 arrays)
// S_i is ICGenerator::select with a sphere (ic.hpp:1458-1500): the cells whose
// centroids lie closer than the radius (as a float) to the centre, with
// box-wrapped offsets.  The covector of the mean overdensity in S_i is
// 1_{S_i} / N_i (linearmodification.hpp, OverdensityModification), carried to
// white-noise space by sqrtP_dm; the Gram solve is the Hoffman-Ribak
// correction of modificationmanager.hpp:160-172,266-283.
#include "context.h"

namespace gic {

namespace {

constexpr int MAXCONS = 32;        // constraints per realisation
constexpr int GRAM_THREADS = 256;
constexpr int GRAM_BLOCKS = 512;

__device__ __forceinline__ double stored_mode_weight(int x, int y, int z, int h) {
  // each conjugate pair once: the kz = 0 and kz = N/2 planes hold both halves
  if (z > 0 && z < h) return 2;
  if (x > 0 && x < h) return 2;
  if (x > h) return 0;
  if (y > 0 && y < h) return 2;
  if (y > h) return 0;
  return 1;
}

// 1 on the cells of each constraint's sphere, 0 elsewhere (padding included);
// cnt[f] += the number of cells.  The whole-field form, for spheres too large
// for a box.
template <typename T>
__global__ __launch_bounds__(256) void k_batch_tophat(T *__restrict__ cov, long fs, int n, double dx, double ox,
                                                      double oy, double oz, double periodic,
                                                      const double *__restrict__ cons, uint32_t *__restrict__ cnt) {
#pragma clang fp contract(off)
  int f = blockIdx.y;
  // 32-bit index arithmetic: a field holds n^2 (n+2) < 2^31 values for n <= 1024
  unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  unsigned tot = unsigned(n) * unsigned(n) * unsigned(n + 2);
  bool inside = false;
  bool live = i < tot;
  if (live) {
    unsigned row = i / unsigned(n + 2);
    int z = int(i - row * unsigned(n + 2));
    int x = int(row / unsigned(n)), y = int(row - unsigned(x) * unsigned(n));
    if (z < n) {
      const double *q = cons + 5 * f;
      double half = periodic / 2;
      auto off = [&](int idx, double o, double c) {
        double r = double(idx) * dx;
        r = r + o;
        r = r + dx / 2;
        r = r - c;
        if (r > half) r -= periodic;
        if (r < -half) r += periodic;
        return r;
      };
      double rx = off(x, ox, q[0]), ry = off(y, oy, q[1]), rz = off(z, oz, q[2]);
      float rf = float(q[3]);
      float rr = rf * rf;
      double d2 = rx * rx + ry * ry;
      d2 = d2 + rz * rz;
      inside = d2 < double(rr);
    }
  }
  unsigned long long m = __ballot(inside);
  if ((threadIdx.x & 63) == 0 && m) atomicAdd(cnt + f, uint32_t(__popcll(m)));
  if (live) cov[size_t(f) * fs + i] = inside ? T(1) : T(0);
}

// The rows of each constraint's box (wl x wl cells in x, y from (winx[f],
// winy[f]) mod n, all z): 1 on the cells of the sphere, 0 elsewhere; row
// (f wl + i) wl + j is x = winx[f]+i, y = winy[f]+j.
// cnt[f] += the number of cells of constraint f.  The box holds every selected cell: a cell is selected only if its centroid
// lies within the radius of the centre, and the box spans the centre's
// +-radius with a cell to spare.
template <typename T>
__global__ __launch_bounds__(256) void k_batch_box_rows(T *__restrict__ rows, unsigned nrows, int wl, int n,
                                                        double dx, double ox, double oy, double oz, double periodic,
                                                        const double *__restrict__ cons, const int *__restrict__ winx,
                                                        const int *__restrict__ winy, uint32_t *__restrict__ cnt) {
#pragma clang fp contract(off)
  unsigned e = blockIdx.x * blockDim.x + threadIdx.x;
  bool live = e < nrows * unsigned(n);
  unsigned row = live ? e / unsigned(n) : 0u;
  int z = live ? int(e - row * unsigned(n)) : 0;
  unsigned ww = unsigned(wl) * unsigned(wl);
  int f = int(row / ww);
  bool inside = false;
  if (live) {
    unsigned r2 = row - unsigned(f) * ww;
    int i = int(r2 / unsigned(wl)), j = int(r2 - unsigned(i) * unsigned(wl));
    int x = (winx[f] + i) % n, y = (winy[f] + j) % n;
    const double *q = cons + 5 * f;
    double half = periodic / 2;
    auto off = [&](int idx, double o, double c) {
      double r = double(idx) * dx;
      r = r + o;
      r = r + dx / 2;
      r = r - c;
      if (r > half) r -= periodic;
      if (r < -half) r += periodic;
      return r;
    };
    double rx = off(x, ox, q[0]), ry = off(y, oy, q[1]), rz = off(z, oz, q[2]);
    float rf = float(q[3]);
    float rr = rf * rf;
    double d2 = rx * rx + ry * ry;
    d2 = d2 + rz * rz;
    inside = d2 < double(rr);
  }
  // one atomic per wavefront when its lanes share a constraint
  int f0 = __shfl(f, 0);
  unsigned long long m = __ballot(inside);
  if (__all(!live || f == f0)) {
    if ((threadIdx.x & 63) == 0 && m) atomicAdd(cnt + f0, uint32_t(__popcll(m)));
  } else if (inside) {
    atomicAdd(cnt + f, 1u);
  }
  if (live) rows[e] = inside ? T(1) : T(0);
}

// where the product of v_i and v_j (i >= j) sits among the tile sums
__device__ __forceinline__ int gram_slot(int i, int j) {
  int ti = i >> 2, tj = j >> 2;
  return ((ti * (ti + 1) / 2 + tj) << 4) + ((i & 3) << 2) + (j & 3);
}

// Partial sums of the products of the covectors c_i among themselves and with
// the field w, weighted by the stored-mode weights, in FP64: a contraction
// over modes with matrix instructions, covectors in NB blocks of 16 rows.
// Lane l reads 16 bytes of covector l % 16 of a block (2 FP32 modes or 1 FP64
// mode), l / 16 apart, straight from memory; each of their components is one
// k of a 16 x 16 x 4 product, the same registers serving as both operands (A
// times the weight).  A wavefront's loads are whole 64-byte pieces of each
// covector, so nothing goes through LDS.  Block b of the grid writes the
// products in gram_slot's order (0 where there is none) to its own piece of part.
//
// It is bound by reading the covectors: 8 realisations of 16 at 128^3 FP32,
// 1.16 GB, 298 us (3.9 TB/s); with tiles of 4 x 4 products in vector registers,
// their operands widened from LDS for each, 726 us.  5 of 3 at 64^3 FP64: 27 us,
// 270 before, when most threads had no tile.
typedef double gram_acc __attribute__((ext_vector_type(4)));
template <typename T> struct GramVec;
template <> struct GramVec<float> {
  typedef float type __attribute__((ext_vector_type(4)));
};
template <> struct GramVec<double> {
  typedef double type __attribute__((ext_vector_type(2)));
};

template <typename T, int NB>
__global__ __launch_bounds__(GRAM_THREADS) void k_batch_gram(const cx<T> *__restrict__ cov, long fs,
                                                             const cx<T> *__restrict__ w, int nm, int n,
                                                             double *__restrict__ part) {
  using V = typename GramVec<T>::type;
  constexpr int MPL = 16 / int(sizeof(cx<T>)), C = 2 * MPL;   // modes and components of a lane's load
  constexpr int U = 2, STEP = 4 * MPL, PAIRS = NB * (NB + 1) / 2;
  cov += size_t(blockIdx.y) * nm * fs;
  w += size_t(blockIdx.y) * fs;
  const int h = n / 2, lane = int(threadIdx.x) % 64, row = lane % 16, kk = lane / 16;
  const unsigned nz = unsigned(h + 1), nmodes = unsigned(n) * unsigned(n) * nz;   // a multiple of STEP: n >= 4
  const unsigned wave = blockIdx.x * (GRAM_THREADS / 64) + threadIdx.x / 64, waves = gridDim.x * (GRAM_THREADS / 64);
  const cx<T> *v[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) v[b] = cov + size_t(min(16 * b + row, nm - 1)) * fs;
  gram_acc acc[PAIRS];
  double dot[NB];
#pragma unroll
  for (int p = 0; p < PAIRS; ++p) acc[p] = gram_acc{0, 0, 0, 0};
#pragma unroll
  for (int b = 0; b < NB; ++b) dot[b] = 0;
  for (unsigned m0 = wave * (U * STEP); m0 < nmodes; m0 += waves * (U * STEP)) {
    V x[U][NB], y[U];
    unsigned m[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      m[u] = m0 + u * STEP + kk * MPL;
      const unsigned at = min(m[u], nmodes - MPL);   // past the end: weight 0
#pragma unroll
      for (int b = 0; b < NB; ++b) x[u][b] = *reinterpret_cast<const V *>(v[b] + at);
      y[u] = *reinterpret_cast<const V *>(w + at);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      double wt[MPL];
#pragma unroll
      for (int q = 0; q < MPL; ++q) {
        const unsigned mq = m[u] + q, r = mq / nz;
        wt[q] = mq < nmodes ? stored_mode_weight(int(r / unsigned(n)), int(r % unsigned(n)), int(mq - r * nz), h) : 0.0;
      }
#pragma unroll
      for (int c = 0; c < C; ++c) {
        double a[NB], aw[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          a[b] = double(x[u][b][c]);
          aw[b] = a[b] * wt[c / 2];
          dot[b] += aw[b] * double(y[u][c]);
        }
#pragma unroll
        for (int bi = 0; bi < NB; ++bi)
#pragma unroll
          for (int bj = 0; bj <= bi; ++bj) {
            const int p = bi * (bi + 1) / 2 + bj;
            acc[p] = __builtin_amdgcn_mfma_f64_16x16x4f64(aw[bi], a[bj], acc[p], 0, 0, 0);
          }
      }
    }
  }
  // the wavefronts of the block one after the other: a fixed order of the sums
  __shared__ double red[PAIRS * 256 + NB * 16];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    dot[b] += __shfl_xor(dot[b], 16);
    dot[b] += __shfl_xor(dot[b], 32);
  }
  for (int e = int(threadIdx.x); e < PAIRS * 256 + NB * 16; e += GRAM_THREADS) red[e] = 0;
  __syncthreads();
  for (int g = 0; g < GRAM_THREADS / 64; ++g) {
    if (int(threadIdx.x) / 64 == g) {
      // register r of lane l holds row 4 r + l / 16, column l % 16
#pragma unroll
      for (int p = 0; p < PAIRS; ++p)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[p * 256 + (4 * r + kk) * 16 + row] += acc[p][r];
      if (kk == 0) {
#pragma unroll
        for (int b = 0; b < NB; ++b) red[PAIRS * 256 + 16 * b + row] += dot[b];
      }
    }
    __syncthreads();
  }
  const int nt = (nm + 4) / 4, np = nt * (nt + 1) / 2 * 16;
  part += (size_t(blockIdx.y) * gridDim.x + blockIdx.x) * np;
  for (int e = int(threadIdx.x); e < np; e += GRAM_THREADS) {
    int ti = 0;
    while ((ti + 1) * (ti + 2) / 2 <= e / 16) ++ti;
    const int i = 4 * ti + (e % 16) / 4, j = 4 * (e / 16 - ti * (ti + 1) / 2) + e % 4;
    double s = 0;
    if (i < nm && j < nm) {   // j's block is i's or one before
      const int bi = i / 16, bj = j / 16;
      s = red[(bi * (bi + 1) / 2 + bj) * 256 + (i % 16) * 16 + j % 16];
    } else if (i == nm && j < nm) {
      s = red[PAIRS * 256 + j];
    }
    part[e] = s;
  }
}

// sums[p] = sum over blocks of part[b * np + p], one block per pair, fixed order
__global__ __launch_bounds__(256) void k_batch_reduce(const double *__restrict__ part, int nblk, int np,
                                                      double *__restrict__ sums) {
  __shared__ double sh[256];
  int p = blockIdx.x;
  part += size_t(blockIdx.y) * nblk * np;
  sums += size_t(blockIdx.y) * np;
  double s = 0;
  for (int b = threadIdx.x; b < nblk; b += 256) s += part[size_t(b) * np + p];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (threadIdx.x < k) sh[threadIdx.x] += sh[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) sums[p] = sh[0];
}

// The FP64 solve of one realisation on one wavefront, lane i holding row i
// (nm <= MAXCONS): G = L L^T by right-looking Cholesky with the column
// broadcast by lane shuffles, then L y = t - d / N and L^T x = y;
// coef_i = x_i / N_i.  *flag gets 2 if a constraint selects no cell, 4 if
// the constraints are not linearly independent (the RNG coverage check uses
// 1); either leaves the coefficients at 0.
__global__ __launch_bounds__(64) void k_batch_solve(const double *__restrict__ sums, const uint32_t *__restrict__ cnt,
                                                    const double *__restrict__ cons, int nm, int np,
                                                    double *__restrict__ coef, uint32_t *__restrict__ flag) {
  __shared__ double Ls[MAXCONS * MAXCONS];
  sums += size_t(blockIdx.x) * np;
  cnt += size_t(blockIdx.x) * nm;
  cons += size_t(blockIdx.x) * nm * 5;
  coef += size_t(blockIdx.x) * nm;
  flag += blockIdx.x;
  const int i = threadIdx.x;
  const bool row = i < nm;
  const uint32_t ni = row ? cnt[i] : 1u;
  if (row) coef[i] = 0;
  if (__ballot(ni == 0u)) {
    if (i == 0) *flag |= 2u;
    return;
  }
  const double inv = 1.0 / double(ni);
  double a[MAXCONS];
#pragma unroll
  for (int j = 0; j < MAXCONS; ++j) {
    double invj = __shfl(inv, j);
    a[j] = (row && j <= i) ? sums[gram_slot(i, j)] * inv * invj : 0.0;
  }
  // constant trip counts (k < nm as a predicate) keep a[] in registers
#pragma unroll
  for (int k = 0; k < MAXCONS; ++k) {
    const bool act = k < nm;
    double dkk = __shfl(a[k], k);
    if (act && !(dkk > 0)) {
      if (i == 0) *flag |= 4u;
      if (row) coef[i] = 0;
      return;
    }
    double lkk = act ? sqrt(dkk) : 1.0;
    if (act && i == k) a[k] = lkk;
    if (act && i > k) a[k] /= lkk;
#pragma unroll
    for (int j = k + 1; j < MAXCONS; ++j) {
      double ljk = __shfl(a[k], j);
      if (act && i >= j) a[j] -= a[k] * ljk;
    }
  }
  // forward substitution, column by column
  double y = row ? cons[5 * i + 4] - sums[gram_slot(nm, i)] * inv : 0.0;
#pragma unroll
  for (int k = 0; k < MAXCONS; ++k) {
    const bool act = k < nm;
    double yk = __shfl(y / a[k], k);
    if (act && i == k) y = yk;
    if (act && i > k) y -= a[k] * yk;
  }
  if (row) {
#pragma unroll
    for (int j = 0; j < MAXCONS; ++j)
      if (j <= i) Ls[i * MAXCONS + j] = a[j];
  }
  __syncthreads();
  // back substitution with L^T: x_k final once rows above it are folded in
  for (int k = nm - 1; k >= 0; --k) {
    double xk = __shfl(y / Ls[k * MAXCONS + k], k);
    if (i == k) y = xk;
    if (i < k) y -= Ls[k * MAXCONS + i] * xk;
  }
  if (row) coef[i] = y * inv;
}

// w <- sqrtP (w + sum_i coef_i c_i), mode by mode
template <typename T>
__global__ __launch_bounds__(256) void k_batch_update(cx<T> *__restrict__ w, const cx<T> *__restrict__ cov, long fs,
                                                      int nm, const double *__restrict__ coef,
                                                      const T *__restrict__ sqrtp, int n) {
  __shared__ T s[MAXCONS];
  w += size_t(blockIdx.y) * fs;
  cov += size_t(blockIdx.y) * nm * fs;
  coef += size_t(blockIdx.y) * nm;
  if (threadIdx.x < nm) s[threadIdx.x] = T(coef[threadIdx.x]);
  __syncthreads();
  size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  size_t nmodes = size_t(n) * n * (n / 2 + 1);
  if (i >= nmodes) return;
  cx<T> v = w[i];
  for (int j = 0; j < nm; ++j) {
    cx<T> c = cov[size_t(j) * fs + i];
    v.x += s[j] * c.x;
    v.y += s[j] * c.y;
  }
  int h = n / 2;
  int iz = int(i % size_t(h + 1));
  size_t r = i / size_t(h + 1);
  int iy = int(r % size_t(n)), ix = int(r / size_t(n));
  if (ix > h) ix -= n;
  if (iy > h) iy -= n;
  T f = sqrtp[ix * ix + iy * iy + iz * iz];
  w[i] = cx<T>{v.x * f, v.y * f};
}

// Re(w_0) = 0 of each spectrum (randomfieldgenerator.hpp:194-195)
template <typename T> __global__ void k_batch_dc(cx<T> *__restrict__ w, long fs, int nb) {
  int g = threadIdx.x;
  if (g < nb) w[size_t(g) * fs].x = T(0);
}

}  // namespace

// Device memory of a batch's groups, kept for the next call
struct BatchState {
  DevBuf cons, flags, win, plans, rng_ws;
  DevBuf w, cov, part, sums, cnt, coef;
  DevBuf rows, zbuf, ybuf;   // covectors from the constraints' boxes
};

// Realisations per launch: up to GROUP_MAX, while a group's covectors take no
// more than GROUP_BYTES; at least the concurrency the caller asks for.
constexpr int GROUP_MAX = 16;
constexpr double GROUP_BYTES = 192e6;
// A realisation's fields in the groups' buffers: its noise, and the
// covectors, over which the four fields of its output are made.
static int batch_fields(int ncons) { return 1 + std::max(ncons, 4); }
// Wavefronts of a draw (240 MB of chunk states, 32 for every SIMD); more
// realisations than they hold are drawn one part after the other.
constexpr long DRAW_SEGS = 32768;

template <typename T>
void do_batch(gic_context *c, int nreal, const uint64_t *seeds, int ncons, const double *cons, T *out, int nlanes,
              double *ms) {
  if (c->levels.size() != 1) throw std::runtime_error("batched realisations need exactly one grid level");
  if (!c->have_camb) throw std::runtime_error("No power spectrum has been set (use the camb command)");
  if (nreal < 1 || !seeds || !out) throw std::runtime_error("batch: no realisations, seeds or output");
  if (ncons < 1 || ncons > MAXCONS || !cons)
    throw std::runtime_error("batch: between 1 and " + std::to_string(MAXCONS) + " constraints per realisation");
  if (nlanes < 1 || nlanes > 16) throw std::runtime_error("batch: 1 to 16 concurrent chains");
  for (int i = 0; i < nreal * ncons; ++i)
    if (!(cons[5 * i + 3] > 0) || !std::isfinite(cons[5 * i + 4]))
      throw std::runtime_error("batch: each constraint needs a positive radius and a finite target");
  Level &L = *c->levels[0];
  const LevelGeom &g = L.g;
  const int n = g.n;
  const long fs_reals = long(g.padded_reals());
  const long fs = long(g.nmodes());   // complex elements per padded field
  const size_t n3 = g.n3();
  const int ntile = (ncons + 1 + 3) / 4;
  const int np = ntile * (ntile + 1) / 2 * 16;   // tile sums of the Gram kernel

  hipEvent_t t0 = nullptr, t1 = nullptr;
  if (ms) {
    GIC_HIP(hipEventCreate(&t0));
    GIC_HIP(hipEventCreate(&t1));
    GIC_HIP(hipEventRecord(t0, c->st));
  }
  build_sqrtp<T>(c, L);
  build_sqrtp_dm<T>(c, L);
  if (!c->batch) c->batch = std::make_shared<BatchState>();
  BatchState &B = *c->batch;
  // The realisations' streams, in as few draws as DRAW_SEGS allows: each goes,
  // dense, into the first of its output arrays, which its transform reads.
  auto plan_of = [&](int r0, int k) {
    std::vector<RngStream> streams;
    for (int r = r0; r < r0 + k; ++r) streams.push_back({(unsigned long)seeds[r], n3, size_t(r) * 4 * n3});
    RngPlan p;
    rng_plan(streams, p);
    return p;
  };
  std::vector<RngPlan> draws{plan_of(0, nreal)};
  if (draws[0].nseg > DRAW_SEGS) {
    const int k = std::max(1, int(double(nreal) * DRAW_SEGS / double(draws[0].nseg)));
    draws.clear();
    for (int r = 0; r < nreal; r += k) draws.push_back(plan_of(r, std::min(k, nreal - r)));
  }
  std::vector<size_t> plan_at(1, 0);
  for (auto &p : draws) {
    B.rng_ws.ensure(rng_workspace_bytes(p));
    plan_at.push_back(plan_at.back() + rng_dev_bytes(p));
  }
  // boxes around the spheres: x, y windows of wl cells from
  // floor((c - o - R)/dx - 1/2) (mod n), which hold every selected cell
  int wl = 0;
  for (int q = 0; q < nreal * ncons; ++q) {
    double span = 2.0 * std::ceil(cons[5 * q + 3] / g.dx) + 3.0;
    wl = std::max(wl, span >= double(n) ? n : int(span));
  }
  // (the row kernel indexes rows x n values in 32 bits)
  const bool boxes = wl < n && double(ncons) * wl * wl * n < 2e9;
  // (with fewer than four constraints the output's fields decide: no more
  // memory than ncons + 3 fields for each of the caller's lanes)
  const int lanes = std::max(1, std::min(nlanes, nlanes * (ncons + 3) / batch_fields(ncons)));
  int group = std::max(lanes, std::min(GROUP_MAX, int(GROUP_BYTES / (double(ncons) * fs_reals * sizeof(T)))));
  group = std::min(group, nreal);
  if (boxes) group = std::min(group, int(2e9 / (double(ncons) * wl * wl * n)));
  auto nrows_of = [&](int k) { return boxes ? long(k) * ncons * wl * wl : 0; };
  // the boxes' x origins of every constraint, then the y origins
  std::vector<int> win(boxes ? size_t(nreal) * ncons * 2 : 0);
  if (boxes) {
    const double org[2] = {g.ox, g.oy};
    for (int a = 0; a < 2; ++a)
      for (int q = 0; q < nreal * ncons; ++q) {
        long w0 = long(std::floor((cons[5 * q + a] - org[a] - cons[5 * q + 3]) / g.dx - 0.5));
        w0 %= n;
        if (w0 < 0) w0 += n;
        win[size_t(a) * nreal * ncons + q] = int(w0);
      }
    B.rows.ensure(size_t(nrows_of(group)) * n * sizeof(T));
    B.zbuf.ensure(size_t(nrows_of(group)) * (n + 2) * sizeof(T));
    B.ybuf.ensure(size_t(group) * ncons * wl * n * (n + 2) * sizeof(T));
  }
  B.w.ensure(size_t(group) * fs_reals * sizeof(T));
  B.cov.ensure(size_t(group) * (batch_fields(ncons) - 1) * fs_reals * sizeof(T));
  B.part.ensure(size_t(group) * GRAM_BLOCKS * np * sizeof(double));
  B.sums.ensure(size_t(group) * np * sizeof(double));
  B.cnt.ensure(size_t(group) * ncons * sizeof(uint32_t));
  B.coef.ensure(size_t(group) * ncons * sizeof(double));
  B.cons.ensure(size_t(nreal) * ncons * 5 * sizeof(double));
  B.flags.ensure(size_t(nreal) * sizeof(uint32_t));
  GIC_HIP(hipMemcpyAsync(B.cons.p, cons, size_t(nreal) * ncons * 5 * sizeof(double), hipMemcpyHostToDevice, c->st));
  if (boxes) {
    B.win.ensure(win.size() * sizeof(int));
    GIC_HIP(hipMemcpyAsync(B.win.p, win.data(), win.size() * sizeof(int), hipMemcpyHostToDevice, c->st));
  }
  fill<uint32_t>((uint32_t *)B.flags.p, size_t(nreal), 0u, c->st);
  std::vector<char> hplan(plan_at.back(), 0);
  for (size_t i = 0; i < draws.size(); ++i) rng_dev_pack(draws[i], hplan.data() + plan_at[i]);
  B.plans.ensure(hplan.size());
  GIC_HIP(hipMemcpyAsync(B.plans.p, hplan.data(), hplan.size(), hipMemcpyHostToDevice, c->st));

  hipStream_t st = c->st;
  TimingHook *hook = c->hook();
  const double *dcons = (const double *)B.cons.p;
  uint32_t *dflags = (uint32_t *)B.flags.p;
  size_t drawn = 0;
  for (size_t i = 0; i < draws.size(); ++i) {
    rng_draw_real<T>(draws[i], {{out, 0, size_t(nreal) * 4 * n3}}, B.rng_ws.p, B.rng_ws.bytes, st, hook, 1.0,
                     dflags + drawn, 1, (const char *)B.plans.p + plan_at[i]);
    drawn += draws[i].streams.size();
  }
  for (int r0 = 0; r0 < nreal; r0 += group) {
    const int nb = std::min(group, nreal - r0), nc = nb * ncons;
    T *w = (T *)B.w.p, *cv = (T *)B.cov.p, *o = out + size_t(r0) * 4 * n3;
    const double *rc = dcons + size_t(r0) * ncons * 5;
    // the white noise's spectra
    FftZFwd<T> zf;
    zf.add(o, w, true);
    zf.nb = nb;
    zf.src_bs = long(4 * n3);
    zf.out_bs = fs_reals;
    fft_z_forward<T>(zf, n, st, hook);
    FftYFwd<T> yf;
    yf.add(w, nullptr, w);
    yf.nb = nb;
    yf.bs = fs_reals;
    fft_y_forward<T>(yf, n, st, hook);
    FftX<T> xf;
    xf.in = xf.spec = w;
    xf.forward = true;
    xf.nb = nb;
    xf.in_bs = xf.spec_bs = fs_reals;
    xf.kmin = g.kmin();
    fft_x<T>(xf, n, st, hook);
    hipLaunchKernelGGL(k_batch_dc<T>, dim3(1), dim3(64), 0, st, reinterpret_cast<cx<T> *>(w), fs, nb);
    GIC_HIP(hipGetLastError());
    // the constraints' covectors in white-noise space
    fill<uint32_t>((uint32_t *)B.cnt.p, size_t(nc), 0u, st);
    if (boxes) {
      const int *wx = (const int *)B.win.p + size_t(r0) * ncons, *wy = wx + size_t(nreal) * ncons;
      const long nrows = nrows_of(nb);
      unsigned ne = unsigned(nrows) * unsigned(n);
      hipLaunchKernelGGL(k_batch_box_rows<T>, dim3((ne + 255) / 256), dim3(256), 0, st, (T *)B.rows.p, unsigned(nrows),
                         wl, n, g.dx, g.ox, g.oy, g.oz, g.periodic, rc, wx, wy, (uint32_t *)B.cnt.p);
      GIC_HIP(hipGetLastError());
      fft_r2c_boxes<T>((const T *)B.rows.p, n, nrows, nc, wl, wx, wy, (T *)B.zbuf.p, (T *)B.ybuf.p, cv, fs,
                       (const T *)L.sqrtp_dm.p, st, hook);
    } else {
      hipLaunchKernelGGL(k_batch_tophat<T>, dim3(unsigned((fs_reals + 255) / 256), nc), dim3(256), 0, st, cv, fs_reals,
                         n, g.dx, g.ox, g.oy, g.oz, g.periodic, rc, (uint32_t *)B.cnt.p);
      GIC_HIP(hipGetLastError());
      fft_r2c_batch<T>(cv, n, nc, (const T *)L.sqrtp_dm.p, st, hook);
    }
    // Gram matrices and current values, FP64 solves, update with the transfer function
    auto gram = ncons <= 16 ? k_batch_gram<T, 1> : k_batch_gram<T, 2>;
    hipLaunchKernelGGL(gram, dim3(GRAM_BLOCKS, nb), dim3(GRAM_THREADS), 0, st, reinterpret_cast<const cx<T> *>(cv), fs,
                       reinterpret_cast<const cx<T> *>(w), ncons, n, (double *)B.part.p);
    GIC_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_batch_reduce, dim3(np, nb), dim3(256), 0, st, (const double *)B.part.p, GRAM_BLOCKS, np,
                       (double *)B.sums.p);
    GIC_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_batch_solve, dim3(nb), dim3(64), 0, st, (const double *)B.sums.p, (const uint32_t *)B.cnt.p,
                       rc, ncons, np, (double *)B.coef.p, dflags + r0);
    GIC_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_batch_update<T>, dim3(unsigned((fs + 255) / 256), nb), dim3(256), 0, st,
                       reinterpret_cast<cx<T> *>(w), reinterpret_cast<const cx<T> *>(cv), fs, ncons,
                       (const double *)B.coef.p, (const T *)L.sqrtp.p, n);
    GIC_HIP(hipGetLastError());
    // delta and the Zel'dovich displacements, dense, into the caller's arrays
    T *X = cv;   // per realisation: of delta, delta/k^2 and i k_x delta/k^2, and one more
    FftX<T> x;
    x.in = w;
    x.in_bs = fs_reals;
    for (int i = 0; i < 3; ++i) x.out[i] = X + i * fs_reals;
    x.out_bs = 4 * fs_reals;
    x.nb = nb;
    x.inv_k2 = 1.0;
    x.kmin = g.kmin();
    fft_x<T>(x, n, st, hook);
    FftY<T> y;
    y.nb = nb;
    y.in_bs = y.out_bs = 4 * fs_reals;
    y.kmin = g.kmin();
    y.add(X, X, FFT_YZ_ONE);
    y.add(X + 2 * fs_reals, X + 2 * fs_reals, FFT_YZ_ONE);
    y.add(X + fs_reals, X + fs_reals, FFT_YZ_IKY, X + 3 * fs_reals, FFT_YZ_ONE);
    fft_y<T>(y, n, st, hook);
    FftZ<T> z;
    z.nb = nb;
    z.in_bs = 4 * fs_reals;
    z.dense_bs = long(4 * n3);
    z.kmin = g.kmin();
    z.add(X, nullptr, o, FFT_YZ_ONE);
    z.add(X + 2 * fs_reals, nullptr, o + n3, FFT_YZ_ONE);
    z.add(X + fs_reals, nullptr, o + 2 * n3, FFT_YZ_ONE);
    z.add(X + 3 * fs_reals, nullptr, o + 3 * n3, FFT_YZ_IKZ);
    fft_z<T>(z, n, st, hook);
  }
  if (ms) GIC_HIP(hipEventRecord(t1, c->st));
  std::vector<uint32_t> fl(nreal);
  GIC_HIP(hipMemcpyAsync(fl.data(), B.flags.p, size_t(nreal) * sizeof(uint32_t), hipMemcpyDeviceToHost, c->st));
  GIC_HIP(hipStreamSynchronize(c->st));
  if (ms) {
    float e = 0;
    GIC_HIP(hipEventElapsedTime(&e, t0, t1));
    *ms = e;
    (void)hipEventDestroy(t0);
    (void)hipEventDestroy(t1);
  }
  for (int r = 0; r < nreal; ++r) {
    if (fl[r] & 1u) throw std::runtime_error("internal error: RNG plan produced too few Gaussians");
    if (fl[r] & 2u)
      throw std::runtime_error("batch realisation " + std::to_string(r) + ": a constraint selects no cells");
    if (fl[r] & 4u)
      throw std::runtime_error("batch realisation " + std::to_string(r) +
                               ": Modifications are not linearly independent");
  }
}

template void do_batch<float>(gic_context *, int, const uint64_t *, int, const double *, float *, int, double *);
template void do_batch<double>(gic_context *, int, const uint64_t *, int, const double *, double *, int, double *);

}  // namespace gic
