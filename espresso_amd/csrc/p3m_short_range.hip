// Device real-space pair forces of P3M Coulomb over cell lists; see
// p3m_short_range.hpp.
#include "p3m_short_range.hpp"
#include "p3m_batch.hpp"
#include "p3m_kernels.hpp"

#include <algorithm>
#include <cmath>
#include <numbers>
#include <stdexcept>
#include <vector>

namespace espresso_amd {
namespace {
using namespace dev;

constexpr int kSRMaxCells = 64; // cells per dimension at most (z bins of columns: 4 x)
constexpr int kColWaves = 4;    // waves per block of k_sr_columns
constexpr int kSortedSlack = 8; // particles k_sr_columns may read past the sorted ones
constexpr int kColBatch = 4;    // candidates tested before the lists are looked at
constexpr int kColRuns = 75;    // runs of candidates of a home group: 25 columns, 3 box images

/** Cell grid: nc cells per dimension of edge L / nc >= r_cut / nsub. */
struct CellGrid {
  int nc[3];
  double L[3];
  double inv_cell[3]; // nc / L
};

/** x folded into [0, L). */
__device__ __forceinline__ double fold(double x, double L) {
  double xf = x - L * floor(x / L);
  if (xf >= L) xf -= L;
  return xf < 0. ? 0. : xf;
}

__global__ void k_sr_fill(int *p, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
}

/** Cell of every charged particle (uncharged ones take no part in pair
 *  terms, p3m.hpp:150) and its rank in the cell. */
__global__ __launch_bounds__(256) void k_sr_bin(int64_t n, double const *__restrict__ pos,
                                                double const *__restrict__ q, CellGrid g,
                                                int *counts, int *p_cell, int *p_rank) {
  int64_t const i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (q[i] == 0.) {
    p_cell[i] = -1;
    return;
  }
  int c[3];
#pragma unroll
  for (int d = 0; d < 3; ++d)
    c[d] = min(g.nc[d] - 1, static_cast<int>(fold(pos[3 * i + d], g.L[d]) * g.inv_cell[d]));
  int const cell = (c[0] * g.nc[1] + c[1]) * g.nc[2] + c[2];
  p_cell[i] = cell;
  p_rank[i] = atomicAdd(&counts[cell], 1);
}

/** Exclusive scan of one value per thread of a 1024-thread block, and the sum
 *  of all. */
__device__ __forceinline__ int block_scan_1024(int v, int *wsum, int &total) {
  int const lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int s = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    int const t = __shfl_up(s, off, 64);
    if (lane >= off) s += t;
  }
  if (lane == 63) wsum[wid] = s;
  __syncthreads();
  int before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    int const t = wsum[w];
    before += (w < wid) ? t : 0;
    all += t;
  }
  __syncthreads(); // wsum may be written again
  total = all;
  return before + s - v;
}

/** Exclusive scan of the cell counts (one block, four cells per thread and
 *  pass); offsets[ncells] = total.  With goff, the cells are the z bins of
 *  columns of nz bins: goff[c] = 64-particle home groups in the columns
 *  before c (a group never crosses a column), goff[ncol] = all of them. */
__global__ __launch_bounds__(1024) void k_sr_scan(int const *counts, int ncells, int *offsets,
                                                  int nz, int *goff, int *arrived) {
  __shared__ int wsum[16];
  int carry = 0;
  for (int base = 0; base < ncells; base += 4096) {
    int const i = base + 4 * static_cast<int>(threadIdx.x);
    int4 c = {0, 0, 0, 0};
    if (i + 3 < ncells) {
      c = *reinterpret_cast<int4 const *>(counts + i);
    } else {
      if (i < ncells) c.x = counts[i];
      if (i + 1 < ncells) c.y = counts[i + 1];
      if (i + 2 < ncells) c.z = counts[i + 2];
    }
    int total;
    int4 o;
    o.x = carry + block_scan_1024(c.x + c.y + c.z + c.w, wsum, total);
    o.y = o.x + c.x;
    o.z = o.y + c.y;
    o.w = o.z + c.z;
    if (i + 3 < ncells) {
      *reinterpret_cast<int4 *>(offsets + i) = o;
    } else {
      if (i < ncells) offsets[i] = o.x;
      if (i + 1 < ncells) offsets[i + 1] = o.y;
      if (i + 2 < ncells) offsets[i + 2] = o.z;
    }
    carry += total;
  }
  if (threadIdx.x == 0) offsets[ncells] = carry;
  if (!goff) return;
  __syncthreads(); // offsets written by this block
  int const ncol = ncells / nz;
  int gcarry = 0;
  for (int base = 0; base < ncol; base += 1024) {
    int const c = base + static_cast<int>(threadIdx.x);
    int const cnt = (c < ncol) ? offsets[(c + 1) * nz] - offsets[c * nz] : 0;
    int total;
    int const before = block_scan_1024((cnt + 63) >> 6, wsum, total);
    if (c < ncol) goff[c] = gcarry + before;
    gcarry += total;
  }
  for (int i = threadIdx.x; i < gcarry; i += 1024) arrived[i] = 0; // blocks done per group
  if (threadIdx.x == 0) goff[ncol] = gcarry;
}

/** Charged particles in cell order: folded position and charge, and the
 *  original index.  With grp, the first particle of every 64-particle home
 *  group of a column writes the group's (column, first sorted index). */
__global__ __launch_bounds__(256) void k_sr_scatter(int64_t n, double const *__restrict__ pos,
                                                    double const *__restrict__ q, CellGrid g,
                                                    int const *p_cell, int const *p_rank,
                                                    int const *offsets, double4 *spos,
                                                    int *sidx, int nz, int const *goff,
                                                    int2 *grp) {
  int64_t const i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  int const cell = p_cell[i];
  if (cell < 0) return;
  int const slot = offsets[cell] + p_rank[i];
  spos[slot] = double4{fold(pos[3 * i], g.L[0]), fold(pos[3 * i + 1], g.L[1]),
                       fold(pos[3 * i + 2], g.L[2]), q[i]};
  sidx[slot] = static_cast<int>(i);
  if (!grp) return;
  int const col = cell / nz;
  int const r = slot - offsets[col * nz];
  if ((r & 63) == 0) grp[goff[col] + (r >> 6)] = make_int2(col, slot);
}

/** 1/x and 1/sqrt(x) in FP64: the hardware estimate (relative error e of
 *  about 2^-26) refined by one third-order step, y (1 + e + e^2) with e = 1 -
 *  x y, and y (1 + e/2 + 3 e^2/8) with e = 1 - x y^2. */
__device__ __forceinline__ double nr_rcp(double x) {
  double const y = __builtin_amdgcn_rcp(x);
  double const e = fma(-x, y, 1.);
  return fma(y, fma(e, e, e), y);
}
__device__ __forceinline__ double nr_rsq(double x) {
  double const y = __builtin_amdgcn_rsq(x);
  double const e = fma(-x, y * y, 1.);
  return fma(y * e, fma(0.375, e, 0.5), y);
}

/** Pair term of CoulombP3M::pair_force / pair_energy (p3m.hpp:146-180) with
 *  the A&S erfc of AS_erfc_part.hpp:29-40 (the published 7.1.26 constants)
 *  for a pair already known to lie within the cutoff: d = r_i - r_j,
 *  r2 = |d|^2 > 0, qq = prefactor q_i q_j.  Adds the force on i and, with
 *  EV, the pair energy and F (x) d (upper triangle: xx xy xz yy yz zz). */
template <bool EV>
__device__ __forceinline__ void pair_term(double dx, double dy, double dz, double r2, double qq,
                                          double alpha, double two_a_sqrt_pi_i, double &fx,
                                          double &fy, double &fz, double (&ev)[7]) {
  double const rinv = nr_rsq(r2);
  double const adist = alpha * (r2 * rinv);
  double const t = nr_rcp(fma(0.3275911, adist, 1.));
  double const erfc_part =
      t * (0.254829592 +
           t * (-0.284496736 + t * (1.421413741 + t * (-1.453152027 + t * 1.061405429))));
  double const ex = exp(-adist * adist);
  double const erfc_ri = erfc_part * rinv;
  double const fac = ex * (erfc_ri + two_a_sqrt_pi_i) * (rinv * rinv) * qq;
  fx += fac * dx;
  fy += fac * dy;
  fz += fac * dz;
  if constexpr (EV) {
    ev[0] += qq * erfc_ri * ex;
    ev[1] += fac * dx * dx;
    ev[2] += fac * dx * dy;
    ev[3] += fac * dx * dz;
    ev[4] += fac * dy * dy;
    ev[5] += fac * dy * dz;
    ev[6] += fac * dz * dz;
  }
}

/** ELC image terms of dielectric contrasts (off when on == 0). */
struct SrImages {
  int on;
  double h, sl, dt, db;
};

/** Pair term of particle i with the image of itself in its layer against
 *  partner j (add_pair_force_corrections / pair_energy_correction,
 *  elc.hpp:250-296; dielectric_layers_contribution, :119-138): q_eff =
 *  delta q_i q_j, d = r_j - r_i' with r_i' = (x_i, y_i, -z_i) below the
 *  layer bound or (x_i, y_i, 2h - z_i) above it, minimum image along z.
 *  dx, dy = r_i - r_j in the plane; zj is the partner's folded z.  Force on
 *  i and, with EV, the pair energy (ev[0]). */
template <bool EV>
__device__ __forceinline__ void image_terms(SrImages const &im, double zi, double zj, double dx,
                                            double dy, double Lz, double qq, double rc2,
                                            double alpha, double two_a, double &fx, double &fy,
                                            double &fz, double (&ev)[7]) {
  auto one = [&](double delta, double dz) {
    dz -= Lz * rint(dz / Lz);
    double const r2 = dx * dx + dy * dy + dz * dz;
    if (!(r2 < rc2) || !(r2 > 0.) || delta == 0.) return;
    double ax = -dx, ay = -dy, az = dz; // d = r_j - r_i'
    double const rinv = nr_rsq(r2);
    double const adist = alpha * (r2 * rinv);
    double const t = nr_rcp(fma(0.3275911, adist, 1.));
    double const erfc_part =
        t * (0.254829592 +
             t * (-0.284496736 + t * (1.421413741 + t * (-1.453152027 + t * 1.061405429))));
    double const ex = exp(-adist * adist);
    double const erfc_ri = erfc_part * rinv;
    double const q = qq * delta;
    double const fac = ex * (erfc_ri + two_a) * (rinv * rinv) * q;
    fx += fac * ax;
    fy += fac * ay;
    fz += fac * az;
    if constexpr (EV) ev[0] += q * erfc_ri * ex;
  };
  if (zi < im.sl) one(im.db, zj + zi);
  if (zi > im.h - im.sl) one(im.dt, zj - (2. * im.h - zi));
}

/** Displacement r_i - r_j, with the minimum image when MI. */
template <bool MI>
__device__ __forceinline__ void displacement(double4 const &pi, double4 const &pj,
                                             CellGrid const &g, double &dx, double &dy,
                                             double &dz) {
  dx = pi.x - pj.x;
  dy = pi.y - pj.y;
  dz = pi.z - pj.z;
  if constexpr (MI) {
    dx -= g.L[0] * rint(dx / g.L[0]);
    dy -= g.L[1] * rint(dy / g.L[1]);
    dz -= g.L[2] * rint(dz / g.L[2]);
  }
}

/** The staged candidates tile[0, cnt) against this thread's particle, in
 *  groups of 64: a cheap pass marks the partners within the cutoff in a
 *  64-bit mask, then each lane evaluates only its own marked pairs (the
 *  expensive pair term runs with the lanes that have work, instead of on
 *  every candidate that any lane of the wave needs). */
template <bool MI, bool EV>
__device__ __forceinline__ void tile_pairs(double4 const *tile, int cnt, double4 const &pi,
                                           double qpi, CellGrid const &g, double rc2,
                                           double alpha, double two_a, double &fx, double &fy,
                                           double &fz, double (&ev)[7], SrImages const &im,
                                           double sz) {
  for (int kb = 0; kb < cnt; kb += 64) {
    int const kn = min(64, cnt - kb);
    unsigned long long mask = 0;
    for (int k = 0; k < kn; ++k) {
      double dx, dy, dz;
      displacement<MI>(pi, tile[kb + k], g, dx, dy, dz);
      double const r2 = dx * dx + dy * dy + dz * dz;
      if (r2 < rc2 && r2 > 0.) mask |= 1ull << k;
    }
    while (mask) {
      int const k = __builtin_ctzll(mask);
      mask &= mask - 1;
      double4 const pj = tile[kb + k];
      double dx, dy, dz;
      displacement<MI>(pi, pj, g, dx, dy, dz);
      double const r2 = dx * dx + dy * dy + dz * dz;
      pair_term<EV>(dx, dy, dz, r2, qpi * pj.w, alpha, two_a, fx, fy, fz, ev);
      if (!MI || im.on) // cells are searched with images only
        image_terms<EV>(im, pi.z, pj.z - sz, dx, dy, g.L[2], qpi * pj.w, rc2, alpha, two_a, fx,
                        fy, fz, ev);
    }
  }
}

/** One block of NT threads per cell: the cell's particles (NT at a time)
 *  against the (2 NSUB + 1)^3 neighbour cells, each staged through LDS with
 *  its periodic shift (nc >= 2 NSUB + 1 per dimension: every neighbour is a
 *  distinct cell).  Each thread sums its particle's force over all partners
 *  (both orders of a pair are evaluated), so no atomics are needed. */
template <int NSUB, int NT, bool EV>
__global__ __launch_bounds__(NT) void k_sr_cells(CellGrid g, int const *__restrict__ offsets,
                                                 double4 const *__restrict__ spos,
                                                 int const *__restrict__ sidx, double prefactor,
                                                 double alpha, double rc2,
                                                 double *__restrict__ force, double *partials,
                                                 SrImages im) {
  __shared__ double4 tile[NT];
  __shared__ double red[8 * 16];
  constexpr int W = 2 * NSUB + 1;
  int const cell = blockIdx.x;
  int const cz = cell % g.nc[2], cy = (cell / g.nc[2]) % g.nc[1], cx = cell / (g.nc[2] * g.nc[1]);
  int const beg = offsets[cell], end = offsets[cell + 1];
  double const two_a = 2. * alpha * std::numbers::inv_sqrtpi;
  double ev[7] = {0., 0., 0., 0., 0., 0., 0.};
  for (int hb = beg; hb < end; hb += NT) {
    int const i = hb + static_cast<int>(threadIdx.x);
    bool const has = i < end;
    double4 const pi = has ? spos[i] : double4{0., 0., 0., 0.};
    double const qpi = prefactor * pi.w;
    double fx = 0., fy = 0., fz = 0.;
    for (int o = 0; o < W * W * W; ++o) {
      int nx = cx + o / (W * W) - NSUB, ny = cy + (o / W) % W - NSUB, nz = cz + o % W - NSUB;
      double sx = 0., sy = 0., sz = 0.;
      if (nx < 0) { nx += g.nc[0]; sx = -g.L[0]; } else if (nx >= g.nc[0]) { nx -= g.nc[0]; sx = g.L[0]; }
      if (ny < 0) { ny += g.nc[1]; sy = -g.L[1]; } else if (ny >= g.nc[1]) { ny -= g.nc[1]; sy = g.L[1]; }
      if (nz < 0) { nz += g.nc[2]; sz = -g.L[2]; } else if (nz >= g.nc[2]) { nz -= g.nc[2]; sz = g.L[2]; }
      int const nb = (nx * g.nc[1] + ny) * g.nc[2] + nz;
      int const jb = offsets[nb], je = offsets[nb + 1];
      for (int tb = jb; tb < je; tb += NT) {
        __syncthreads(); // the previous tile is consumed
        int const j = tb + static_cast<int>(threadIdx.x);
        if (j < je) {
          double4 const pj = spos[j];
          tile[threadIdx.x] = double4{pj.x + sx, pj.y + sy, pj.z + sz, pj.w};
        }
        __syncthreads();
        if (has)
          tile_pairs<false, EV>(tile, min(NT, je - tb), pi, qpi, g, rc2, alpha, two_a, fx, fy,
                                fz, ev, im, sz);
      }
    }
    if (has) {
      double *f = force + 3 * static_cast<int64_t>(sidx[i]);
      f[0] += fx;
      f[1] += fy;
      f[2] += fz;
    }
  }
  if constexpr (EV) {
    block_sum<7>(ev, red);
    if (threadIdx.x == 0)
      for (int k = 0; k < 7; ++k) partials[blockIdx.x * 8 + k] = ev[k];
  }
}

/** All charged pairs with the minimum-image displacement (boxes narrower
 *  than three cells of edge r_cut); one block per NT sorted particles. */
template <int NT, bool EV>
__global__ __launch_bounds__(NT) void k_sr_allpairs(int nq, CellGrid g,
                                                    double4 const *__restrict__ spos,
                                                    int const *__restrict__ sidx,
                                                    double prefactor, double alpha, double rc2,
                                                    double *__restrict__ force,
                                                    double *partials, SrImages im) {
  __shared__ double4 tile[NT];
  __shared__ double red[8 * 16];
  int const i = blockIdx.x * NT + static_cast<int>(threadIdx.x);
  bool const has = i < nq;
  double4 const pi = has ? spos[i] : double4{0., 0., 0., 0.};
  double const qpi = prefactor * pi.w;
  double const two_a = 2. * alpha * std::numbers::inv_sqrtpi;
  double fx = 0., fy = 0., fz = 0.;
  double ev[7] = {0., 0., 0., 0., 0., 0., 0.};
  for (int tb = 0; tb < nq; tb += NT) {
    __syncthreads();
    int const j = tb + static_cast<int>(threadIdx.x);
    if (j < nq) tile[threadIdx.x] = spos[j];
    __syncthreads();
    if (has)
      tile_pairs<true, EV>(tile, min(NT, nq - tb), pi, qpi, g, rc2, alpha, two_a, fx, fy, fz,
                           ev, im, 0.);
  }
  if (has) {
    double *f = force + 3 * static_cast<int64_t>(sidx[i]);
    f[0] += fx;
    f[1] += fy;
    f[2] += fz;
  }
  if constexpr (EV) {
    block_sum<7>(ev, red);
    if (threadIdx.x == 0)
      for (int k = 0; k < 7; ++k) partials[blockIdx.x * 8 + k] = ev[k];
  }
}

/** |mu|^2 of every particle (the dipolar binning key: zero dipoles take no
 *  part, dp3m.hpp:162); the cell counters are cleared on the way. */
__global__ __launch_bounds__(256) void k_sr_mu2(int64_t n, double const *__restrict__ dip,
                                                double *__restrict__ mu2,
                                                int *__restrict__ counts, int ncells) {
  int64_t const i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  for (int64_t c = i; c < ncells; c += (int64_t)gridDim.x * blockDim.x) counts[c] = 0;
  if (i >= n) return;
  double const a = dip[3 * i], b = dip[3 * i + 1], c = dip[3 * i + 2];
  mu2[i] = a * a + b * b + c * c;
}

/** Dipoles in cell order. */
__global__ __launch_bounds__(256) void k_sr_sort_dip(int64_t n, int const *__restrict__ total,
                                                     int const *__restrict__ sidx,
                                                     double const *__restrict__ dip,
                                                     double4 *__restrict__ sdip) {
  int64_t const s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (s >= n || s >= *total) return;
  int64_t const i = sidx[s];
  sdip[s] = double4{dip[3 * i], dip[3 * i + 1], dip[3 * i + 2], 0.};
}

/** Dipolar pair term (DipolarP3M::pair_force / pair_energy,
 *  dp3m.hpp:160-235) of dipole mi with partner mj at d = r_i - r_j, r2 =
 *  |d|^2, without the prefactor and with mi taken out of the sums over
 *  partners: the force is v[0..2] + mi v[6], the torque mi x v[3..5]; pair
 *  energy e with EV.  EXACT takes the library's erfc, else the rational
 *  approximation of Abramowitz and Stegun 7.1.26. */
template <bool EV, bool EXACT>
__device__ __forceinline__ void dip_pair(double dx, double dy, double dz, double r2,
                                         double4 const &mi, double4 const &mj, double alpha,
                                         double two_a, double (&v)[7], double &e) {
  double const rinv = nr_rsq(r2);
  double const ad = alpha * (r2 * rinv);
  double const ex = exp(-ad * ad);
  double const r2i = rinv * rinv;
  double B;
  if constexpr (EXACT) {
    B = (erfc(ad) * rinv + two_a * ex) * r2i;
  } else {
    double const tt = nr_rcp(fma(0.3275911, ad, 1.));
    double const ep =
        tt * (0.254829592 +
              tt * (-0.284496736 + tt * (1.421413741 + tt * (-1.453152027 + tt * 1.061405429))));
    B = (ep * rinv + two_a) * ex * r2i;
  }
  double const alpsq = alpha * alpha;
  double const common = alpsq * two_a * ex;
  double const Cr = r2i * (3. * B + 2. * common);
  double const Dr = r2i * (5. * Cr + 4. * common * alpsq);
  double const mimj = mi.x * mj.x + mi.y * mj.y + mi.z * mj.z;
  double const mir = mi.x * dx + mi.y * dy + mi.z * dz;
  double const mjr = mj.x * dx + mj.y * dy + mj.z * dz;
  double const cd = mimj * Cr - mir * mjr * Dr, cj = mir * Cr, c1 = mjr * Cr;
  v[0] += cd * dx + cj * mj.x;
  v[1] += cd * dy + cj * mj.y;
  v[2] += cd * dz + cj * mj.z;
  v[3] += c1 * dx - B * mj.x;
  v[4] += c1 * dy - B * mj.y;
  v[5] += c1 * dz - B * mj.z;
  v[6] += c1;
  if constexpr (EV) e += mimj * B - mir * c1;
}

/** Pair terms over columns: Coulomb without ELC images, or dipolar (DIP, sdip
 *  the sorted dipoles).  The cells are columns of edge >= r_cut / rx (x) and
 *  r_cut / ry (y), cut into z bins of edge >= r_cut / rz, z fastest, so that
 *  the candidates of a column within reach of a home group are one contiguous
 *  run of the sorted particles (split at the periodic boundary).  One block of W waves per home group of 64 sorted
 *  particles of one column: lane = home particle, position and force in
 *  registers; the waves share the runs of the (2 rx + 1)(2 ry + 1) columns,
 *  kColBatch candidates at a time, and their forces are added through LDS at the end.
 *
 *  What bounds it: FP64 VALU issue, first of the distance tests, then of the
 *  pair terms.  A candidate is the same for all lanes, so its position comes
 *  through the scalar cache and enters the test as a scalar operand; the test
 *  appends the candidate's index to the lane's own list without a branch (a
 *  miss is overwritten by the next candidate), and the pair terms run when a
 *  list is nearly full, with most lanes busy (85 % of them; 42 % when every
 *  list is emptied each time and the columns are swept once, in order).
 *  Measured (250,000 charges, 311 partners each): 0.57 ms, 73 % VALU issue,
 *  against 2.94 ms with lanes over the home particles of one r_cut/2 cell,
 *  which kept 10 of 64 lanes busy; 1000 charges: 27 against 89 us.  50,000
 *  dipoles, 66 partners each: 77 us, against 144 with lanes over the home
 *  particles of one r_cut cell and a queue of hits per block; 200,000 dipoles
 *  with 100, 420 and 4300 partners (calls): 0.36, 0.86 and 6.8 ms against 0.71,
 *  1.9 and 20.  Few sparse dipoles are latency: 300 16 against 11 us, 8000 of 33
 *  partners 26 against 23. */
template <bool DIP, bool EV, bool EXACT>
__global__ __launch_bounds__(kColWaves * 64, DIP ? 3 : EV ? 4 : 5) void k_sr_columns(
    CellGrid g, int rx, int ry, int rz, int split, int sweeps, int const *__restrict__ offsets,
    int const *__restrict__ goff, int2 const *__restrict__ grp,
    double4 const *__restrict__ spos, double4 const *__restrict__ sdip,
    int const *__restrict__ sidx, double prefactor, double alpha, double rc2,
    double *__restrict__ force, double *__restrict__ torque, double *__restrict__ shares,
    int *__restrict__ arrived, double *__restrict__ partials) {
  constexpr int W = kColWaves, U = kColBatch, CAP = 24; // CAP: list length
  constexpr int NV = DIP ? 6 : 3, NE = DIP ? 1 : 7; // force (and torque); reduced terms
  static_assert(CAP >= 2 * U && CAP * 64 * sizeof(int) >= NV * 64 * sizeof(double));
  __shared__ __align__(16) int list[W][CAP * 64];
  __shared__ double red[8 * 16];
  __shared__ int last;
  __shared__ int4 runs[kColRuns];
  __shared__ int nruns;
  int const ngroups = goff[g.nc[0] * g.nc[1]];
  int const b = blockIdx.x, nblocks = ngroups * split;
  if (b >= nblocks) {
    if (EV && threadIdx.x < NE) partials[static_cast<int64_t>(b) * 8 + threadIdx.x] = 0.;
    return;
  }
  // contiguous groups per XCD (their candidates overlap)
  int const xq = nblocks >> 3, xr = nblocks & 7;
  int const bi = (b & 7) * xq + min(b & 7, xr) + (b >> 3);
  int const gi = bi / split, share = bi - gi * split;
  int const col = __builtin_amdgcn_readfirstlane(grp[gi].x);
  int const h0 = __builtin_amdgcn_readfirstlane(grp[gi].y);
  int const nz = g.nc[2];
  int const nh = min(64, offsets[(col + 1) * nz] - h0);
  int const cx = col / g.nc[1], cy = col - cx * g.nc[1];
  int const lane = static_cast<int>(threadIdx.x & 63);
  int const wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  int const me = share * W + wave, all = split * W; // of the group's waves (a power of two)
  bool const home = lane < nh;
  double4 hp = spos[h0 + min(lane, nh - 1)];
  int64_t const row = 3 * static_cast<int64_t>(sidx[h0 + min(lane, nh - 1)]);
  double const qpi = prefactor * hp.w;
  double4 hm{0., 0., 0., 0.};
  if constexpr (DIP) hm = sdip[h0 + min(lane, nh - 1)];
  // z bins of the group (sorted by bin): first and last particle
  auto zbin = [&](double z) { return min(nz - 1, static_cast<int>(z * g.inv_cell[2])); };
  int const b0 = zbin(readlane_f64(hp.z, 0)), b1 = zbin(readlane_f64(hp.z, nh - 1));
  if (!home) hp.x = 1e300; // beyond every cutoff
  bool const wrap = cx < rx || cx + rx >= g.nc[0] || cy < ry || cy + ry >= g.nc[1] ||
                    b0 < rz || b1 + rz >= nz;
  double const two_a = 2. * alpha * std::numbers::inv_sqrtpi;
  double f[DIP ? 7 : 3] = {}; // sums of pair_term or dip_pair
  double ev[NE] = {};
  // byte offsets into `list` of the lane's first slot, of the slot the next
  // hit goes to, and of the last one a batch may start at
  char *const lists = reinterpret_cast<char *>(list);
  int const slot0 = (wave * CAP * 64 + lane) * 4, full = slot0 + (CAP - U) * 256;
  int slot = slot0;
  double const iLx = 1. / g.L[0], iLy = 1. / g.L[1], iLz = 1. / g.L[2];

  // pair terms of the listed candidates, one per lane and round: until too
  // few lanes have one left (but at least U rounds, so that the next batch
  // fits), or all of them at the end; what is left moves to the front
  auto listed = [&](int s) { return *reinterpret_cast<int const *>(lists + s); };
  auto drain = [&](bool rest) {
    int s = slot0;
    int j = (s < slot) ? listed(s) : h0;
    double4 next = spos[j], next_dip{0., 0., 0., 0.};
    if constexpr (DIP) next_dip = sdip[j];
    for (int round = 0;; ++round) {
      uint64_t const busy = __ballot(s < slot);
      if (!busy || (!rest && round >= U && __popcll(busy) < 40)) break;
      double4 const pj = next, mj = next_dip;
      bool const on = s < slot;
      s += 256;
      if (s < slot) { // in flight during this round
        j = listed(s);
        next = spos[j];
        if constexpr (DIP) next_dip = sdip[j];
      }
      if (on) {
        double dx = hp.x - pj.x, dy = hp.y - pj.y, dz = hp.z - pj.z;
        if (wrap) {
          dx -= g.L[0] * rint(dx * iLx);
          dy -= g.L[1] * rint(dy * iLy);
          dz -= g.L[2] * rint(dz * iLz);
        }
        double const r2 = dx * dx + dy * dy + dz * dz;
        if (r2 > 0.) {
          if constexpr (DIP) {
            dip_pair<EV, EXACT>(dx, dy, dz, r2, hm, mj, alpha, two_a, f, ev[0]);
          } else {
            pair_term<EV>(dx, dy, dz, r2, qpi * pj.w, alpha, two_a, f[0], f[1], f[2], ev);
          }
        }
      }
    }
    int d = slot0;
    if (!rest)
      while (__any(s < slot)) {
        if (s < slot) {
          *reinterpret_cast<int *>(lists + d) = listed(s);
          d += 256;
        }
        s += 256;
      }
    slot = d;
  };
  // the next candidate: listed if within the limit, else overwritten
  auto test = [&](double hx, double hy, double hz, double4 const &cj, int j, double lim) {
    double const dx = hx - cj.x, dy = hy - cj.y, dz = hz - cj.z;
    double const r2 = dx * dx + dy * dy + dz * dz;
    *reinterpret_cast<int *>(lists + slot) = j;
    slot += (r2 < lim) ? 256 : 0;
  };

  // Runs of candidates: first and end particle of every column and box image
  // along z in reach, and the image.  One lane of the first wave looks up one
  // of them and the empty ones are dropped: with the look-ups in the loop they
  // are a chain of loads (100 dipoles 17.1 us, so 14.6; 50,000 77.6 and 73.0)
  int const ncy = 2 * ry + 1, ncols = (2 * rx + 1) * ncy;
  if (wave == 0) {
    int n = 0;
    for (int r0 = 0; r0 < 3 * ncols; r0 += 64) {
      int const r = r0 + lane, q = r / 3, k = r - 3 * q - 1;
      int const c = (4 * q) % ncols; // 9, 15 or 25 columns: all of them once
      int nx = cx + c / ncy - rx, ny = cy + c % ncy - ry, ix = 0, iy = 0;
      if (nx < 0) { nx += g.nc[0]; ix = -1; } else if (nx >= g.nc[0]) { nx -= g.nc[0]; ix = 1; }
      if (ny < 0) { ny += g.nc[1]; iy = -1; } else if (ny >= g.nc[1]) { ny -= g.nc[1]; iy = 1; }
      int const *const off = offsets + (nx * g.nc[1] + ny) * nz;
      int const lo = max(b0 - rz - k * nz, 0), hi = min(b1 + rz - k * nz, nz - 1);
      int jb = 0, je = 0;
      if (r < 3 * ncols && lo <= hi) {
        jb = off[lo];
        je = off[hi + 1];
      }
      uint64_t const some = __ballot(jb < je);
      if (jb < je)
        runs[n + __popcll(some & ((1ull << lane) - 1ull))] =
            int4{jb, je, ix + 1 + 4 * (iy + 1), k};
      n += __popcll(some);
    }
    if (lane == 0) nruns = n;
  }
  __syncthreads();

  // `sweeps` passes over all runs, each over every sweeps-th batch of a run,
  // the columns out of order: lanes at different corners of the group then fill
  // their lists at about the same rate
  int const nr = __builtin_amdgcn_readfirstlane(nruns);
  int turn = 0; // batches so far: batch t goes to wave t % all
  for (int sweep = 0; sweep < sweeps; ++sweep) {
    for (int r = 0; r < nr; ++r) {
      int4 const run = runs[r];
      int const jb = __builtin_amdgcn_readfirstlane(run.x) + sweep * U;
      int const je = __builtin_amdgcn_readfirstlane(run.y);
      int const xy = __builtin_amdgcn_readfirstlane(run.z);
      int const nb = max(0, (je - jb + sweeps * U - 1) / (sweeps * U));
      double const hx = hp.x - ((xy & 3) - 1) * g.L[0], hy = hp.y - ((xy >> 2) - 1) * g.L[1],
                   hz = hp.z - __builtin_amdgcn_readfirstlane(run.w) * g.L[2];
      for (int t = (me - turn) & (all - 1); t < nb; t += all) {
        int const j0 = jb + t * (sweeps * U);
        // the last batch of a run reads past it, never past the allocation
        // (kSortedSlack), and lists nothing from there
        double4 const *const cj = spos + j0;
        if (j0 + U <= je) {
#pragma unroll
          for (int u = 0; u < U; ++u) test(hx, hy, hz, cj[u], j0 + u, rc2);
        } else {
#pragma unroll
          for (int u = 0; u < U; ++u)
            test(hx, hy, hz, cj[u], j0 + u, (j0 + u < je) ? rc2 : -1.);
        }
        if (__any(slot > full)) drain(false);
      }
      turn += nb;
    }
  }
  drain(true);
  if constexpr (DIP) {
    double const h[3] = {f[3], f[4], f[5]};
    f[0] = prefactor * (f[0] + hm.x * f[6]);
    f[1] = prefactor * (f[1] + hm.y * f[6]);
    f[2] = prefactor * (f[2] + hm.z * f[6]);
    f[3] = prefactor * (hm.y * h[2] - hm.z * h[1]);
    f[4] = prefactor * (hm.z * h[0] - hm.x * h[2]);
    f[5] = prefactor * (hm.x * h[1] - hm.y * h[0]);
    ev[0] *= prefactor;
  }
  // the caller's rows, in flight while the sums are added (nobody else writes
  // them before this group's last block does)
  double was[NV] = {};
  if (wave == 0 && home) {
    if (!DIP || force) {
#pragma unroll
      for (int k = 0; k < 3; ++k) was[k] = force[row + k];
    }
    if constexpr (DIP) {
      if (torque) {
#pragma unroll
        for (int k = 0; k < 3; ++k) was[3 + k] = torque[row + k];
      }
    }
  }
  // the waves' sums, in wave order
  double *const own = reinterpret_cast<double *>(list[wave]);
#pragma unroll
  for (int k = 0; k < NV; ++k) own[64 * k + lane] = f[k];
  __syncthreads();
  if (wave == 0) {
#pragma unroll
    for (int v = 1; v < W; ++v) {
      double const *o = reinterpret_cast<double const *>(list[v]);
#pragma unroll
      for (int k = 0; k < NV; ++k) f[k] += o[64 * k + lane];
    }
  }
  bool add = wave == 0 && home;
  if (split > 1) {
    // the group's last block adds all shares, in share order
    double *const mine = shares + static_cast<int64_t>(gi) * split * (64 * NV);
    if (wave == 0) {
      double *const o = mine + share * (64 * NV);
#pragma unroll
      for (int k = 0; k < NV; ++k)
        __hip_atomic_store(o + 64 * k + lane, f[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      // the shares are written and read past the caches of the XCDs (agent
      // scope), so the count only has to wait for the stores to complete
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (lane == 0)
        last = __hip_atomic_fetch_add(arrived + gi, 1, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT) == split - 1;
    }
    __syncthreads();
    add = add && last;
    if (add) {
#pragma unroll
      for (int k = 0; k < NV; ++k) f[k] = 0.;
      for (int v = 0; v < split; ++v) {
        double *const o = mine + v * (64 * NV);
#pragma unroll
        for (int k = 0; k < NV; ++k)
          f[k] += __hip_atomic_load(o + 64 * k + lane, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  if (add) {
    if (!DIP || force) {
#pragma unroll
      for (int k = 0; k < 3; ++k) force[row + k] = was[k] + f[k];
    }
    if constexpr (DIP) {
      if (torque) {
#pragma unroll
        for (int k = 0; k < 3; ++k) torque[row + k] = was[3 + k] + f[3 + k];
      }
    }
  }
  if constexpr (EV) {
    block_sum<NE>(ev, red);
    if (threadIdx.x == 0)
      for (int k = 0; k < NE; ++k) partials[static_cast<int64_t>(b) * 8 + k] = ev[k];
  }
}

/** Columns of a box for k_sr_columns: edge >= r_cut (>= r_cut/2 along an axis
 *  that does not hold three of those; wider columns make the 64-particle
 *  groups compact), z bins of r_cut/4 while those hold about eight particles,
 *  else r_cut/2. */
struct Columns {
  CellGrid g;
  int reach[3];
  int ncol, max_groups, split, sweeps;
};
Columns make_columns(ShortRangeParams const &p, int64_t n, bool exact_erfc = false) {
  Columns c;
  double const per_cut = static_cast<double>(n) * p.r_cut * p.r_cut * p.r_cut /
                         (p.box[0] * p.box[1] * p.box[2]);
  for (int d = 0; d < 2; ++d) {
    c.reach[d] = (std::floor(p.box[d] / p.r_cut) >= 3.) ? 1 : 2;
    c.g.nc[d] =
        std::min(kSRMaxCells, static_cast<int>(std::floor(p.box[d] * c.reach[d] / p.r_cut)));
  }
  c.reach[2] = (per_cut >= 32.) ? 4 : 2;
  c.g.nc[2] = std::min(4 * kSRMaxCells,
                       static_cast<int>(std::floor(p.box[2] * c.reach[2] / p.r_cut)));
  for (int d = 0; d < 3; ++d) {
    c.g.L[d] = p.box[d];
    c.g.inv_cell[d] = c.g.nc[d] / p.box[d];
  }
  c.ncol = c.g.nc[0] * c.g.nc[1];
  c.max_groups =
      static_cast<int>(std::min<int64_t>(n, n / 64 + c.ncol)); // one partial group per column
  // Few groups are shared by several blocks, each taking every split-th batch
  // of candidates: twice as many while there are fewer than 4096 blocks, four
  // rounds of what the chip holds (so fewer than 8192 in the end), as long as
  // the lists of one wave still fill: its candidates must be a twentieth of the
  // number of blocks, and two batches (a little more with the exact erfc,
  // whose registers leave three waves per SIMD instead of four: 225 groups of
  // 800 candidates 33 us in 2 blocks, 35 in 4).  Dipolar and Coulomb kernel, at that
  // split against twice and half of it: 1006 groups of 980 candidates each
  // 84 us in 2 blocks, 103 in 4, 111 in 1; 40 groups of 1900 32 us in 8, 36 in
  // 16; 321 groups of 16,700 0.62 ms in 16, 0.71 in 8.  Few candidates, dipoles:
  // 20 groups of 300 15 us in 8, 16 in 4, 20 in 2; 31 of 230 15 in 4, 17 in 2;
  // 115 of 120 14.5 in 2, 14.9 in 1.
  double const columns = (2. * c.reach[0] + 1.) * (2. * c.reach[1] + 1.);
  double const in_reach = per_cut / (c.g.nc[0] * c.g.nc[1]) * p.box[0] * p.box[1] /
                          (p.r_cut * p.r_cut); // candidates of one column per r_cut of z
  double const tests = columns * (std::min(64., static_cast<double>(n) / c.ncol) +
                                  2. * in_reach * (1. + 1. / c.reach[2]));
  double const per_block = exact_erfc ? 0.06 : 0.05;
  c.split = 1;
  while (c.split < 16 && c.max_groups * c.split < 4096 &&
         tests / (2 * c.split * kColWaves) >= std::max(2. * kColBatch, per_block * c.max_groups * 2 * c.split))
    c.split *= 2;
  // one pass over the columns per 16 candidates (four batches) that a wave
  // takes of each: with 4 against 16 passes, 200,000 dipoles of 4300 partners
  // 9.3 against 6.9 ms; 2 against 4 passes at 105 partners 0.39 against 0.44 ms
  c.sweeps = std::clamp(static_cast<int>(tests / (columns * 16. * c.split * kColWaves)), 1, 16);
  return c;
}

template <typename T> void sr_grow(T *&p, size_t &cap, size_t need, char const *what) {
  if (need <= cap) return;
  if (p) (void)hipFree(p);
  p = nullptr;
  cap = 0; // of a null pointer, should the allocation fail
  size_t const n = need + need / 4 + 64;
  hip_check(hipMalloc(&p, sizeof(T) * n), what);
  cap = n;
}
} // namespace

struct ShortRange::Impl {
  int device = 0;
  int nc[3] = {0, 0, 0};
  double *mu2 = nullptr;
  double4 *sdip = nullptr;
  size_t cap_mu2 = 0, cap_sdip = 0;
  int *counts = nullptr, *offsets = nullptr, *p_cell = nullptr, *p_rank = nullptr,
      *sidx = nullptr;
  double *shares = nullptr; // and, in the same allocation:
  int2 *grp = nullptr;
  int *goff = nullptr, *arrived = nullptr;
  size_t cap_shares = 0;
  double4 *spos = nullptr;
  double *partials = nullptr;
  size_t cap_cells = 0, cap_off = 0, cap_pc = 0, cap_pr = 0, cap_si = 0, cap_sp = 0, cap_part = 0;

  /** Buffers of the column search (nv sums per particle), one allocation. */
  void grow_columns(Columns const &c, int nv) {
    size_t const groups = static_cast<size_t>(c.max_groups), ints = c.ncol + 1 + groups;
    size_t const sums = (c.split > 1) ? groups * c.split * 64 * nv : 0;
    sr_grow(shares, cap_shares, sums + groups + (ints + 1) / 2, "hipMalloc home groups");
    grp = reinterpret_cast<int2 *>(shares + sums);
    goff = reinterpret_cast<int *>(grp + groups);
    arrived = goff + c.ncol + 1;
  }
};

ShortRange::ShortRange(int device) : m(new Impl) { m->device = device; }

ShortRange::~ShortRange() {
  (void)hipSetDevice(m->device);
  for (void *p : {static_cast<void *>(m->counts), static_cast<void *>(m->offsets),
                  static_cast<void *>(m->p_cell), static_cast<void *>(m->p_rank),
                  static_cast<void *>(m->sidx), static_cast<void *>(m->spos),
                  static_cast<void *>(m->partials), static_cast<void *>(m->mu2),
                  static_cast<void *>(m->sdip), static_cast<void *>(m->shares)})
    if (p) (void)hipFree(p);
  delete m;
}

void ShortRange::cells(int out[3]) const {
  for (int d = 0; d < 3; ++d) out[d] = m->nc[d];
}

void ShortRange::compute(hipStream_t st, ShortRangeParams const &p, int64_t n, double const *pos,
                         double const *q, double *force, ShortRangeResult *out) {
  if (out) *out = ShortRangeResult{};
  if (!(p.r_cut > 0.)) throw std::invalid_argument("P3M: short range needs r_cut > 0");
  for (int d = 0; d < 3; ++d)
    if (!(p.box[d] > 0.)) throw std::invalid_argument("P3M: short range needs a box");
  if (n > INT32_MAX) throw std::invalid_argument("P3M: too many particles for the short range");
  if (n == 0) return;
  hip_check(hipSetDevice(m->device), "hipSetDevice");
  // cells of edge >= r_cut / nsub, two per r_cut or one with subdivision 1, in
  // boxes that hold 2 nsub + 1 distinct ones along every axis; else all pairs
  // (a box too narrow for five of r_cut/2 does not hold three of r_cut either)
  if (p.subdivision < 0 || p.subdivision > 2)
    throw std::invalid_argument("P3M: short-range subdivision must be 0, 1 or 2");
  int nsub = (p.subdivision == 1) ? 1 : 2;
  int nc[3];
  for (int d = 0; d < 3; ++d)
    nc[d] = std::min(kSRMaxCells, static_cast<int>(std::floor(p.box[d] * nsub / p.r_cut)));
  if (std::min({nc[0], nc[1], nc[2]}) < 2 * nsub + 1) {
    nsub = 0;
    nc[0] = nc[1] = nc[2] = 1;
  }
  CellGrid g;
  for (int d = 0; d < 3; ++d) {
    m->nc[d] = g.nc[d] = nc[d];
    g.L[d] = p.box[d];
  }
  // without ELC images the pairs run over columns of merged cells
  bool const columns = nsub != 0 && !p.elc_images;
  Columns cols{};
  if (columns) {
    cols = make_columns(p, n);
    g = cols.g;
  }
  for (int d = 0; d < 3; ++d) g.inv_cell[d] = g.nc[d] / p.box[d];
  int const ncells = g.nc[0] * g.nc[1] * g.nc[2];
  sr_grow(m->counts, m->cap_cells, static_cast<size_t>(ncells), "hipMalloc cell counts");
  sr_grow(m->offsets, m->cap_off, static_cast<size_t>(ncells) + 1, "hipMalloc cell offsets");
  sr_grow(m->p_cell, m->cap_pc, static_cast<size_t>(n), "hipMalloc cell ids");
  sr_grow(m->p_rank, m->cap_pr, static_cast<size_t>(n), "hipMalloc cell ranks");
  sr_grow(m->sidx, m->cap_si, static_cast<size_t>(n), "hipMalloc cell order");
  sr_grow(m->spos, m->cap_sp, static_cast<size_t>(n) + kSortedSlack, "hipMalloc cell positions");
  if (columns) m->grow_columns(cols, 3);
  int const nb = static_cast<int>((n + 255) / 256);
  k_sr_fill<<<std::min((ncells + 255) / 256, 1024), 256, 0, st>>>(m->counts, ncells);
  k_sr_bin<<<nb, 256, 0, st>>>(n, pos, q, g, m->counts, m->p_cell, m->p_rank);
  k_sr_scan<<<1, 1024, 0, st>>>(m->counts, ncells, m->offsets, g.nc[2],
                                columns ? m->goff : nullptr, m->arrived);
  k_sr_scatter<<<nb, 256, 0, st>>>(n, pos, q, g, m->p_cell, m->p_rank, m->offsets, m->spos,
                                   m->sidx, g.nc[2], m->goff, columns ? m->grp : nullptr);
  double const rc2 = p.r_cut * p.r_cut;
  int blocks = columns ? cols.max_groups * cols.split : ncells;
  int nq = 0;
  if (nsub == 0) {
    // all-pairs: the number of charged particles decides the grid
    hip_check(hipMemcpyAsync(&nq, m->offsets + ncells, sizeof(int), hipMemcpyDeviceToHost, st),
              "copy charged count");
    hip_check(hipStreamSynchronize(st), "sync short range");
    blocks = std::max(1, (nq + 255) / 256);
  }
  if (out) sr_grow(m->partials, m->cap_part, static_cast<size_t>(blocks) * 8, "hipMalloc partials");
  SrImages im{p.elc_images ? 1 : 0, p.elc_h, p.elc_sl, p.elc_dt, p.elc_db};
  auto launch = [&](auto EVc) {
    constexpr bool EV = decltype(EVc)::value;
    if (columns) {
      k_sr_columns<false, EV, false><<<blocks, kColWaves * 64, 0, st>>>(
          g, cols.reach[0], cols.reach[1], cols.reach[2], cols.split, cols.sweeps,
          m->offsets, m->goff, m->grp,
          m->spos, nullptr, m->sidx, p.prefactor, p.alpha, rc2, force, nullptr, m->shares,
          m->arrived, m->partials);
    } else if (nsub == 2) {
      k_sr_cells<2, 64, EV><<<blocks, 64, 0, st>>>(g, m->offsets, m->spos, m->sidx, p.prefactor,
                                                   p.alpha, rc2, force, m->partials, im);
    } else if (nsub == 1) {
      k_sr_cells<1, 256, EV><<<blocks, 256, 0, st>>>(g, m->offsets, m->spos, m->sidx,
                                                     p.prefactor, p.alpha, rc2, force,
                                                     m->partials, im);
    } else {
      k_sr_allpairs<256, EV><<<blocks, 256, 0, st>>>(nq, g, m->spos, m->sidx, p.prefactor,
                                                     p.alpha, rc2, force, m->partials, im);
    }
  };
  if (out)
    launch(std::true_type{});
  else
    launch(std::false_type{});
  hip_check(hipGetLastError(), "short-range kernels");
  if (!out) return;
  std::vector<double> part(static_cast<size_t>(blocks) * 8);
  hip_check(hipMemcpyAsync(part.data(), m->partials, sizeof(double) * part.size(),
                           hipMemcpyDeviceToHost, st),
            "copy short-range partials");
  hip_check(hipStreamSynchronize(st), "sync short range");
  double s[7] = {0., 0., 0., 0., 0., 0., 0.};
  for (int b = 0; b < blocks; ++b)
    for (int k = 0; k < 7; ++k) s[k] += part[static_cast<size_t>(b) * 8 + k];
  // every pair was evaluated from both sides
  out->energy = 0.5 * s[0];
  double const v[3][3] = {{s[1], s[2], s[3]}, {s[2], s[4], s[5]}, {s[3], s[5], s[6]}};
  for (int a = 0; a < 3; ++a)
    for (int b = 0; b < 3; ++b) out->virial[3 * a + b] = 0.5 * v[a][b];
}

bool ShortRange::compute_dipolar(hipStream_t st, ShortRangeParams const &p, bool exact_erfc,
                                 int64_t n, double const *pos, double const *dip, double *force,
                                 double *torque, double *energy) {
  if (energy) *energy = 0.;
  if (!(p.r_cut > 0.)) throw std::invalid_argument("P3M: short range needs r_cut > 0");
  if (n > INT32_MAX) throw std::invalid_argument("P3M: too many particles for the short range");
  // three cells of r_cut along every axis, or five of r_cut/2 if allowed
  for (int d = 0; d < 3; ++d)
    if (std::floor(p.box[d] / p.r_cut) < 3. &&
        (p.subdivision == 1 || std::floor(2. * p.box[d] / p.r_cut) < 5.))
      return false;
  if (n == 0) return true;
  hip_check(hipSetDevice(m->device), "hipSetDevice");
  Columns const cols = make_columns(p, n, exact_erfc);
  CellGrid const &g = cols.g;
  int const ncells = cols.ncol * g.nc[2];
  sr_grow(m->counts, m->cap_cells, static_cast<size_t>(ncells), "hipMalloc cell counts");
  sr_grow(m->offsets, m->cap_off, static_cast<size_t>(ncells) + 1, "hipMalloc cell offsets");
  sr_grow(m->p_cell, m->cap_pc, static_cast<size_t>(n), "hipMalloc cell ids");
  sr_grow(m->p_rank, m->cap_pr, static_cast<size_t>(n), "hipMalloc cell ranks");
  sr_grow(m->sidx, m->cap_si, static_cast<size_t>(n), "hipMalloc cell order");
  sr_grow(m->spos, m->cap_sp, static_cast<size_t>(n) + kSortedSlack, "hipMalloc cell positions");
  sr_grow(m->mu2, m->cap_mu2, static_cast<size_t>(n), "hipMalloc dipole norms");
  sr_grow(m->sdip, m->cap_sdip, static_cast<size_t>(n), "hipMalloc cell dipoles");
  m->grow_columns(cols, 6);
  int const blocks = cols.max_groups * cols.split;
  if (energy) sr_grow(m->partials, m->cap_part, static_cast<size_t>(blocks) * 8, "hipMalloc partials");
  int const nb = static_cast<int>((n + 255) / 256);
  k_sr_mu2<<<nb, 256, 0, st>>>(n, dip, m->mu2, m->counts, ncells);
  k_sr_bin<<<nb, 256, 0, st>>>(n, pos, m->mu2, g, m->counts, m->p_cell, m->p_rank);
  k_sr_scan<<<1, 1024, 0, st>>>(m->counts, ncells, m->offsets, g.nc[2], m->goff, m->arrived);
  k_sr_scatter<<<nb, 256, 0, st>>>(n, pos, m->mu2, g, m->p_cell, m->p_rank, m->offsets, m->spos,
                                   m->sidx, g.nc[2], m->goff, m->grp);
  k_sr_sort_dip<<<nb, 256, 0, st>>>(n, m->offsets + ncells, m->sidx, dip, m->sdip);
  double const rc2 = p.r_cut * p.r_cut;
  auto launch = [&](auto EVc, auto EXc) {
    k_sr_columns<true, decltype(EVc)::value, decltype(EXc)::value>
        <<<blocks, kColWaves * 64, 0, st>>>(g, cols.reach[0], cols.reach[1], cols.reach[2],
                                            cols.split, cols.sweeps, m->offsets,
                                            m->goff, m->grp, m->spos, m->sdip, m->sidx,
                                            p.prefactor, p.alpha, rc2, force, torque, m->shares,
                                            m->arrived, m->partials);
  };
  if (energy && exact_erfc)
    launch(std::true_type{}, std::true_type{});
  else if (energy)
    launch(std::true_type{}, std::false_type{});
  else if (exact_erfc)
    launch(std::false_type{}, std::true_type{});
  else
    launch(std::false_type{}, std::false_type{});
  hip_check(hipGetLastError(), "dipolar short-range kernels");
  if (!energy) return true;
  std::vector<double> part(static_cast<size_t>(blocks) * 8);
  hip_check(hipMemcpyAsync(part.data(), m->partials, sizeof(double) * part.size(),
                           hipMemcpyDeviceToHost, st),
            "copy partials");
  hip_check(hipStreamSynchronize(st), "sync dipolar short range");
  double s = 0.;
  for (int b = 0; b < blocks; ++b) s += part[static_cast<size_t>(b) * 8];
  *energy = 0.5 * s;
  return true;
}

} // namespace espresso_amd
