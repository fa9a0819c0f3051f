// smac_refgmg.hip -- the reference's geometric multigrid preconditioner
// (G_GMGSolver, CFD/pressure_solver/G_GMGSolver.cu:10-998) on gfx950.
//
// Algorithm (kept as the reference, so the iterates match):
//   * level 0 is already coarse (N/2); a direction stops coarsening when its
//     halved size would drop below 6 (G_GMGSolver.h:20);
//   * coarse face coefficient = mean of the 2x2x2 fine face coefficients,
//     two fine faces along the face's own axis (k_create_level*_coeffs,
//     G_GMGSolver.cu:499-644); level operator a = beta/h^2, diag = sum,
//     inv = 0 when |diag| < 1e-12 (k_create_level_A, 646-685);
//   * weighted Jacobi, omega = 0.6, from zero (692-746);
//   * residual, mean restriction over the children (152-226, 416-493);
//   * constant prolongation-add into the children (285-389);
//   * coarse ghosts stay zero; periodic directions (absent in the reference)
//     wrap face and cell indices.
//
// MI355X form: the finest-grid kernels work on the PCG vectors in their
// row-split layout (wave per row, XCD-aware row order); the residual is fused
// into the restriction (each coarse thread forms its children's residuals in
// the reference's summation order), so no residual array is written. Level
// arrays use a natural x-fastest layout with one ghost layer and pitches
// (n+3); the level count is small and their traffic is a fraction of the fine
// level's.
#include "smac_internal.hpp"

namespace smac {

namespace {

constexpr double RG_OMEGA = 0.6;   // G_GMGSolver.cu:695
constexpr double RG_EPS = 1.E-12;  // CFD/hardCodedParameters.h:7
constexpr int RGB = 256;

__device__ __forceinline__ size_t ridx(const RgLv& L, int i, int j, int k) {
  return ((size_t)k * (size_t)L.py + (size_t)j) * (size_t)L.px + (size_t)i;
}
__device__ __forceinline__ int rwrap(int i, int n) { return i < 1 ? i + n : (i > n ? i - n : i); }

// thread -> cell (i,j,k) of a level, x fastest
__device__ __forceinline__ bool rg_cell(const RgLv& L, int& i, int& j, int& k) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t nxy = (size_t)L.n[0] * (size_t)L.n[1];
  if (t >= nxy * (size_t)L.n[2]) return false;
  k = (int)(t / nxy) + 1;
  const size_t r = t % nxy;
  j = (int)(r / (size_t)L.n[0]) + 1;
  i = (int)(r % (size_t)L.n[0]) + 1;
  return true;
}

// grid face coefficient of a uniform-density grid: beta0 on interior faces,
// 0 on boundary and ghost faces (SMACSolver.cpp:341-420)
__device__ __forceinline__ double grid_beta(const Geo& g, int d, const int f[3]) {
  int fd = f[d];
  if (g.per[d]) return g.beta0;
  if (fd <= 1 || fd >= g.n[d] + 1) return 0.0;
  return g.beta0;
}

// coarse face coefficients of axis d on level C (k_create_level0_coeffs when
// fb == nullptr, else k_create_level_coeffs from level F)
__global__ __launch_bounds__(RGB) void k_rg_beta(Geo g, BetaF gb, RgLv C, RgLv F, const double* __restrict__ fb,
                                                 int d, double* __restrict__ cb) {
  int hi[3] = {C.n[0], C.n[1], C.n[2]};
  hi[d] += 1;
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t nxy = (size_t)hi[0] * (size_t)hi[1];
  if (t >= nxy * (size_t)hi[2]) return;
  const int k = (int)(t / nxy) + 1;
  const size_t r = t % nxy;
  const int j = (int)(r / (size_t)hi[0]) + 1;
  const int i = (int)(r % (size_t)hi[0]) + 1;
  const int q[3] = {i, j, k};
  int B[3], R[3];
#pragma unroll
  for (int e = 0; e < 3; e++) {
    B[e] = C.co[e] ? 2 * q[e] - 1 : q[e];
    R[e] = C.co[e] ? 2 : 1;
  }
  double count = 0., tmp = 0.;
  for (int iz = 0; iz < R[2]; iz++)
    for (int iy = 0; iy < R[1]; iy++)
      for (int ix = 0; ix < R[0]; ix++) {
        int f[3] = {B[0] + ix, B[1] + iy, B[2] + iz};
        double v;
        if (fb == nullptr) {
          if (gb.b[0]) {  // the grid's face coefficients (two-phase grids)
            if (g.per[d]) f[d] = rwrap(f[d], g.n[d]);
            v = f[d] > g.n[d] + 1 ? 0.0 : gb.b[d][idx(g, f[0], f[1], f[2])];
          } else {
            v = grid_beta(g, d, f);
          }
        } else {
          if (F.per[d]) f[d] = rwrap(f[d], F.n[d]);
          v = f[d] > F.n[d] + 1 ? 0.0 : fb[ridx(F, f[0], f[1], f[2])];
        }
        tmp += v;
        count += 1.0;
      }
  cb[ridx(C, i, j, k)] = tmp / count;
}

struct RgCoef {
  double a[6];
  double diag, inv;
};
__device__ __forceinline__ RgCoef rg_coef(const RgLv& L, const double* __restrict__ bx,
                                          const double* __restrict__ by, const double* __restrict__ bz, int i,
                                          int j, int k) {
  RgCoef c;
  c.a[0] = bx[ridx(L, i + 1, j, k)] * L.inv_d2[0];
  c.a[1] = bx[ridx(L, i, j, k)] * L.inv_d2[0];
  c.a[2] = by[ridx(L, i, j + 1, k)] * L.inv_d2[1];
  c.a[3] = by[ridx(L, i, j, k)] * L.inv_d2[1];
  c.a[4] = bz[ridx(L, i, j, k + 1)] * L.inv_d2[2];
  c.a[5] = bz[ridx(L, i, j, k)] * L.inv_d2[2];
  c.diag = (c.a[0] + c.a[1] + c.a[2] + c.a[3] + c.a[4] + c.a[5]);
  c.inv = fabs(c.diag) < RG_EPS ? 0. : 1. / c.diag;
  return c;
}
__device__ __forceinline__ double rg_nbsum(const RgLv& L, const double* __restrict__ x, const RgCoef& c, int i,
                                           int j, int k) {
  const int ip = L.per[0] ? rwrap(i + 1, L.n[0]) : i + 1, im = L.per[0] ? rwrap(i - 1, L.n[0]) : i - 1;
  const int jp = L.per[1] ? rwrap(j + 1, L.n[1]) : j + 1, jm = L.per[1] ? rwrap(j - 1, L.n[1]) : j - 1;
  const int kp = L.per[2] ? rwrap(k + 1, L.n[2]) : k + 1, km = L.per[2] ? rwrap(k - 1, L.n[2]) : k - 1;
  return c.a[0] * x[ridx(L, ip, j, k)] + c.a[1] * x[ridx(L, im, j, k)] + c.a[2] * x[ridx(L, i, jp, k)] +
         c.a[3] * x[ridx(L, i, jm, k)] + c.a[4] * x[ridx(L, i, j, kp)] + c.a[5] * x[ridx(L, i, j, km)];
}

// k_jacobi_level_iteration (G_GMGSolver.cu:692-717)
__global__ __launch_bounds__(RGB) void k_rg_jacobi(RgLv L, const double* __restrict__ bx,
                                                   const double* __restrict__ by, const double* __restrict__ bz,
                                                   const double* __restrict__ q, double* __restrict__ qt,
                                                   const double* __restrict__ rhs) {
  int i, j, k;
  if (!rg_cell(L, i, j, k)) return;
  const RgCoef c = rg_coef(L, bx, by, bz, i, j, k);
  const double tmp_p = rg_nbsum(L, q, c, i, j, k);
  const size_t id = ridx(L, i, j, k);
  const double omega = RG_OMEGA;
  qt[id] = (1.0 - omega) * q[id] + omega * (tmp_p + rhs[id]) * c.inv;
}

// k_get_res_levels + k_restrict_level_to_level (G_GMGSolver.cu:152-188,457-493):
// crhs = mean over the children in F of rhs - A q
__global__ __launch_bounds__(RGB) void k_rg_res_restrict(RgLv F, const double* __restrict__ bx,
                                                         const double* __restrict__ by,
                                                         const double* __restrict__ bz,
                                                         const double* __restrict__ q,
                                                         const double* __restrict__ rhs, RgLv C,
                                                         double* __restrict__ crhs) {
  int i, j, k;
  if (!rg_cell(C, i, j, k)) return;
  const int Q[3] = {i, j, k};
  int B[3], R[3];
#pragma unroll
  for (int e = 0; e < 3; e++) {
    B[e] = C.co[e] ? 2 * Q[e] - 1 : Q[e];
    R[e] = C.co[e] ? 2 : 1;
  }
  double count = 0., tmp = 0.;
  for (int iz = 0; iz < R[2]; iz++)
    for (int iy = 0; iy < R[1]; iy++)
      for (int ix = 0; ix < R[0]; ix++) {
        const int fi = B[0] + ix, fj = B[1] + iy, fk = B[2] + iz;
        const RgCoef c = rg_coef(F, bx, by, bz, fi, fj, fk);
        const size_t id = ridx(F, fi, fj, fk);
        const double Ap = q[id] * c.diag - rg_nbsum(F, q, c, fi, fj, fk);
        tmp += rhs[id] - Ap;
        count += 1.0;
      }
  crhs[ridx(C, i, j, k)] = tmp / count;
}

// k_propagate_level_to_level (G_GMGSolver.cu:355-389)
__global__ __launch_bounds__(RGB) void k_rg_prolong(RgLv C, const double* __restrict__ cq, RgLv F,
                                                    double* __restrict__ fq) {
  int i, j, k;
  if (!rg_cell(C, i, j, k)) return;
  const int Q[3] = {i, j, k};
  int B[3], R[3];
#pragma unroll
  for (int e = 0; e < 3; e++) {
    B[e] = C.co[e] ? 2 * Q[e] - 1 : Q[e];
    R[e] = C.co[e] ? 2 : 1;
  }
  const double prop = cq[ridx(C, i, j, k)];
  for (int iz = 0; iz < R[2]; iz++)
    for (int iy = 0; iy < R[1]; iy++)
      for (int ix = 0; ix < R[0]; ix++) fq[ridx(F, B[0] + ix, B[1] + iy, B[2] + iz)] += prop;
}

// finest grid, row-split PCG vectors -----------------------------------------

// k_jacobi_iteration_general (G_GMGSolver.cu:719-746) with the grid operator
// of k_build_vof_poisson_A: out = (1-omega) x + omega (sum a_nb x_nb + r) / Adiag.
// zero_start: x is known to be zero (the first sweep of a V-cycle).
__global__ __launch_bounds__(256) void k_rg_fine_jacobi(Geo g, BetaF gb, const double* __restrict__ x,
                                                        double* __restrict__ out, const double* __restrict__ r,
                                                        int zero_start) {
  ROW_SETUP
  const int nx = g.n[0];
  const size_t ypr = idx(g, 0, W(g, 1, j + 1), k), ymr = idx(g, 0, W(g, 1, j - 1), k);
  const size_t zpr = idx(g, 0, j, W(g, 2, k + 1)), zmr = idx(g, 0, j, W(g, 2, k - 1));
  const double omega = RG_OMEGA;
  for (int i = 1 + lane; i <= nx; i += 64) {
    const Coef c = gb.b[0] ? coef_var(g, gb.b, i, j, k) : coef_uniform(g.n, g.per, g.inv_d2, g.beta0, i, j, k);
    const int p = spos(i, nx);
    double xc = 0.0, xp = 0.0, xm = 0.0, yp = 0.0, ym = 0.0, zp = 0.0, zm = 0.0;
    if (!zero_start) {
      xc = x[rb + p];
      xp = x[rb + spos(W(g, 0, i + 1), nx)];
      xm = x[rb + spos(W(g, 0, i - 1), nx)];
      yp = x[ypr + p];
      ym = x[ymr + p];
      zp = x[zpr + p];
      zm = x[zmr + p];
    }
    const double tmp_p = c.a[0] * xp + c.a[1] * xm + c.a[2] * yp + c.a[3] * ym + c.a[4] * zp + c.a[5] * zm;
    out[rb + p] = (1.0 - omega) * xc + omega * (tmp_p + r[rb + p]) * (1. / c.diag);
  }
}

// k_get_res_general + k_restrict_grid_to_level0 (G_GMGSolver.cu:191-226,416-455)
__global__ __launch_bounds__(RGB) void k_rg_fine_res_restrict(Geo g, BetaF gb, const double* __restrict__ x,
                                                              const double* __restrict__ r, RgLv C,
                                                              double* __restrict__ crhs) {
  int i, j, k;
  if (!rg_cell(C, i, j, k)) return;
  const int Q[3] = {i, j, k};
  int B[3], R[3];
#pragma unroll
  for (int e = 0; e < 3; e++) {
    B[e] = C.co[e] ? 2 * Q[e] - 1 : Q[e];
    R[e] = C.co[e] ? 2 : 1;
  }
  const int nx = g.n[0];
  double count = 0., tmp = 0.;
  for (int iz = 0; iz < R[2]; iz++)
    for (int iy = 0; iy < R[1]; iy++)
      for (int ix = 0; ix < R[0]; ix++) {
        const int fi = B[0] + ix, fj = B[1] + iy, fk = B[2] + iz;
        const Coef c =
            gb.b[0] ? coef_var(g, gb.b, fi, fj, fk) : coef_uniform(g.n, g.per, g.inv_d2, g.beta0, fi, fj, fk);
        const size_t rb = idx(g, 0, fj, fk);
        const int p = spos(fi, nx);
        const double xc = x[rb + p];
        const double xp = x[rb + spos(W(g, 0, fi + 1), nx)], xm = x[rb + spos(W(g, 0, fi - 1), nx)];
        const double yp = x[idx(g, 0, W(g, 1, fj + 1), fk) + p], ym = x[idx(g, 0, W(g, 1, fj - 1), fk) + p];
        const double zp = x[idx(g, 0, fj, W(g, 2, fk + 1)) + p], zm = x[idx(g, 0, fj, W(g, 2, fk - 1)) + p];
        const double s = c.a[0] * xp + c.a[1] * xm + c.a[2] * yp + c.a[3] * ym + c.a[4] * zp + c.a[5] * zm;
        tmp += r[rb + p] - (c.diag * xc - s);
        count += 1.0;
      }
  crhs[ridx(C, i, j, k)] = tmp / count;
}

// k_propagate_level0_to_array (G_GMGSolver.cu:285-316) into the row-split x
__global__ __launch_bounds__(RGB) void k_rg_prolong_fine(RgLv C, const double* __restrict__ cq, Geo g,
                                                         double* __restrict__ x) {
  int i, j, k;
  if (!rg_cell(C, i, j, k)) return;
  const int Q[3] = {i, j, k};
  int B[3], R[3];
#pragma unroll
  for (int e = 0; e < 3; e++) {
    B[e] = C.co[e] ? 2 * Q[e] - 1 : Q[e];
    R[e] = C.co[e] ? 2 : 1;
  }
  const double prop = cq[ridx(C, i, j, k)];
  for (int iz = 0; iz < R[2]; iz++)
    for (int iy = 0; iy < R[1]; iy++)
      for (int ix = 0; ix < R[0]; ix++)
        x[idx(g, 0, B[1] + iy, B[2] + iz) + spos(B[0] + ix, g.n[0])] += prop;
}

__global__ __launch_bounds__(RGB) void k_rg_zero(double* __restrict__ x, size_t n) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) x[t] = 0.0;
}

// r += a*S[slot] on interior cells; part0 <- row sums of r^2, part1 <- row max |r|
// (subtract_cell_mean, G_PressureSolverBase.cu:142-155, with the norms of the
// convergence check taken on the result)
__global__ __launch_bounds__(256) void k_add_scalar_norms(Geo g, double* __restrict__ r, double a,
                                                          const double* __restrict__ S, int slot,
                                                          double* __restrict__ part0,
                                                          double* __restrict__ part1) {
  ROW_SETUP
  const double s = S[slot];
  double a0 = 0.0, mx = 0.0;
  for (int i = 1 + lane; i <= g.n[0]; i += 64) {
    const size_t o = rb + spos(i, g.n[0]);
    const double v = r[o] + a * s;
    r[o] = v;
    a0 += v * v;
    const double ar = fabs(v);
    if (ar > mx || ar != ar) mx = ar;
  }
  a0 = wave_tree_sum(a0);
  mx = wave_max(mx);
  if (lane == 0) {
    part0[row] = a0;
    part1[row] = mx;
  }
}

// ------------------------------------------------------------- small levels
// On levels and grids of up to RG_TILE_CELLS cells a sweep is bound by its
// launch (2.8 us for a few thousand cells), and the V-cycle takes 46 of them.
//
// k_rg_down / k_rg_up do a level's four sweeps with its residual and
// restriction, or with the prolongation before them, in one launch: a block
// owns an 8^3 tile, holds it with a halo of 4 in LDS (two copies, as Jacobi
// reads the old values) and repeats its neighbours' work there, each sweep on
// a region one cell smaller. k_rg_tail does all levels that fit one
// workgroup's LDS, from the first of them down to the coarsest sweeps and
// back. Per cell the operations and their order are those of the sweeps above.
// Bound by latency: 64x32x32 11 us down and 11 us up where nine launches took
// 28 and 20 us; the 32x16x16 level 8 us each way against 20; the 38 sweeps of
// the levels 16x8x8 and 8x8x8 16.6 us against 115 (18.8 while
// each sweep formed its neighbours' places anew).
constexpr int RB_T = 8, RB_H = 4, RB_W = RB_T + 2 * RB_H, RB_N = RB_W * RB_W * RB_W;

// FINE: the finest grid (row-split vectors, its own operator), else a level
template <bool FINE, bool VAR>
struct RgView {
  Geo g;
  BetaF gb;
  RgLv L;
  const double* b[3];
  __device__ __forceinline__ int n(int d) const { return FINE ? g.n[d] : L.n[d]; }
  __device__ __forceinline__ int per(int d) const { return FINE ? g.per[d] : L.per[d]; }
  __device__ __forceinline__ size_t at(int i, int j, int k) const {
    if constexpr (FINE) return idx(g, 0, j, k) + (size_t)spos(i, g.n[0]);
    return ridx(L, i, j, k);
  }
  __device__ __forceinline__ RgCoef coef(int i, int j, int k) const {
    if constexpr (FINE) {
      const Coef c = VAR ? coef_var(g, gb.b, i, j, k) : coef_uniform(g.n, g.per, g.inv_d2, g.beta0, i, j, k);
      RgCoef r;
#pragma unroll
      for (int m = 0; m < 6; m++) r.a[m] = c.a[m];
      r.diag = c.diag;
      r.inv = 1. / c.diag;
      return r;
    }
    return rg_coef(L, b[0], b[1], b[2], i, j, k);
  }
};
// one sweep's new value at p of x, neighbours at p +- 1, +- sy, +- sz
__device__ __forceinline__ double rg_relax(const double* x, int p, int sy, int sz, const RgCoef& c, double rhs) {
  const double omega = RG_OMEGA;
  const double s = c.a[0] * x[p + 1] + c.a[1] * x[p - 1] + c.a[2] * x[p + sy] + c.a[3] * x[p - sy] +
                   c.a[4] * x[p + sz] + c.a[5] * x[p - sz];
  return (1.0 - omega) * x[p] + omega * (s + rhs) * c.inv;
}
__device__ __forceinline__ int rg_dist(int l) { return max(max(RB_H - l, l - (RB_H + RB_T - 1)), 0); }
// image of v in 1..n of a periodic axis: -3 <= v <= n + 11, n >= 4
__device__ __forceinline__ int rg_image(int v, int n) {
  v += v < 1 ? n : 0;
#pragma unroll
  for (int u = 0; u < 3; u++) v -= v > n ? n : 0;
  return v;
}
// The four cells of a thread in the box (planes lz = t >> 8, + 4, + 8, + 12)
struct RgCell {
  int i, j, k, d;  // in 1..n; cells outside the tile, 15 = none
  bool own;        // in the tile and the grid, not an image
};
template <class V>
__device__ __forceinline__ RgCell rg_box_cell(const V& v, const int o[3], int m) {
  const int t = (int)threadIdx.x;
  const int l[3] = {t & 15, (t >> 4) & 15, (t >> 8) + 4 * m};
  int q[3];
  RgCell c;
  c.d = 0;
  c.own = true;
  bool ok = true;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const int x = o[d] - RB_H + l[d];
    const bool in = x >= 1 && x <= v.n(d);
    c.d = max(c.d, rg_dist(l[d]));
    c.own = c.own && in;
    q[d] = v.per(d) ? rg_image(x, v.n(d)) : x;
    ok = ok && (in || v.per(d));
  }
  c.own = c.own && c.d == 0;
  if (!ok) c.d = 15;
  c.i = q[0];
  c.j = q[1];
  c.k = q[2];
  return c;
}

template <bool FINE, bool VAR>
__global__ __launch_bounds__(1024) void k_rg_down(RgView<FINE, VAR> V, const double* __restrict__ rhs,
                                                  double* __restrict__ q, RgLv C, double* __restrict__ crhs) {
  __shared__ double X[2][RB_N];
  constexpr int SY = RB_W, SZ = RB_W * RB_W;
  const int t = (int)threadIdx.x;
  const int o[3] = {1 + RB_T * (int)blockIdx.x, 1 + RB_T * (int)blockIdx.y, 1 + RB_T * (int)blockIdx.z};
  RgCell c[4];
  RgCoef k[4];
  double f[4];
#pragma unroll
  for (int m = 0; m < 4; m++) {
    c[m] = rg_box_cell(V, o, m);
    f[m] = 0.0;
    if (c[m].d <= 4) {
      f[m] = rhs[V.at(c[m].i, c[m].j, c[m].k)];
      k[m] = V.coef(c[m].i, c[m].j, c[m].k);
    }
  }
  const double omega = RG_OMEGA;
#pragma unroll
  for (int m = 0; m < 4; m++) {
    // from zero: the neighbour sum is 0
    X[0][t + 1024 * m] = c[m].d <= 4 ? (1.0 - omega) * 0.0 + omega * (0.0 + f[m]) * k[m].inv : 0.0;
    X[1][t + 1024 * m] = 0.0;
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < 3; s++) {
#pragma unroll
    for (int m = 0; m < 4; m++)
      if (c[m].d <= 3 - s) X[(s + 1) & 1][t + 1024 * m] = rg_relax(X[s & 1], t + 1024 * m, SY, SZ, k[m], f[m]);
    __syncthreads();
  }
  // the sweeps' result is in X[1]; residual of the tile's cells into X[0]
#pragma unroll
  for (int m = 0; m < 4; m++) {
    if (c[m].own) {
      const int p = t + 1024 * m;
      const double* x = X[1];
      const double s = k[m].a[0] * x[p + 1] + k[m].a[1] * x[p - 1] + k[m].a[2] * x[p + SY] + k[m].a[3] * x[p - SY] +
                       k[m].a[4] * x[p + SZ] + k[m].a[5] * x[p - SZ];
      const double Ap = x[p] * k[m].diag - s;
      X[0][p] = f[m] - Ap;
      q[V.at(c[m].i, c[m].j, c[m].k)] = x[p];
    }
  }
  __syncthreads();
  const int w[3] = {C.co[0] ? RB_T / 2 : RB_T, C.co[1] ? RB_T / 2 : RB_T, C.co[2] ? RB_T / 2 : RB_T};
  if (t < w[0] * w[1] * w[2]) {
    const int a[3] = {t % w[0], (t / w[0]) % w[1], t / (w[0] * w[1])};
    int Q[3], l0[3], R[3];
    bool in = true;
#pragma unroll
    for (int d = 0; d < 3; d++) {
      R[d] = C.co[d] ? 2 : 1;
      l0[d] = RB_H + R[d] * a[d];
      Q[d] = (C.co[d] ? (o[d] + 1) / 2 : o[d]) + a[d];
      in = in && Q[d] <= C.n[d];
    }
    if (in) {
      double count = 0., tmp = 0.;
      for (int iz = 0; iz < R[2]; iz++)
        for (int iy = 0; iy < R[1]; iy++)
          for (int ix = 0; ix < R[0]; ix++) {
            tmp += X[0][(l0[2] + iz) * SZ + (l0[1] + iy) * SY + l0[0] + ix];
            count += 1.0;
          }
      crhs[ridx(C, Q[0], Q[1], Q[2])] = tmp / count;
    }
  }
}

template <bool FINE, bool VAR>
__global__ __launch_bounds__(1024) void k_rg_up(RgView<FINE, VAR> V, RgLv C, const double* __restrict__ cq,
                                                const double* __restrict__ qi, const double* __restrict__ rhs,
                                                double* __restrict__ qo) {
  __shared__ double X[2][RB_N];
  constexpr int SY = RB_W, SZ = RB_W * RB_W;
  const int t = (int)threadIdx.x;
  const int o[3] = {1 + RB_T * (int)blockIdx.x, 1 + RB_T * (int)blockIdx.y, 1 + RB_T * (int)blockIdx.z};
  RgCell c[4];
  RgCoef k[4];
  double f[4];
#pragma unroll
  for (int m = 0; m < 4; m++) {
    c[m] = rg_box_cell(V, o, m);
    f[m] = 0.0;
    double x = 0.0;
    if (c[m].d <= 4) {
      const int ci = C.co[0] ? (c[m].i + 1) / 2 : c[m].i, cj = C.co[1] ? (c[m].j + 1) / 2 : c[m].j,
                ck = C.co[2] ? (c[m].k + 1) / 2 : c[m].k;
      x = qi[V.at(c[m].i, c[m].j, c[m].k)] + cq[ridx(C, ci, cj, ck)];
    }
    if (c[m].d <= 3) {
      f[m] = rhs[V.at(c[m].i, c[m].j, c[m].k)];
      k[m] = V.coef(c[m].i, c[m].j, c[m].k);
    }
    X[0][t + 1024 * m] = x;
    X[1][t + 1024 * m] = 0.0;
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < 3; s++) {
#pragma unroll
    for (int m = 0; m < 4; m++)
      if (c[m].d <= 3 - s) X[(s + 1) & 1][t + 1024 * m] = rg_relax(X[s & 1], t + 1024 * m, SY, SZ, k[m], f[m]);
    __syncthreads();
  }
#pragma unroll
  for (int m = 0; m < 4; m++)
    if (c[m].own) qo[V.at(c[m].i, c[m].j, c[m].k)] = rg_relax(X[1], t + 1024 * m, SY, SZ, k[m], f[m]);
}

// Levels first..last in one workgroup: a thread owns the cells t, t + 1024, ..
// of the current level (its coefficients in registers), the level's values lie
// in LDS with a zero ghost layer, twice.
template <int CPT>
__global__ __launch_bounds__(1024) void k_rg_tail(const RgTailLv* __restrict__ T, int first, int last, int nf, int nc) {
  __shared__ double X[2][RG_TAIL_PAD];
  const int t = (int)threadIdx.x;
  double a[CPT][6], inv[CPT], f[CPT];
  // LDS index (-1: no cell), the neighbours' (two to a word where the registers are short)
  constexpr bool PACK = CPT > 1;
  double own[PACK ? 1 : CPT];  // the cell's value in X[cur]
  int p[CPT], nb[CPT][PACK ? 3 : 6];
  size_t at[CPT];
  int cur = 0;
  // the level's coefficients and right-hand side, both copies of X zero
  auto load = [&](int l) {
    const RgTailLv& V = T[l];
    const RgLv& L = V.L;
    const int sy = L.n[0] + 2, sz = sy * (L.n[1] + 2), pad = sz * (L.n[2] + 2);
    for (int e = t; e < pad; e += 1024) {
      X[0][e] = 0.0;
      X[1][e] = 0.0;
    }
    cur = 0;
    const int nxy = L.n[0] * L.n[1], cells = nxy * L.n[2];
#pragma unroll
    for (int u = 0; u < CPT; u++) {
      const int e = t + 1024 * u;
      p[u] = -1;
      f[u] = 0.0;
      if constexpr (!PACK) own[u] = 0.0;
      if (e < cells) {
        const int i = e % L.n[0] + 1, j = (e / L.n[0]) % L.n[1] + 1, k = e / nxy + 1;
        p[u] = k * sz + j * sy + i;
        at[u] = ridx(L, i, j, k);
        f[u] = V.rhs[at[u]];
        const RgCoef c = rg_coef(L, V.b[0], V.b[1], V.b[2], i, j, k);
#pragma unroll
        for (int m = 0; m < 6; m++) a[u][m] = c.a[m];
        inv[u] = c.inv;
        const int q[3] = {i, j, k}, st[3] = {1, sy, sz};
#pragma unroll
        for (int d = 0; d < 3; d++) {
          const int hi = L.per[d] && q[d] == L.n[d] ? -(L.n[d] - 1) * st[d] : st[d];
          const int lo = L.per[d] && q[d] == 1 ? (L.n[d] - 1) * st[d] : -st[d];
          if constexpr (PACK) {
            nb[u][d] = (p[u] + hi) | (p[u] + lo) << 16;
          } else {
            nb[u][2 * d] = p[u] + hi;
            nb[u][2 * d + 1] = p[u] + lo;
          }
        }
      }
    }
  };
  auto nbsum = [&](const double* x, int u) -> double {
    double v[6];
#pragma unroll
    for (int m = 0; m < 6; m++) {
      if constexpr (PACK) v[m] = x[m & 1 ? nb[u][m / 2] >> 16 : nb[u][m / 2] & 0xffff];
      else v[m] = x[nb[u][m]];
    }
    return a[u][0] * v[0] + a[u][1] * v[1] + a[u][2] * v[2] + a[u][3] * v[3] + a[u][4] * v[4] + a[u][5] * v[5];
  };
  // the cell's value in x = X[cur]
  auto val = [&](const double* x, int u) -> double {
    if constexpr (PACK) return x[p[u]];
    else return own[u];
  };
  auto sweep = [&](const double* x, double* y) {
    const double omega = RG_OMEGA;
#pragma unroll
    for (int u = 0; u < CPT; u++)
      if (p[u] >= 0) {
        const double v = (1.0 - omega) * val(x, u) + omega * (nbsum(x, u) + f[u]) * inv[u];
        y[p[u]] = v;
        if constexpr (!PACK) own[u] = v;
      }
    __syncthreads();
  };
  // n sweeps from X[0]; with one cell a thread two at a time, so that the copies'
  // addresses are fixed (with four the longer loop costs more than it saves)
  auto sweeps = [&](int n) {
    if constexpr (PACK) {
#pragma unroll 1
      for (int it = 0; it < n; it++) {
        sweep(X[cur], X[1 - cur]);
        cur = 1 - cur;
      }
    } else {
#pragma unroll 1
      for (int it = 0; it + 1 < n; it += 2) {
        sweep(X[0], X[1]);
        sweep(X[1], X[0]);
      }
      if (n & 1) sweep(X[0], X[1]);
      cur = n & 1;
    }
  };
  auto store = [&](int l) {
#pragma unroll
    for (int u = 0; u < CPT; u++)
      if (p[u] >= 0) T[l].q[at[u]] = val(X[cur], u);
  };
#pragma unroll 1
  for (int l = first; l < last; l++) {
    load(l);
    __syncthreads();
    sweeps(nf);
    store(l);
    double* res = X[1 - cur];
#pragma unroll
    for (int u = 0; u < CPT; u++)
      if (p[u] >= 0) {
        const double diag = (a[u][0] + a[u][1] + a[u][2] + a[u][3] + a[u][4] + a[u][5]);
        const double Ap = val(X[cur], u) * diag - nbsum(X[cur], u);
        res[p[u]] = f[u] - Ap;
      }
    __syncthreads();
    const RgLv& L = T[l].L;
    const RgLv& C = T[l + 1].L;
    const int sy = L.n[0] + 2, sz = sy * (L.n[1] + 2);
    for (int e = t; e < C.n[0] * C.n[1] * C.n[2]; e += 1024) {
      const int Q[3] = {e % C.n[0] + 1, (e / C.n[0]) % C.n[1] + 1, e / (C.n[0] * C.n[1]) + 1};
      int B[3], R[3];
#pragma unroll
      for (int d = 0; d < 3; d++) {
        B[d] = C.co[d] ? 2 * Q[d] - 1 : Q[d];
        R[d] = C.co[d] ? 2 : 1;
      }
      double count = 0., tmp = 0.;
      for (int iz = 0; iz < R[2]; iz++)
        for (int iy = 0; iy < R[1]; iy++)
          for (int ix = 0; ix < R[0]; ix++) {
            tmp += res[(B[2] + iz) * sz + (B[1] + iy) * sy + B[0] + ix];
            count += 1.0;
          }
      T[l + 1].rhs[ridx(C, Q[0], Q[1], Q[2])] = tmp / count;
    }
    __syncthreads();
  }
  load(last);
  __syncthreads();
  sweeps(nc);
  store(last);
  __syncthreads();
#pragma unroll 1
  for (int l = last - 1; l >= first; l--) {
    load(l);
    __syncthreads();
    const RgTailLv& V = T[l];
    const RgLv& C = T[l + 1].L;
#pragma unroll
    for (int u = 0; u < CPT; u++)
      if (p[u] >= 0) {
        const int e = t + 1024 * u;
        int Q[3] = {e % V.L.n[0] + 1, (e / V.L.n[0]) % V.L.n[1] + 1, e / (V.L.n[0] * V.L.n[1]) + 1};
#pragma unroll
        for (int d = 0; d < 3; d++) Q[d] = C.co[d] ? (Q[d] + 1) / 2 : Q[d];
        const double v = V.q[at[u]] + T[l + 1].q[ridx(C, Q[0], Q[1], Q[2])];
        X[0][p[u]] = v;
        if constexpr (!PACK) own[u] = v;
      }
    __syncthreads();
    sweeps(nf);
    store(l);
    __syncthreads();
  }
}

dim3 cells_grid(const RgLv& L) {
  size_t n = (size_t)L.n[0] * L.n[1] * L.n[2];
  return dim3((unsigned)((n + RGB - 1) / RGB));
}
dim3 rows_grid_g(const Geo& g) { return dim3((unsigned)((g.n[1] * g.n[2] + 3) / 4)); }

}  // namespace

void launch_rg_beta(const Geo& g, const BetaF* gb, const RgLv& C, const RgLv& F, const double* fb, int d,
                    double* cb, hipStream_t st) {
  size_t n = (size_t)(C.n[0] + (d == 0)) * (size_t)(C.n[1] + (d == 1)) * (size_t)(C.n[2] + (d == 2));
  hipLaunchKernelGGL(k_rg_beta, dim3((unsigned)((n + RGB - 1) / RGB)), dim3(RGB), 0, st, g, gb ? *gb : BetaF{}, C,
                     F, fb, d, cb);
}
void launch_rg_jacobi(const RgLv& L, double* const b[3], const double* q, double* qt, const double* rhs,
                      hipStream_t st) {
  hipLaunchKernelGGL(k_rg_jacobi, cells_grid(L), dim3(RGB), 0, st, L, b[0], b[1], b[2], q, qt, rhs);
}
void launch_rg_res_restrict(const RgLv& F, double* const b[3], const double* q, const double* rhs, const RgLv& C,
                            double* crhs, hipStream_t st) {
  hipLaunchKernelGGL(k_rg_res_restrict, cells_grid(C), dim3(RGB), 0, st, F, b[0], b[1], b[2], q, rhs, C, crhs);
}
void launch_rg_prolong(const RgLv& C, const double* cq, const RgLv& F, double* fq, hipStream_t st) {
  hipLaunchKernelGGL(k_rg_prolong, cells_grid(C), dim3(RGB), 0, st, C, cq, F, fq);
}
void launch_rg_fine_jacobi(const Geo& g, const BetaF* gb, const double* x, double* out, const double* r,
                           int zero_start, hipStream_t st) {
  hipLaunchKernelGGL(k_rg_fine_jacobi, rows_grid_g(g), dim3(256), 0, st, g, gb ? *gb : BetaF{}, x, out, r,
                     zero_start);
}
void launch_rg_fine_res_restrict(const Geo& g, const BetaF* gb, const double* x, const double* r, const RgLv& C,
                                 double* crhs, hipStream_t st) {
  hipLaunchKernelGGL(k_rg_fine_res_restrict, cells_grid(C), dim3(RGB), 0, st, g, gb ? *gb : BetaF{}, x, r, C,
                     crhs);
}
void launch_rg_prolong_fine(const RgLv& C, const double* cq, const Geo& g, double* x, hipStream_t st) {
  hipLaunchKernelGGL(k_rg_prolong_fine, cells_grid(C), dim3(RGB), 0, st, C, cq, g, x);
}
static dim3 rg_tiles(const int n[3]) {
  return dim3((unsigned)((n[0] + RB_T - 1) / RB_T), (unsigned)((n[1] + RB_T - 1) / RB_T),
              (unsigned)((n[2] + RB_T - 1) / RB_T));
}
// every axis at least 4 cells (the box's periodic images), few enough of them
bool rg_tile_applies(const int n[3]) {
  return n[0] >= 4 && n[1] >= 4 && n[2] >= 4 && (size_t)n[0] * n[1] * n[2] <= RG_TILE_CELLS;
}
bool rg_tail_applies(const RgLv& L) {
  return L.n[0] * L.n[1] * L.n[2] <= RG_TAIL_CELLS && (L.n[0] + 2) * (L.n[1] + 2) * (L.n[2] + 2) <= RG_TAIL_PAD;
}
void launch_rg_down(const RgLv& L, double* const b[3], const double* rhs, double* q, const RgLv& C, double* crhs,
                    hipStream_t st) {
  RgView<false, true> V{};
  V.L = L;
  for (int d = 0; d < 3; d++) V.b[d] = b[d];
  hipLaunchKernelGGL((k_rg_down<false, true>), rg_tiles(L.n), dim3(1024), 0, st, V, rhs, q, C, crhs);
}
void launch_rg_up(const RgLv& L, double* const b[3], const RgLv& C, const double* cq, const double* qi,
                  const double* rhs, double* qo, hipStream_t st) {
  RgView<false, true> V{};
  V.L = L;
  for (int d = 0; d < 3; d++) V.b[d] = b[d];
  hipLaunchKernelGGL((k_rg_up<false, true>), rg_tiles(L.n), dim3(1024), 0, st, V, C, cq, qi, rhs, qo);
}
void launch_rg_fine_down(const Geo& g, const BetaF* gb, const double* r, double* x, const RgLv& C, double* crhs,
                         hipStream_t st) {
  if (gb) {
    RgView<true, true> V{};
    V.g = g;
    V.gb = *gb;
    hipLaunchKernelGGL((k_rg_down<true, true>), rg_tiles(g.n), dim3(1024), 0, st, V, r, x, C, crhs);
  } else {
    RgView<true, false> V{};
    V.g = g;
    hipLaunchKernelGGL((k_rg_down<true, false>), rg_tiles(g.n), dim3(1024), 0, st, V, r, x, C, crhs);
  }
}
void launch_rg_fine_up(const Geo& g, const BetaF* gb, const RgLv& C, const double* cq, const double* xi,
                       const double* r, double* xo, hipStream_t st) {
  if (gb) {
    RgView<true, true> V{};
    V.g = g;
    V.gb = *gb;
    hipLaunchKernelGGL((k_rg_up<true, true>), rg_tiles(g.n), dim3(1024), 0, st, V, C, cq, xi, r, xo);
  } else {
    RgView<true, false> V{};
    V.g = g;
    hipLaunchKernelGGL((k_rg_up<true, false>), rg_tiles(g.n), dim3(1024), 0, st, V, C, cq, xi, r, xo);
  }
}
void launch_rg_tail(const RgTailLv* T, int first, int last, int nf, int nc, int small, hipStream_t st) {
  if (small) hipLaunchKernelGGL(k_rg_tail<1>, dim3(1), dim3(1024), 0, st, T, first, last, nf, nc);
  else hipLaunchKernelGGL(k_rg_tail<4>, dim3(1), dim3(1024), 0, st, T, first, last, nf, nc);
}
void launch_rg_zero(double* x, size_t n, hipStream_t st) {
  hipLaunchKernelGGL(k_rg_zero, dim3((unsigned)((n + RGB - 1) / RGB)), dim3(RGB), 0, st, x, n);
}
void launch_add_scalar_norms(const Geo& g, double* r, double a, const double* S, int slot, double* p0, double* p1,
                             hipStream_t st) {
  hipLaunchKernelGGL(k_add_scalar_norms, rows_grid_g(g), dim3(256), 0, st, g, r, a, S, slot, p0, p1);
}

}  // namespace smac
