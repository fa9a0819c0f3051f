// smac_adjoint.hip -- adjoint (vector-Jacobian product) of one SMAC step.
//
// Forward step, from (u^n, p^n):
//   u*      = F(u^n) - dt beta G p^n           predictor (F holds
//                                              the time, stress and MUSCL terms)
//   b       = -(1/dt) D u*                     RHS
//   dp      = A^+ (b - mean b)                 pressure solve
//   u^{n+1} = u* - dt beta G dp  (interior faces; wall faces keep u^n)
//   p^{n+1} = p^n + dp
// With cotangents (ub', pb') of (u^{n+1}, p^{n+1}) the cotangents of (u^n, p^n):
//   dpb  = pb' + dt D_i(beta ub')              D_i: divergence over interior faces
//   bb   = A^+ (dpb - mean dpb)                second (self-adjoint) Poisson solve
//   ub*  = ub' + (1/dt) G bb      on interior faces
//   pb   = pb' + dt D_i(beta ub*)
//   ub   = (dF/du)^T ub*  (+ ub' on wall faces)
// (dF/du)^T is formed face by face: each interior face re-evaluates its
// predictor stencil, sums the partial derivatives of the branch the forward took
// (upwind side, minmod slope) per entry read, and adds them with FP64 atomics to
// a tile in LDS, whose finished planes go to ub with FP64 atomics. Sums over the
// scatter are therefore order-dependent in the last bits; every other stage is
// a deterministic gather.
#include <type_traits>

#include "smac_internal.hpp"
#include "smac_predict.hpp"

namespace smac {

namespace {

constexpr dim3 CELLB_A(64, 4);

struct Acc {
  double* ub[3];
};
// Cotangent sinks of the VoF adjoint (the step after a transport): Fb = the
// accumulated alpha flux of each axis (faces), anp1 = alpha^{n+1} (the
// properties rho, mu, beta of the step), an = alpha^n (rho_old); the
// property derivatives d rho / d alpha = drho, d mu / d alpha = dmu.
struct AccV {
  double* Fb[3];
  double* anp1;
  double* an;
  double drho, dmu;
};

// branch of minmod(dpv, dmv): 0 -> 0, 1 -> dpv, 2 -> dmv (d_minmod,
// CFD/G_SMACSolver.cu:67-88)
__device__ __forceinline__ int minmod_sel(double dp, double dm) {
  if (dp * dm > 0.) return fabs(dp) < fabs(dm) ? 1 : 2;
  return 0;
}

// adjoint of M = m (uw + sgn(m) 0.5 s) of one side on the five values c: cM =
// cotangent of M; to the values in cb; returns that of m. hi: the side's minus
// value is c[hi-1], its plus value c[hi] (3 for the + side, 2 for the -); mine:
// the upwind value is c[2]; slope: is its slope used?
template <int HI>
__device__ __forceinline__ double flux_vjp(double m, const double c[5], bool inner, double cM, double cb[5]) {
  const bool low = m > 0.;  // the upwind value is c[HI-1], else c[HI]
  const bool slope = (HI == 3 ? low : !low) || inner;
  const double uw = low ? c[HI - 1] : c[HI];
  const double dpv = low ? c[HI] - c[HI - 1] : c[HI + 1] - c[HI];
  const double dmv = low ? c[HI - 1] - c[HI - 2] : c[HI] - c[HI - 1];
  const int sel = slope ? minmod_sel(dpv, dmv) : 0;
  const double s = sel == 1 ? dpv : (sel == 2 ? dmv : 0.0);
  const int dir = sgn(m);
  const double up = uw + dir * 0.5 * s;
  // dM/dm = up; dM/duw = m; dM/ds = m sgn(m) 0.5, s = sa - sb (1) or sb - sc (2)
  const double cs = m * dir * 0.5 * cM;
  const double sa = sel == 1 ? cs : 0.0, sc = sel == 2 ? -cs : 0.0;
  const double sb = m * cM + (sel == 1 ? -cs : (sel == 2 ? cs : 0.0));
  cb[HI + 1] += low ? 0.0 : sa;
  cb[HI] += low ? sa : sb;
  cb[HI - 1] += low ? sb : sc;
  cb[HI - 2] += low ? sc : 0.0;
  return up * cM;
}

// (d u*_A(q) / d u^n)^T w (the pressure term is separate): addu(c, d, s, r, v)
// adds v to component c at q + s e_d + r e_A, once per entry; an axis is finished
// before the next, so that few sums are held at a time.
// VOF: the step after a VoF transport -- mass flux with the accumulated alpha
// flux and the property cotangents: beta = 1/rho_f and mu of alpha^{n+1},
// rho_old of alpha^n; addq(f, d, s, r, v) likewise, f = the axis of the flux, 3 =
// alpha^{n+1}, 4 = alpha^n
template <int A, bool VAR, bool VOF, class AddU, class AddQ>
__device__ __forceinline__ void face_vjp(const Geo& g, const Props& P, const VofF& M, const AccV& AV, const double* p,
                                         const Face<A, true>& F, double dt, double w, AddU addu, AddQ addq) {
  constexpr MassFlux MF = VOF ? MF_VOF : MF_RHO;
  const double v0 = F.c[A][2], beta = F.template beta<VAR>(g, P), rho_old_f = F.template rho_old<VAR>(g, P);
  double mp[3], mm[3];
  F.template mass<MF>(g, M, mp, mm);
  // u* = beta (v0 rho_old_f) + dt (beta tmp + g)
  double c0 = beta * rho_old_f * w;  // cotangent of v0
  const double W = dt * beta * w;    // cotangent of tmp
  const double muq = VAR ? P.mu[F.id] : g.mu0, mucm = VAR ? P.mu[F.at(A, -1)] : g.mu0;
  const double k2 = 2. * g.inv_d2[A] * W;
  double x0 = 0.0, xm = 0.0;  // cotangents of alpha^{n+1} in cells q and q - e_A
  if constexpr (VOF) {
    // beta = 1/(0.5 (rho_q + rho_cm)): d beta / d rho_c = -0.5 beta^2
    const double tmp = F.template bracket<VAR, MF>(g, P, M, nullptr, p, mp, mm);
    const double bb = w * (v0 * rho_old_f + dt * tmp);
    const double kr = AV.drho * (-0.5 * beta * beta * bb);
    // own-axis stresses mu_q (vp1 - v0) and mu_cm (v0 - vm1)
    x0 = kr + AV.dmu * (k2 * (F.c[A][3] - v0));
    xm = kr + AV.dmu * (-k2 * (v0 - F.c[A][1]));
    // rho_old_f = 0.5 (rho_old_q + rho_old_cm)
    const double ko = AV.drho * (0.5 * (w * beta * v0));
    addq(4, A, 0, 0, ko);
    addq(4, A, 0, -1, ko);
  }
#pragma unroll
  for (int B = 0; B < 3; B++) {
    if (B == A) continue;
    double mu_p, mu_m;
    F.template mu_edge<VAR>(g, P, B, mu_p, mu_m);
    const double k = W * g.inv_d[B];  // cotangent of t_p; -k of t_m
    const double kp = k * mu_p, km = k * mu_m;
    double c[5] = {0.0, km * g.inv_d[B], 0.0, kp * g.inv_d[B], 0.0};
    c0 += -kp * g.inv_d[B] - km * g.inv_d[B];
    // convection: -W (Mp - Mm) / h
    const double bp = 0.5 * flux_vjp<3>(mp[B], F.c[B], F.inp[B], -k, c);
    const double bm = 0.5 * flux_vjp<2>(mm[B], F.c[B], F.inm[B], k, c);
    double wpp = kp * g.inv_d[A] + g.rho0 * bp, wmp = -kp * g.inv_d[A] + g.rho0 * bp;
    double wp0 = -km * g.inv_d[A] + g.rho0 * bm, wm0 = km * g.inv_d[A] + g.rho0 * bm;
    c0 += c[2];
    const int x = F.q.v[B], n = g.n[B];
    const bool wl = !g.per[B] && x == 1, wh = !g.per[B] && x == n;
    if (!g.per[B]) {
      // mirrored values pass their cotangent on, a wall's own are constants
      const double fl = wall_even(g, 2 * B) ? 1.0 : -1.0, fh = wall_even(g, 2 * B + 1) ? 1.0 : -1.0;
      if (x == n - 1) {
        c[3] += fh * c[4];
        c[4] = 0.0;
      }
      if (wh) {
        c0 += fh * c[3];
        c[3] = 0.0;
        if (!wall_stored(g, B, 2 * B + 1)) wpp = wmp = 0.0;
      }
      if (x == 2) {
        c[1] += fl * c[0];
        c[0] = 0.0;
      }
      if (wl) {
        c0 += fl * c[1];
        c[1] = 0.0;
        if (!wall_stored(g, B, 2 * B)) wp0 = wm0 = 0.0;
      }
    }
    addu(A, B, -2, 0, c[0]);
    addu(A, B, -1, 0, c[1]);
    addu(A, B, 1, 0, c[3]);
    addu(A, B, 2, 0, c[4]);
    addu(B, B, 1, 0, wpp);
    addu(B, B, 1, -1, wmp);
    addu(B, B, 0, 0, wp0);
    addu(B, B, 0, -1, wm0);
    if constexpr (VOF) {
      const double kf = M.drho * M.hbydt[B], fp = kf * bp, fm = kf * bm;
      addq(B, B, 1, 0, fp);
      addq(B, B, 1, -1, fp);
      addq(B, B, 0, 0, fm);
      addq(B, B, 0, -1, fm);
      // mu_p = 0.5 (muf(q + e_B) + muf(q + e_B - e_A)), mu_m at q; muf is the mean
      // of its two cells on an interior face, the inner cell on a boundary face
      const double xp = AV.dmu * (0.5 * k * F.strain_p(g, B)), xq = AV.dmu * (-0.5 * k * F.strain_m(g, B));
      const double both = (wh ? xp : 0.5 * xp) + (wl ? xq : 0.5 * xq);
      x0 += both;
      xm += both;
      const double ap = wh ? 0.0 : 0.5 * xp, am = wl ? 0.0 : 0.5 * xq;
      addq(3, B, 1, 0, ap);
      addq(3, B, 1, -1, ap);
      addq(3, B, -1, 0, am);
      addq(3, B, -1, -1, am);
    }
  }
  double c[5] = {0.0, k2 * mucm, 0.0, k2 * muq, 0.0};
  const double k = W * g.inv_d[A];
  const double bp = 0.5 * flux_vjp<3>(mp[A], F.c[A], F.inp[A], -k, c);
  const double bm = 0.5 * flux_vjp<2>(mm[A], F.c[A], F.inm[A], k, c);
  c[1] += g.rho0 * bm;
  c[2] += g.rho0 * (bm + bp) + c0 - k2 * muq - k2 * mucm;
  c[3] += g.rho0 * bp;
  if (!g.per[A]) {
    const int x = F.q.v[A], n = g.n[A];
    const bool lo = wall_stored(g, A, 2 * A), hi = wall_stored(g, A, 2 * A + 1);
    if (x == 2 && !lo) c[1] = 0.0;
    if (x == 3 && !lo) c[0] = 0.0;
    if (x == n && !hi) c[3] = 0.0;
    if (x == n - 1 && !hi) c[4] = 0.0;
  }
#pragma unroll
  for (int s = -2; s <= 2; s++) addu(A, A, s, 0, c[s + 2]);
  if constexpr (VOF) {
    const double kf = M.drho * M.hbydt[A];
    addq(A, A, -1, 0, kf * bm);
    addq(A, A, 0, 0, kf * (bm + bp));
    addq(A, A, 1, 0, kf * bp);
    addq(3, A, 0, 0, x0);
    addq(3, A, 0, -1, xm);
  }
}

// (dF/du)^T ub*: a block marches a column of VX x VY cells through kc planes, the
// three components side by side (four waves each). The cotangents are summed in
// LDS, for the velocities in the five planes k-2 .. k+2 that plane k reaches, for
// the VoF sinks in three; a finished plane goes out with one atomic per entry
// touched. Each face's own sum over its ~50 partial derivatives is formed in
// registers first (21 entries, with VOF 44). Bound by the latency of the stencil
// reads and the LDS atomics: 128^3 204 us, 128x64x64 with VOF 182 us; one kernel
// per component with a global atomic per partial derivative took 2300 and 2100.
constexpr int VX = 64, VY = 4;
template <bool VAR, bool VOF>
__global__ __launch_bounds__(768) void k_predict_vjp(Geo g, Props P, Vel V, VofF M, const double* __restrict__ p,
                                                     Vel wbar, Acc U, AccV AV, double dt, int kc) {
  constexpr int PX = VX + 4, PL = PX * (VY + 4);  // velocity planes, two cells around
  constexpr int QX = VX + 2, QL = QX * (VY + 2);  // VoF planes, one cell around
  constexpr int NQ = VOF ? 3 * QL : 1;
  __shared__ double su[3][5 * PL];
  __shared__ double sf[VOF ? 5 : 1][NQ];  // Fb, anp1, an
  const int t = (int)threadIdx.x;
  const int x0 = 1 + VX * (int)blockIdx.x, y0 = 1 + VY * (int)blockIdx.y, z0 = 1 + kc * (int)blockIdx.z;
  const int z1 = min(z0 + kc - 1, g.n[2]);
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6), a = wv >> 2;
  const int lx = t & 63, ly = wv & 3, i = x0 + lx, j = y0 + ly;
  for (int e = t; e < 15 * PL; e += 768) su[0][e] = 0.0;
  if constexpr (VOF)
    for (int e = t; e < 5 * NQ; e += 768) sf[0][e] = 0.0;
  // plane z of the velocity sums / of the VoF sums
  auto pu = [&](int z) { return (z - z0 + 2) % 5 * PL; };
  auto pq = [&](int z) { return (z - z0 + 1) % 3 * QL; };
  auto face = [&](auto ac, int k) {
    constexpr int A = decltype(ac)::value;
    if (i > g.n[0] || j > g.n[1]) return;
    const I3 q = mk(i, j, k);
    if (!g.per[A] && q.v[A] < 2) return;
    const double w = wbar.c[A][IX(g, q)];
    if (w == 0.0) return;
    const Face<A, true> F(g, V, q);
    const int lo = ly * PX + lx, lq = ly * QX + lx;
    auto addu = [&](int c, int d, int s, int r, double v) {
      int o[3] = {0, 0, 0};
      o[d] += s;
      o[A] += r;
      unsafeAtomicAdd(su[c] + pu(k + o[2]) + (o[1] + 2) * PX + (o[0] + 2) + lo, v);
    };
    auto addq = [&](int f, int d, int s, int r, double v) {
      int o[3] = {0, 0, 0};
      o[d] += s;
      o[A] += r;
      unsafeAtomicAdd(sf[f] + pq(k + o[2]) + (o[1] + 1) * QX + (o[0] + 1) + lq, v);
    };
    face_vjp<A, VAR, VOF>(g, P, M, AV, p, F, dt, w, addu, addq);
  };
  auto out = [&](double* base, double* s, int x, int y, int z) {
    const double v = *s;
    if (v == 0.0) return;
    *s = 0.0;
    unsafeAtomicAdd(base + idx(g, W(g, 0, x), W(g, 1, y), W(g, 2, z)), v);
  };
  auto flush_u = [&](int z) {
    for (int e = t; e < 3 * PL; e += 768) {
      const int c = e / PL, r = e - c * PL;
      out(c == 0 ? U.ub[0] : (c == 1 ? U.ub[1] : U.ub[2]), su[c] + pu(z) + r, x0 - 2 + r % PX, y0 - 2 + r / PX, z);
    }
  };
  auto flush_q = [&](int z) {
    for (int e = t; e < 5 * QL; e += 768) {
      const int f = e / QL, r = e - f * QL;
      double* b = f == 0 ? AV.Fb[0] : (f == 1 ? AV.Fb[1] : (f == 2 ? AV.Fb[2] : (f == 3 ? AV.anp1 : AV.an)));
      out(b, sf[f] + pq(z) + r, x0 - 1 + r % QX, y0 - 1 + r / QX, z);
    }
  };
  for (int k = z0; k <= z1; k++) {
    __syncthreads();
    if (a == 0) face(std::integral_constant<int, 0>{}, k);
    else if (a == 1) face(std::integral_constant<int, 1>{}, k);
    else face(std::integral_constant<int, 2>{}, k);
    __syncthreads();
    flush_u(k - 2);
    if constexpr (VOF) flush_q(k - 1);
  }
  for (int z = z1 - 1; z <= z1 + 2; z++) flush_u(z);
  if constexpr (VOF) {
    flush_q(z1);
    flush_q(z1 + 1);
  }
}

// out_c = pin_c + s * sum over the interior faces f of cell c of +-beta_f ub_f / h
// (s dt D_i(beta ub)); cells natural, beta == nullptr: beta0
__global__ __launch_bounds__(256) void k_adj_div(Geo g, BetaF bf, const double* __restrict__ ub0,
                                                 const double* __restrict__ ub1, const double* __restrict__ ub2,
                                                 const double* __restrict__ pin, double* __restrict__ out, double s) {
  ROW_SETUP
  const double* ub[3] = {ub0, ub1, ub2};
  for (int i = 1 + lane; i <= g.n[0]; i += 64) {
    const int q[3] = {i, j, k};
    double acc = 0.0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
      int qp[3] = {i, j, k};
      qp[d] = W(g, d, q[d] + 1);
      const size_t fp = idx(g, qp[0], qp[1], qp[2]), fm = idx(g, i, j, k);
      // a face is interior unless it is a wall face of a wall direction
      const bool inp = g.per[d] || q[d] + 1 <= g.n[d];
      const bool inm = g.per[d] || q[d] >= 2;
      const double bp = bf.b[0] ? bf.b[d][fp] : g.beta0, bm = bf.b[0] ? bf.b[d][fm] : g.beta0;
      double t = 0.0;
      if (inp) t += bp * ub[d][fp];
      if (inm) t -= bm * ub[d][fm];
      acc += t * g.inv_d[d];
    }
    out[rb + i] = pin[rb + i] + s * acc;
  }
}

// ub*_f = ub'_f + (1/dt) (bb_i - bb_(i-1)) / h on interior faces of axis A;
// un_f = ub'_f on wall faces (u^{n+1} keeps u^n there), 0 elsewhere
template <int A>
__global__ __launch_bounds__(256) void k_adj_ustar(Geo g, const double* __restrict__ ubn,
                                                   const double* __restrict__ bb, double* __restrict__ ubs,
                                                   double* __restrict__ un, double inv_dt) {
  const int i = (int)(blockIdx.x * 64 + threadIdx.x);
  const int j = (int)(blockIdx.y * 4 + threadIdx.y);
  const int k = (int)blockIdx.z;
  if (i > g.n[0] + 1 || j > g.n[1] + 1 || k > g.n[2] + 1) return;
  const I3 q = mk(i, j, k);
  const size_t id = IX(g, q);
  int hi[3] = {g.n[0], g.n[1], g.n[2]};
  if (!g.per[A]) hi[A] += 1;
  bool inside = true;
#pragma unroll
  for (int d = 0; d < 3; d++)
    if (q.v[d] < 1 || q.v[d] > hi[d]) inside = false;
  if (!inside) {
    ubs[id] = 0.0;
    un[id] = 0.0;
    return;
  }
  const int fa = q.v[A];
  const bool wall = !g.per[A] && (fa == 1 || fa == g.n[A] + 1);
  if (wall) {
    ubs[id] = 0.0;
    un[id] = ubn[id];
  } else {
    const size_t cm = IX(g, wr(g, sh(q, A, -1)));
    ubs[id] = ubn[id] + inv_dt * ((bb[id] - bb[cm]) * g.inv_d[A]);
    un[id] = 0.0;
  }
}

// canonical row sums of a natural-layout cell field (part0 <- row sums)
__global__ __launch_bounds__(256) void k_rowsum_nat(Geo g, const double* __restrict__ x, double* __restrict__ part0) {
  ROW_SETUP
  double acc = 0.0;
  for (int i = 1 + lane; i <= g.n[0]; i += 64) acc += x[rb + i];
  acc = wave_tree_sum(acc);
  if (lane == 0) part0[row] = acc;
}

// planes per block: at least VJP_BLOCKS blocks, two for each CU in turn (one fits its
// registers), as long as a block has four planes to share its edges
constexpr unsigned VJP_BLOCKS = 512;
template <bool VAR, bool VOF>
void predict_vjp(const Geo& g, const Props& P, const Vel& V, const VofF& M, const double* p, double* const wbar[3],
                 const Acc& U, const AccV& AV, double dt, hipStream_t st) {
  const unsigned bx = (unsigned)((g.n[0] + VX - 1) / VX), by = (unsigned)((g.n[1] + VY - 1) / VY);
  int kc = 32;
  while (kc > 4 && bx * by * (unsigned)((g.n[2] + kc - 1) / kc) < VJP_BLOCKS) kc /= 2;
  Vel wb;
  for (int d = 0; d < 3; d++) wb.c[d] = wbar[d];
  hipLaunchKernelGGL((k_predict_vjp<VAR, VOF>), dim3(bx, by, (unsigned)((g.n[2] + kc - 1) / kc)), dim3(768), 0,
                     st, g, P, V, M, p, wb, U, AV, dt, kc);
}

}  // namespace

void launch_predict_vjp(const Geo& g, const Props* P, const Vel& V, double* const wbar[3], double* ub[3], double dt,
                        hipStream_t st) {
  Acc U;
  for (int d = 0; d < 3; d++) U.ub[d] = ub[d];
  const VofF M0{};
  const AccV AV0{};
  if (P) predict_vjp<true, false>(g, *P, V, M0, nullptr, wbar, U, AV0, dt, st);
  else predict_vjp<false, false>(g, Props{}, V, M0, nullptr, wbar, U, AV0, dt, st);
}

void launch_predict_vjp_vof(const Geo& g, const Props& P, const Vel& V, const VofF& M, const double* p,
                            double* const wbar[3], double* ub[3], double* const Fb[3], double* anp1, double* an,
                            double drho, double dmu, double dt, hipStream_t st) {
  Acc U;
  AccV AV;
  for (int d = 0; d < 3; d++) {
    U.ub[d] = ub[d];
    AV.Fb[d] = Fb[d];
  }
  AV.anp1 = anp1;
  AV.an = an;
  AV.drho = drho;
  AV.dmu = dmu;
  predict_vjp<true, true>(g, P, V, M, p, wbar, U, AV, dt, st);
}

void launch_adj_div(const Geo& g, const BetaF* bf, double* const ub[3], const double* pin, double* out, double s,
                    hipStream_t st) {
  dim3 grid((unsigned)((g.n[1] * g.n[2] + 3) / 4));
  hipLaunchKernelGGL(k_adj_div, grid, dim3(256), 0, st, g, bf ? *bf : BetaF{}, ub[0], ub[1], ub[2], pin, out, s);
}

void launch_adj_ustar(const Geo& g, double* const ubn[3], const double* bb, double* ubs[3], double* un[3],
                      double inv_dt, hipStream_t st) {
  dim3 grid((unsigned)((g.n[0] + 2 + 63) / 64), (unsigned)((g.n[1] + 2 + 3) / 4), (unsigned)(g.n[2] + 2));
  hipLaunchKernelGGL(k_adj_ustar<0>, grid, CELLB_A, 0, st, g, ubn[0], bb, ubs[0], un[0], inv_dt);
  hipLaunchKernelGGL(k_adj_ustar<1>, grid, CELLB_A, 0, st, g, ubn[1], bb, ubs[1], un[1], inv_dt);
  hipLaunchKernelGGL(k_adj_ustar<2>, grid, CELLB_A, 0, st, g, ubn[2], bb, ubs[2], un[2], inv_dt);
}

void launch_rowsum_nat(const Geo& g, const double* x, double* p0, hipStream_t st) {
  dim3 grid((unsigned)((g.n[1] * g.n[2] + 3) / 4));
  hipLaunchKernelGGL(k_rowsum_nat, grid, dim3(256), 0, st, g, x, p0);
}

}  // namespace smac
