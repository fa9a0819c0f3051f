// smac_predict.hpp -- one face of the SMAC predictor as device templates, shared
// by the forward kernels (smac_kernels.hip) and the adjoint (smac_adjoint.hip,
// which differentiates the same terms).
#pragma once

#include "smac_internal.hpp"

namespace smac {

// one side of the convective flux along E, MUSCL-minmod on the five values
// c[-2..2] = u_A at q + s e_E (upwind side from the sign of m)
__device__ __forceinline__ double flux_plus(double m, const double c[5]) {
  // + face: up = q (c0) when m > 0, else q + e (c1)
  double dpv, dmv, uw;
  if (m > 0.) {
    dpv = c[3] - c[2];
    dmv = c[2] - c[1];
    uw = c[2];
  } else {
    dpv = c[4] - c[3];
    dmv = c[3] - c[2];
    uw = c[3];
  }
  double sl = minmod(dpv, dmv);
  int dir = sgn(m);
  return m * (uw + dir * 0.5 * sl);
}
__device__ __forceinline__ double flux_minus(double m, const double c[5]) {
  // - face: up = q - e (c-1) when m > 0, else q (c0)
  double dpv, dmv, uw;
  if (m > 0.) {
    dpv = c[2] - c[1];
    dmv = c[1] - c[0];
    uw = c[1];
  } else {
    dpv = c[3] - c[2];
    dmv = c[2] - c[1];
    uw = c[2];
  }
  double sl = minmod(dpv, dmv);
  int dir = sgn(m);
  return m * (uw + dir * 0.5 * sl);
}

// The value of a wall face of component a on side s, as get_face gives it: the
// array's (stored) or the wall's
__device__ __forceinline__ bool wall_stored(const Geo& g, int a, int s) {
  const int bt = g.btype[s];
  return bt == BC_OUTLET || (bt == BC_SLIP && a != 0);
}
__device__ __forceinline__ double wall_value(const Geo& g, int a, int s, double stored) {
  if (wall_stored(g, a, s)) return stored;
  return g.btype[s] == BC_INFLOW ? (1. - 0.0) * g.bv[s][a] : 0.;
}
// Component a beyond the wall on side s of a tangential axis, next to the value v
// (d_get_v{a}_{b}dir, CFD/G_BoundaryFunctions.h:100-367): v itself at a slip or
// outlet side, else mirrored about the wall velocity. That is there the mean of the
// two wall faces next to it, which both lie on the side, so the side's
__device__ __forceinline__ bool wall_even(const Geo& g, int s) {
  return g.btype[s] == BC_SLIP || g.btype[s] == BC_OUTLET;
}
__device__ __forceinline__ double wall_mirror(const Geo& g, int a, int s, double v) {
  return wall_even(g, s) ? v : 2.0 * g.bv[s][a] - v;
}

// The convective flux through the + and the - side on the five values c[-2..2],
// first-order where the upwind face is no interior one (flux_plus, flux_minus
// with that case of conv_term)
__device__ __forceinline__ double flux_plus_in(double m, const double c[5], bool in) {
  const bool own = m > 0.;
  const double uw = own ? c[2] : c[3];
  const double sl = minmod(own ? c[3] - c[2] : c[4] - c[3], own ? c[2] - c[1] : c[3] - c[2]);
  return m * (own || in ? uw + sgn(m) * 0.5 * sl : uw);
}
__device__ __forceinline__ double flux_minus_in(double m, const double c[5], bool in) {
  const bool own = !(m > 0.);
  const double uw = own ? c[2] : c[1];
  const double sl = minmod(own ? c[3] - c[2] : c[2] - c[1], own ? c[2] - c[1] : c[1] - c[0]);
  return m * (own || in ? uw + sgn(m) * 0.5 * sl : uw);
}

// The mass flux of a face
enum MassFlux {
  MF_RHO,  // rho0 u
  MF_VOF,  // rho0 u + (rho1 - rho0) F h/dt (the alpha flux of a transport)
  MF_EPS   // the two-way form (below)
};

// The velocities that u*_A of face q reads: component A along each axis, c[d][s+2]
// at q + s e_d, and component B on the four faces around the edge of axes A and B
// (q + e_B, q + e_B - e_A, q, q - e_A), all loaded before any branch. RIM: the
// stencil may reach walls, whose values the boundary getters' rules replace, or
// wrap; off[d][s+2] is the array offset of q + s e_d either way. inp, inm: is
// q +- e_d an interior face?
template <int A, bool RIM>
struct Face {
  I3 q;
  size_t id;
  long st[3], off[3][5];
  double c[3][5], wpp[3], wmp[3], wp0[3], wm0[3];
  bool inp[3], inm[3];
  __device__ __forceinline__ size_t at(int d, int s) const { return id + (size_t)off[d][s + 2]; }
  __device__ __forceinline__ size_t at2(int d, int s, int e, int t) const {
    return id + (size_t)(off[d][s + 2] + off[e][t + 2]);
  }
  __device__ __forceinline__ Face(const Geo& g, const Vel& V, I3 q_) : q(q_) {
    st[0] = 1;
    st[1] = (long)g.px;
    st[2] = (long)g.px * (long)g.py;
    id = IX(g, q);
    // beyond a wall the array's own entries, whose values are replaced
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
      for (int s = -2; s <= 2; s++) {
        long o = s;
        if (RIM) {
          if (g.per[d]) o = wrapi(q.v[d] + s, g.n[d]) - q.v[d];
          else if (q.v[d] + s < 0) o = -q.v[d];
        }
        off[d][s + 2] = o * st[d];
      }
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
      for (int s = -2; s <= 2; s++) c[d][s + 2] = V.c[A][at(d, s)];
#pragma unroll
    for (int B = 0; B < 3; B++) {
      inp[B] = inm[B] = true;
      if (B == A) continue;
      const double* w = V.c[B];
      wpp[B] = w[at(B, 1)];
      wmp[B] = w[at2(B, 1, A, -1)];
      wp0[B] = w[id];
      wm0[B] = w[at(A, -1)];
    }
    if constexpr (RIM) {
#pragma unroll
      for (int d = 0; d < 3; d++) {
        if (g.per[d]) continue;
        const int x = q.v[d], n = g.n[d];
        inp[d] = x != n;
        if (d == A) {
          // own axis: faces 1 and n + 1 are the walls (the ghosts beyond are not used)
          if (x == 2) c[d][1] = wall_value(g, A, 2 * d, c[d][1]);
          if (x == 3) c[d][0] = wall_value(g, A, 2 * d, c[d][0]);
          if (x == n) c[d][3] = wall_value(g, A, 2 * d + 1, c[d][3]);
          if (x == n - 1) c[d][4] = wall_value(g, A, 2 * d + 1, c[d][4]);
          inm[d] = x != 2;
        } else {
          if (x == 1) c[d][1] = wall_mirror(g, A, 2 * d, c[d][2]);
          if (x == 2) c[d][0] = wall_mirror(g, A, 2 * d, c[d][1]);
          if (x == n) c[d][3] = wall_mirror(g, A, 2 * d + 1, c[d][2]);
          if (x == n - 1) c[d][4] = wall_mirror(g, A, 2 * d + 1, c[d][3]);
          inm[d] = x != 1;
          // component d on its own wall faces
          if (x == 1) {
            wp0[d] = wall_value(g, d, 2 * d, wp0[d]);
            wm0[d] = wall_value(g, d, 2 * d, wm0[d]);
          }
          if (x == n) {
            wpp[d] = wall_value(g, d, 2 * d + 1, wpp[d]);
            wmp[d] = wall_value(g, d, 2 * d + 1, wmp[d]);
          }
        }
      }
    }
  }
  // mass flux of axis e at q + se e_e + sa e_A with face value v
  template <MassFlux MF>
  __device__ __forceinline__ double mflux(const Geo& g, const VofF& M, int e, int se, int sa, double v) const {
    const double rho0 = g.rho0;
    if constexpr (MF == MF_RHO) {
      return rho0 * v;
    } else {
      const size_t r = e == A ? at(A, se) : at2(e, se, A, sa);
      if constexpr (MF == MF_VOF) {
        return rho0 * v + M.drho * (M.F[e][r] * M.hbydt[e]);
      } else {
        const size_t raw = id + (size_t)(se * st[e]) + (e == A ? 0 : (size_t)(sa * st[A]));
        const int m = q.v[e] + se;  // 0 (a flux of 0) on a periodic axis: no cell before it
        const double hi = M.eps_half[raw], lo = M.eps_half[raw - (RIM && m == 0 ? 0 : (size_t)st[e])];
        double ef = 0.5 * (lo + hi);
        if (RIM && m == 1) ef = hi;
        if (RIM && m == g.n[e] + 1) ef = lo;
        const double f = ef * v;
        double mf = rho0 * f;
        if (M.F[e]) mf = rho0 * f + M.drho * (M.F[e][r] * M.hbydt[e]);
        if (RIM && (m < 1 || m > g.n[e] + 1)) mf = 0.0;
        return mf;
      }
    }
  }
  // the mass fluxes mp[e], mm[e] that carry component A through the + and - sides
  template <MassFlux MF>
  __device__ __forceinline__ void mass(const Geo& g, const VofF& M, double mp[3], double mm[3]) const {
    const double f0 = mflux<MF>(g, M, A, 0, 0, c[A][2]), fp = mflux<MF>(g, M, A, 1, 0, c[A][3]),
                 fm = mflux<MF>(g, M, A, -1, 0, c[A][1]);
    mp[A] = 0.5 * (f0 + fp);
    mm[A] = 0.5 * (fm + f0);
#pragma unroll
    for (int B = 0; B < 3; B++) {
      if (B == A) continue;
      mp[B] = 0.5 * (mflux<MF>(g, M, B, 1, -1, wmp[B]) + mflux<MF>(g, M, B, 1, 0, wpp[B]));
      mm[B] = 0.5 * (mflux<MF>(g, M, B, 0, 0, wp0[B]) + mflux<MF>(g, M, B, 0, -1, wm0[B]));
    }
  }
  // edge viscosities of the cross stresses with axis B
  template <bool VAR>
  __device__ __forceinline__ void mu_edge(const Geo& g, const Props& P, int B, double& mu_p, double& mu_m) const {
    mu_p = mu_m = 0.5 * (g.mu0 + g.mu0);
    if constexpr (VAR) {
      mu_p = 0.5 * (P.muf[B][at(B, 1)] + P.muf[B][at2(B, 1, A, -1)]);
      mu_m = 0.5 * (P.muf[B][id] + P.muf[B][at(A, -1)]);
    }
  }
  // rates of strain around the edges of axes A and B on the + and - side of B
  __device__ __forceinline__ double strain_p(const Geo& g, int B) const {
    return (wpp[B] - wmp[B]) * g.inv_d[A] + (c[B][3] - c[A][2]) * g.inv_d[B];
  }
  __device__ __forceinline__ double strain_m(const Geo& g, int B) const {
    return (wp0[B] - wm0[B]) * g.inv_d[A] + (c[A][2] - c[B][1]) * g.inv_d[B];
  }

  // One face of component A of k_get_vof_vstar_rhouu_consistent_{x,y,z}
  // (CFD/G_SMACSolver.cu:139-392, 441-662, 763-1003), the terms in the
  // reference's order; with MF_EPS of the two-way kernels (1538-2194): the stresses weighted
  // by the t^n volume fraction (cell values for the own-direction stress, the mean
  // of the four cells around the edge, summed in memory order, for the cross
  // stresses), the old pressure gradient by the face mean of eps^n, the mass flux
  // rho0 (eps_f u_f) + (rho1-rho0) F h/dt on the faces 1..N+1 of its axis and 0
  // outside them, eps_f the t^{n+1/2} volume fraction of the face -- the mean of its
  // two cells, the inner cell on faces 1 and N+1 (CFD/G_SMACSolver_VoF.cu:2472-2557,
  // 1954-1967) --, and u* = (beta/eps^{n+1}_f) (eps^n_f rho^n_f u + dt tmp + J/V) +
  // dt g with J the particles' momentum impulse on the face. Volume fractions are
  // read at the raw cell indices, ghosts included; the IBM solid fraction factor
  // (1 - 0) of the reference is 1.
  // The bracket: stresses, convection, old pressure gradient.
  template <bool VAR, MassFlux MF>
  __device__ __forceinline__ double bracket(const Geo& g, const Props& P, const VofF& M, const double* eo,
                                            const double* p, const double mp[3], const double mm[3]) const {
    constexpr bool TW = MF == MF_EPS;
    constexpr int B1 = A == 0 ? 1 : 0, B2 = A == 2 ? 1 : 2;
    const double v0 = c[A][2];
    const size_t rA = id - (size_t)st[A], cm = at(A, -1);
    double tmp;
    {
      const double mup = VAR ? P.mu[id] : g.mu0, mum = VAR ? P.mu[cm] : g.mu0;
      const double tau_p = mup * (c[A][3] - v0);
      const double tau_m = mum * (v0 - c[A][1]);
      if constexpr (TW) tmp = 2. * (eo[id] * tau_p - eo[rA] * tau_m) * g.inv_d2[A];
      else tmp = 2. * (tau_p - tau_m) * g.inv_d2[A];
    }
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const int B = e == 0 ? B1 : B2;
      double mu_p, mu_m;
      mu_edge<VAR>(g, P, B, mu_p, mu_m);
      const double t_p = mu_p * strain_p(g, B);
      const double t_m = mu_m * strain_m(g, B);
      if constexpr (TW) {
        const size_t sB = (size_t)st[B];
        double ep, em;
        if (B > A) {
          ep = 0.25 * (eo[rA] + eo[id] + eo[rA + sB] + eo[id + sB]);
          em = 0.25 * (eo[rA - sB] + eo[id - sB] + eo[rA] + eo[id]);
        } else {
          ep = 0.25 * (eo[rA] + eo[rA + sB] + eo[id] + eo[id + sB]);
          em = 0.25 * (eo[rA - sB] + eo[rA] + eo[id - sB] + eo[id]);
        }
        tmp += (ep * t_p - em * t_m) * g.inv_d[B];
      } else {
        tmp += (t_p - t_m) * g.inv_d[B];
      }
    }
#pragma unroll
    for (int e = 0; e < 3; e++) {
      const double Mp = RIM ? flux_plus_in(mp[e], c[e], inp[e]) : flux_plus(mp[e], c[e]);
      const double Mm = RIM ? flux_minus_in(mm[e], c[e], inm[e]) : flux_minus(mm[e], c[e]);
      tmp -= (Mp - Mm) * g.inv_d[e];
    }
    if constexpr (TW) tmp -= 0.5 * (eo[rA] + eo[id]) * (p[id] - p[cm]) * g.inv_d[A];
    else tmp -= (p[id] - p[cm]) * g.inv_d[A];
    return tmp;
  }
  template <bool VAR>
  __device__ __forceinline__ double beta(const Geo& g, const Props& P) const {
    return VAR ? P.beta[A][id] : g.beta0;
  }
  template <bool VAR>
  __device__ __forceinline__ double rho_old(const Geo& g, const Props& P) const {
    return VAR ? 0.5 * (P.rho_old[id] + P.rho_old[at(A, -1)]) : 0.5 * (g.rho0 + g.rho0);
  }
};

// u*_A of face q. VAR: properties from the arrays
template <int A, bool VAR, MassFlux MF, bool RIM>
__device__ __forceinline__ double face_ustar(const Geo& g, const Props& P, const Vel& V, const VofF& M, const EpsF& E,
                                             const double* __restrict__ p, I3 q, double dt) {
  const Face<A, RIM> F(g, V, q);
  double mp[3], mm[3];
  F.template mass<MF>(g, M, mp, mm);
  const double tmp = F.template bracket<VAR, MF>(g, P, M, E.eps_old, p, mp, mm);
  const double v0 = F.c[A][2], beta = F.template beta<VAR>(g, P), rho = F.template rho_old<VAR>(g, P);
  if constexpr (MF == MF_EPS) {
    const size_t id = F.id, rA = id - (size_t)F.st[A];
    const double eo_f = 0.5 * (E.eps_old[rA] + E.eps_old[id]);
    const double en_f = 0.5 * (E.eps[rA] + E.eps[id]);
    const double jd = E.imp[A] ? E.imp[A][id] * E.inv_vol : 0.0;
    const double inv_eps_rho = beta / en_f;
    return inv_eps_rho * (eo_f * rho * v0 + dt * tmp + jd) + dt * g.g[A];
  }
  return beta * (v0 * rho) + dt * (beta * tmp + g.g[A]);
}

}  // namespace smac
