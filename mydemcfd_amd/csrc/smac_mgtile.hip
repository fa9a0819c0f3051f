// smac_mgtile.hip -- a multigrid level's whole half of the V-cycle in one
// launch, for levels small enough that launches bound them.
//
// k_mg_down: the four half sweeps of V(2,.) from zero, the residual and its
// restriction; k_mg_up: the prolongation and the four half sweeps of V(.,2).
// A block owns an 8 x 8 x 8 tile of the level and holds it with a halo in LDS,
// the two colours in arrays of their own. It repeats its neighbours' work in
// the halo, each half sweep on a region one cell smaller (5 cells down, 4 up),
// so the sweeps need barriers only, no launch between them. Every cell is
// computed with the operations of the row kernels (smac_mg.hip) in their order,
// from the same operands, so the results are theirs bit for bit.
//
// What bounds it: on the levels it takes, latency -- the launch, one round of
// loads, six or seven LDS phases: 8 us down and 8 us up where six row kernels
// each took 3.4 to 4.5 us plus the gap between them. Straight code over more
// cells per thread is slower (512 threads with twelve cells each: 20 and 17 us;
// three cells per colour and division-heavy indexing: 12 and 11 us), since a
// block's instructions are fetched once and run once. The halo costs 5 to 11
// times the tile's cells in LDS work, which is why large levels keep the row
// kernels (mg_tile_applies).
#include "smac_internal.hpp"

namespace smac {

namespace {

constexpr int TL = 8;  // tile edge

__device__ __forceinline__ size_t trow(const Lv& L, int j, int k) {
  return ((size_t)k * (size_t)L.py + (size_t)j) * (size_t)L.px;
}
// the cell's image in 1..n of a periodic axis: the box of a tile reaches from
// -4 to n + 12 at most, so on the smallest levels (4 cells; 2 coarse ones) two
// periods below and three above
__device__ __forceinline__ int twrap(int i, int n) {
#pragma unroll
  for (int u = 0; u < 2; u++) i += i < 1 ? n : 0;
#pragma unroll
  for (int u = 0; u < 3; u++) i -= i > n ? n : 0;
  return i;
}

// the row kernels' division: IEEE, or (RCP) the FP32 reciprocal where the
// level's rows take the two- or four-rows-per-wave smoother
template <bool RCP>
__device__ __forceinline__ float t_div(float a, float b) {
  return RCP ? a * __builtin_amdgcn_rcpf(b) : a / b;
}
template <bool RCP>
__device__ __forceinline__ double t_div(double a, double b) { return a / b; }

template <typename C>
struct TCoef {
  C a[6];
  C diag;
};

// coefficients of the cell (i, j, k) in 1..n: level_coef of the row kernels.
// Uniform levels: `in` holds the coefficients of a cell off every wall.
template <typename C>
__device__ __forceinline__ TCoef<C> tcast(const Coef& c) {
  TCoef<C> r;
#pragma unroll
  for (int m = 0; m < 6; m++) r.a[m] = (C)c.a[m];
  r.diag = (C)c.diag;
  return r;
}
template <typename C>
__device__ __forceinline__ TCoef<C> tcoef_var(const Lv& L, int i, int j, int k) {
  Coef c;
  const int q[3] = {i, j, k};
  const unsigned om = ((unsigned)k * (unsigned)L.py + (unsigned)j) * (unsigned)L.px + (unsigned)i;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    int qp[3] = {i, j, k};
    qp[d] = L.per[d] ? wrapi(q[d] + 1, L.n[d]) : q[d] + 1;
    const unsigned op = ((unsigned)qp[2] * (unsigned)L.py + (unsigned)qp[1]) * (unsigned)L.px + (unsigned)qp[0];
    if constexpr (sizeof(C) == 4) {
      c.a[2 * d] = (double)L.bs[d][op] * L.inv_d2[d];
      c.a[2 * d + 1] = (double)L.bs[d][om] * L.inv_d2[d];
    } else {
      c.a[2 * d] = L.b[d][op] * L.inv_d2[d];
      c.a[2 * d + 1] = L.b[d][om] * L.inv_d2[d];
    }
  }
  c.diag = c.a[0] + c.a[1] + c.a[2] + c.a[3] + c.a[4] + c.a[5];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    if (wall_face(L.per[d], q[d] + 1, L.n[d])) c.a[2 * d] = 0.;
    if (wall_face(L.per[d], q[d], L.n[d])) c.a[2 * d + 1] = 0.;
  }
  return tcast<C>(c);
}

// The coefficients of the cells i0 (odd) and i0 + 1 of a row, their faces read as
// pairs; a load per face and cell (tcoef_var) has its lanes two cells apart. Down and
// up on 64x32x32 FP32 9.8 and 7.4 us, with tcoef_var 11.9 and 8.7; on 48x24x40 FP64
// 13.0 and 8.2, with it 14.4 and 8.9
template <typename C>
struct alignas(2 * sizeof(C)) Pair {
  C v[2];
};
template <typename C>
__device__ __forceinline__ void tcoef_pair(const Lv& L, int i0, int j, int k, TCoef<C> out[2]) {
  const int jp = L.per[1] ? wrapi(j + 1, L.n[1]) : j + 1, kp = L.per[2] ? wrapi(k + 1, L.n[2]) : k + 1;
  const unsigned r0 = ((unsigned)k * (unsigned)L.py + (unsigned)j) * (unsigned)L.px;
  const unsigned ry = ((unsigned)k * (unsigned)L.py + (unsigned)jp) * (unsigned)L.px;
  const unsigned rz = ((unsigned)kp * (unsigned)L.py + (unsigned)j) * (unsigned)L.px;
  const C* b[3];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    if constexpr (sizeof(C) == 4) b[d] = L.bs[d];
    else b[d] = L.b[d];
  }
  auto ld = [&](const C* p, unsigned at) { return *reinterpret_cast<const Pair<C>*>(p + at); };
  const Pair<C> x = ld(b[0], r0 + (unsigned)i0);
  const C x2 = b[0][r0 + (unsigned)(L.per[0] ? wrapi(i0 + 2, L.n[0]) : i0 + 2)];
  const Pair<C> ym = ld(b[1], r0 + (unsigned)i0), yp = ld(b[1], ry + (unsigned)i0);
  const Pair<C> zm = ld(b[2], r0 + (unsigned)i0), zp = ld(b[2], rz + (unsigned)i0);
#pragma unroll
  for (int t = 0; t < 2; t++) {
    Coef c;
    c.a[0] = (double)(t ? x2 : x.v[1]) * L.inv_d2[0];
    c.a[1] = (double)x.v[t] * L.inv_d2[0];
    c.a[2] = (double)yp.v[t] * L.inv_d2[1];
    c.a[3] = (double)ym.v[t] * L.inv_d2[1];
    c.a[4] = (double)zp.v[t] * L.inv_d2[2];
    c.a[5] = (double)zm.v[t] * L.inv_d2[2];
    c.diag = c.a[0] + c.a[1] + c.a[2] + c.a[3] + c.a[4] + c.a[5];
    const int q[3] = {i0 + t, j, k};
#pragma unroll
    for (int d = 0; d < 3; d++) {
      if (wall_face(L.per[d], q[d] + 1, L.n[d])) c.a[2 * d] = 0.;
      if (wall_face(L.per[d], q[d], L.n[d])) c.a[2 * d + 1] = 0.;
    }
    out[t] = tcast<C>(c);
  }
}

// A block's box: the tile with a halo of 4, 16 cells per edge from o - 4, and
// in LDS one more cell around it (lx, ly, lz = -1..16). A colour's values lie in
// [z][y][pair]: pair (lx + 2) >> 1 of 10 holds one cell of each colour. Thread
// t owns the pair h = t & 7 (lx = 2h, 2h + 1) of row ly = (t >> 3) & 15 on the
// planes lz = t >> 7 and lz + 8: two cells of each colour, a wave on one plane.
constexpr int HB = 4, BW = TL + 2 * HB;       // halo, box edge
constexpr int PY = BW / 2 + 2, PZ = PY * (BW + 2), PN = PZ * (BW + 2);
constexpr int TT = (BW / 2) * BW * (BW / 2);  // 1024 threads
constexpr int NO = 15;                        // distance of a cell that is not there
__device__ __forceinline__ int bidx(int lx, int ly, int lz) {
  return (lz + 1) * PZ + (ly + 1) * PY + ((lx + 2) >> 1);
}
// cells outside the tile along one axis
__device__ __forceinline__ int bdist(int l) { return max(max(HB - l, l - (HB + TL - 1)), 0); }

// the level's cell at box coordinate l of axis d: in 1..n (periodic images
// wrapped), or 0 where there is none
__device__ __forceinline__ int bcell(const Lv& L, int o, int d, int l) {
  const int v = o - HB + l;
  if (L.per[d]) return twrap(v, L.n[d]);
  return v >= 1 && v <= L.n[d] ? v : 0;
}

struct Own {
  int ly, lz, s[2], i[2], j, k[2];  // s, i by colour; k by plane
  int dxy[2];                       // distance in the plane by colour
  unsigned at[2][2];                // [colour][plane] offset in the level's arrays
  bool in[2];                       // in the tile's rows and the level by colour
  __device__ __forceinline__ void init(const Lv& L, const int o[3]) {
    const int t = (int)threadIdx.x, h = t & 7;
    ly = (t >> 3) & (BW - 1);
    lz = __builtin_amdgcn_readfirstlane(t >> 7);
    const int par = (o[0] + o[1] + o[2] + ly + lz) & 1;  // the box starts at o - 4
    j = bcell(L, o[1], 1, ly);
    k[0] = bcell(L, o[2], 2, lz);
    k[1] = bcell(L, o[2], 2, lz + BW / 2);
#pragma unroll
    for (int c = 0; c < 2; c++) {
      s[c] = (par + c) & 1;
      const int lx = 2 * h + s[c];
      i[c] = bcell(L, o[0], 0, lx);
      dxy[c] = max(bdist(lx), bdist(ly));
      in[c] = dxy[c] == 0 && o[0] - HB + lx <= L.n[0] && o[1] - HB + ly <= L.n[1];
      if (i[c] == 0 || j == 0) dxy[c] = NO;
#pragma unroll
      for (int m = 0; m < 2; m++)
        at[c][m] = ((unsigned)k[m] * (unsigned)L.py + (unsigned)j) * (unsigned)L.px + (unsigned)spos(i[c], L.n[0]);
    }
  }
  __device__ __forceinline__ int z(int m) const { return lz + (BW / 2) * m; }
  // does the cell lie within D cells of the tile?
  __device__ __forceinline__ bool on(int c, int m, int D) const {
    return bdist(z(m)) <= D && k[m] != 0 && dxy[c] <= D;
  }
  // a cell of the tile and the level, not an image
  __device__ __forceinline__ bool own(const Lv& L, const int o[3], int c, int m) const {
    return bdist(z(m)) == 0 && o[2] - HB + z(m) <= L.n[2] && in[c];
  }
  __device__ __forceinline__ int p(int m) const { return (z(m) + 1) * PZ + (ly + 1) * PY + ((int)threadIdx.x & 7) + 1; }
};

// The coefficients of the cells. Variable levels read a cell's once, ahead of
// the first barrier, and keep them in registers. Uniform levels: one set for
// all cells of a block that reaches no wall.
template <typename C, bool VB>
struct Coefs {
  TCoef<C> inner;
  double A[3];
  bool wall;
  __device__ __forceinline__ void init(const Lv& L, const int o[3]) {
    if constexpr (!VB) {
      inner = tcast<C>(coef_uniform(L.n, L.per, L.inv_d2, L.beta0, 2, 2, 2));
      wall = false;
#pragma unroll
      for (int d = 0; d < 3; d++) {
        A[d] = L.beta0 * L.inv_d2[d];
        wall = wall || (!L.per[d] && (o[d] - HB - 1 <= 1 || o[d] + TL + HB >= L.n[d]));
      }
    }
  }
  // of cell (i, j, k); `kept`: a variable level's, read before
  __device__ __forceinline__ TCoef<C> at(const Lv& L, int i, int j, int k, const TCoef<C>& kept) const {
    if constexpr (VB) return kept;
    if (!wall) return inner;
    Coef f;
    const int q[3] = {i, j, k};
#pragma unroll
    for (int d = 0; d < 3; d++) {
      f.a[2 * d] = wall_face(L.per[d], q[d] + 1, L.n[d]) ? 0.0 : A[d];
      f.a[2 * d + 1] = wall_face(L.per[d], q[d], L.n[d]) ? 0.0 : A[d];
    }
    f.diag = f.a[0] + f.a[1] + f.a[2] + f.a[3] + f.a[4] + f.a[5];
    return tcast<C>(f);
  }
};

// S = sum of a_nb e_nb in the order xp, xm, yp, ym, zp, zm: the other colour's
// values around pair p, `mate` the one in the pair itself
template <typename C>
__device__ __forceinline__ C nbsum(const TCoef<C>& a, int p, int s, C mate, const C* O) {
  const C nx = O[p + (s ? 1 : -1)];
  return a.a[0] * (s ? nx : mate) + a.a[1] * (s ? mate : nx) + a.a[2] * O[p + PY] + a.a[3] * O[p - PY] +
         a.a[4] * O[p + PZ] + a.a[5] * O[p - PZ];
}

// One half sweep of colour c on the region of D cells around the tile
template <typename T, bool RCP, bool VB, typename C>
__device__ __forceinline__ void half_sweep(const Lv& L, const Coefs<C, VB>& K, const Own& P, int c, int D, C (&e)[2][2],
                                           const C (&f)[2][2], const TCoef<C> (&k)[2][VB ? 2 : 1], C (*E)[PN]) {
#pragma unroll
  for (int m = 0; m < 2; m++)
    if (P.on(c, m, D)) {
      const TCoef<C> a = K.at(L, P.i[c], P.j, P.k[m], k[c][VB ? m : 0]);
      const C S = nbsum<C>(a, P.p(m), P.s[c], e[1 - c][m], E[1 - c]);
      e[c][m] = (C)stored_value<T>((double)t_div<RCP>(f[c][m] + S, a.diag));
      E[c][P.p(m)] = e[c][m];
    }
  __syncthreads();
}

// restriction weights of coarse index I: taps 2I-2 .. 2I+1 (at a wall the
// mirrored weight folds onto the boundary cell, the outer tap weighs 0)
template <typename C>
__device__ __forceinline__ void rw4(int per, int nc, int I, C w[4]) {
  const bool lo = !per && I == 1, hi = !per && I == nc;
  w[0] = lo ? (C)0 : (C)0.25;
  w[1] = lo ? (C)1 : (C)0.75;
  w[2] = hi ? (C)1 : (C)0.75;
  w[3] = hi ? (C)0 : (C)0.25;
}

// Pre-smoothing (red, black, red, black) from zero, residual on the red cells
// (it vanishes on the black ones) and restriction: ep <- e on the tile, fc <-
// the tile's coarse cells. The first half sweep, f / diag, covers the box and
// the red cells one further out (868 of them, one per thread).
template <typename T, bool VB, bool RCP>
__global__ __launch_bounds__(TT) void k_mg_down(Lv L, Lv Cl, const T* __restrict__ f, T* __restrict__ ep,
                                                T* __restrict__ fc) {
  using C = typename St<T>::C;
  constexpr int RW = TL + 2, NCT = TL / 2;  // residual box, coarse tile
  __shared__ C E[2][PN];
  __shared__ C res[RW * RW * RW];
  __shared__ C ty[RW * NCT * NCT];
  const int t = (int)threadIdx.x;
  const int o[3] = {1 + TL * (int)blockIdx.x, 1 + TL * (int)blockIdx.y, 1 + TL * (int)blockIdx.z};
  Own P;
  P.init(L, o);
  Coefs<C, VB> K;
  K.init(L, o);
  C e[2][2], fv[2][2];
  TCoef<C> k[2][VB ? 2 : 1];
#pragma unroll
  for (int c = 0; c < 2; c++)
#pragma unroll
    for (int m = 0; m < 2; m++) fv[c][m] = P.on(c, m, 4) ? St<T>::ld(f, P.at[c][m]) : (C)0;
  // the shell cell of this thread: two z faces of 18 x 18, two y faces of
  // 18 x 16, two x faces of 16 x 16, their red halves
  int sx = 0, sy = 0, sz = 0;
  bool shell = true;
  {
    const int c1 = (BW + 2) * (BW + 2) / 2, c2 = BW * (BW + 2) / 2, c3 = BW * BW / 2, HR = (BW + 2) / 2;
    const int rp = (o[0] + o[1] + o[2]) & 1;  // lx + ly + lz = rp (mod 2) on red cells
    int q = t;
    if (q < 2 * c1) {
      sz = q < c1 ? -1 : BW;
      q -= q < c1 ? 0 : c1;
      sy = q / HR - 1;
      sx = 2 * (q % HR) - 1;
      sx += (sx + sy + sz + rp) & 1;
    } else if ((q -= 2 * c1) < 2 * c2) {
      sy = q < c2 ? -1 : BW;
      q -= q < c2 ? 0 : c2;
      sz = q / HR;
      sx = 2 * (q % HR) - 1;
      sx += (sx + sy + sz + rp) & 1;
    } else if ((q -= 2 * c2) < 2 * c3) {
      sx = q < c3 ? -1 : BW;
      q -= q < c3 ? 0 : c3;
      sz = q / (BW / 2);
      sy = 2 * (q % (BW / 2));
      sy += (sx + sy + sz + rp) & 1;
    } else {
      shell = false;
    }
  }
  const int si = bcell(L, o[0], 0, sx), sj = bcell(L, o[1], 1, sy), sk = bcell(L, o[2], 2, sz);
  const bool sin = shell && si && sj && sk;
  C fs = (C)0;
  TCoef<C> ks;
  if (sin) {
    fs = St<T>::ld(f, ((unsigned)sk * (unsigned)L.py + (unsigned)sj) * (unsigned)L.px + (unsigned)spos(si, L.n[0]));
    if constexpr (VB) ks = tcoef_var<C>(L, si, sj, sk);
  }
  if constexpr (VB) {
#pragma unroll
    for (int m = 0; m < 2; m++)
      if (P.on(0, m, 4) || P.on(1, m, 4)) {
        TCoef<C> q[2];
        tcoef_pair<C>(L, P.s[0] ? P.i[1] : P.i[0], P.j, P.k[m], q);
#pragma unroll
        for (int c = 0; c < 2; c++) k[c][m] = P.s[c] ? q[1] : q[0];
      }
  }
  for (int q = t; q < RW * RW * RW; q += TT) res[q] = (C)0;
#pragma unroll
  for (int m = 0; m < 2; m++) {
    e[0][m] = (C)0;
    e[1][m] = (C)0;  // cells beyond a wall keep the ghost value 0
    if (P.on(0, m, 4))
      e[0][m] = (C)stored_value<T>(
          (double)t_div<RCP>(fv[0][m], K.at(L, P.i[0], P.j, P.k[m], k[0][VB ? m : 0]).diag));
    E[0][P.p(m)] = e[0][m];
    E[1][P.p(m)] = (C)0;
  }
  if (shell) {
    C v = (C)0;
    if (sin) v = (C)stored_value<T>((double)t_div<RCP>(fs, K.at(L, si, sj, sk, ks).diag));
    E[0][bidx(sx, sy, sz)] = v;
  }
  __syncthreads();
  half_sweep<T, RCP, VB, C>(L, K, P, 1, 4, e, fv, k, E);
  half_sweep<T, RCP, VB, C>(L, K, P, 0, 3, e, fv, k, E);
  half_sweep<T, RCP, VB, C>(L, K, P, 1, 2, e, fv, k, E);
#pragma unroll
  for (int m = 0; m < 2; m++) {
    if (P.on(0, m, 1)) {
      const TCoef<C> a = K.at(L, P.i[0], P.j, P.k[m], k[0][VB ? m : 0]);
      const C S = nbsum<C>(a, P.p(m), P.s[0], e[1][m], E[1]);
      const int lx = 2 * (t & 7) + P.s[0];
      res[((P.z(m) - HB + 1) * RW + (P.ly - HB + 1)) * RW + (lx - HB + 1)] = fv[0][m] - (a.diag * e[0][m] - S);
    }
#pragma unroll
    for (int c = 0; c < 2; c++)
      if (P.own(L, o, c, m)) St<T>::st(ep, P.at[c][m], e[c][m]);
  }
  __syncthreads();
  // coarse cells of the tile: along x and y for every fine plane, then along z
  const int c0[3] = {(o[0] + 1) >> 1, (o[1] + 1) >> 1, (o[2] + 1) >> 1};
  if (t < RW * NCT * NCT) {
    const int X = t % NCT, Y = (t / NCT) % NCT, z = t / (NCT * NCT);
    C wx[4], wy[4];
    rw4<C>(Cl.per[0], Cl.n[0], c0[0] + X, wx);
    rw4<C>(Cl.per[1], Cl.n[1], c0[1] + Y, wy);
    C a = (C)0;
#pragma unroll
    for (int b = 0; b < 4; b++) {
      const C* r = res + (z * RW + 2 * Y + b) * RW + 2 * X;
      C tx = (C)0;
#pragma unroll
      for (int q = 0; q < 4; q++) tx += wx[q] * r[q];
      a += wy[b] * tx;
    }
    ty[t] = a;
  }
  __syncthreads();
  if (t < NCT * NCT * NCT) {
    const int X = t % NCT, Y = (t / NCT) % NCT, Z = t / (NCT * NCT);
    const int I = c0[0] + X, J = c0[1] + Y, Kc = c0[2] + Z;
    if (I <= Cl.n[0] && J <= Cl.n[1] && Kc <= Cl.n[2]) {
      C wz[4];
      rw4<C>(Cl.per[2], Cl.n[2], Kc, wz);
      C tz = (C)0;
#pragma unroll
      for (int q = 0; q < 4; q++) tz += wz[q] * ty[((2 * Z + q) * NCT + Y) * NCT + X];
      St<T>::st(fc, trow(Cl, J, Kc) + spos(I, Cl.n[0]), (C)0.125 * tz);
    }
  }
}

// own and neighbour coarse cell of fine index i (pweights: 3/4 and 1/4; beyond
// a wall the own cell again), unwrapped
__device__ __forceinline__ void pcells(int per, int nc, int i, int& own, int& nb) {
  own = (i + 1) >> 1;
  nb = (i & 1) ? own - 1 : own + 1;
  if (!per && (nb < 1 || nb > nc)) nb = own;
}

// Prolongation of the coarse correction onto the red cells (the black ones are
// recomputed before they are read), then black, red, black, red: e <- the
// tile. ep: the level's e after the pre-smoothing (other blocks still read it,
// so e is another array).
template <typename T, bool VB, bool RCP>
__global__ __launch_bounds__(TT) void k_mg_up(Lv Cl, Lv L, const T* __restrict__ ec, const T* __restrict__ ep,
                                              const T* __restrict__ f, T* __restrict__ eo) {
  using C = typename St<T>::C;
  constexpr int CW = BW / 2 + 2;  // coarse box: the pairs' own cells and one more on each side
  __shared__ C E[2][PN];
  __shared__ C cs[CW * CW * CW];
  const int t = (int)threadIdx.x;
  const int o[3] = {1 + TL * (int)blockIdx.x, 1 + TL * (int)blockIdx.y, 1 + TL * (int)blockIdx.z};
  // coarse cell of LDS slot 0 along each axis: one below the own coarse cell
  // of the box's first fine cell o - 4
  const int b0[3] = {((o[0] - HB + 1) >> 1) - 1, ((o[1] - HB + 1) >> 1) - 1, ((o[2] - HB + 1) >> 1) - 1};
  if (t < CW * CW * CW) {
    const int q[3] = {b0[0] + t % CW, b0[1] + (t / CW) % CW, b0[2] + t / (CW * CW)};
    int w[3];
    bool ok = true;
#pragma unroll
    for (int d = 0; d < 3; d++) {
      w[d] = Cl.per[d] ? twrap(q[d], Cl.n[d]) : q[d];
      ok = ok && w[d] >= 1 && w[d] <= Cl.n[d];
    }
    cs[t] = ok ? St<T>::ld(ec, trow(Cl, w[1], w[2]) + spos(w[0], Cl.n[0])) : (C)0;
  }
  Own P;
  P.init(L, o);
  Coefs<C, VB> K;
  K.init(L, o);
  C e[2][2], fv[2][2];
  TCoef<C> k[2][VB ? 2 : 1];
#pragma unroll
  for (int m = 0; m < 2; m++) {
    e[0][m] = P.on(0, m, 4) ? St<T>::ld(ep, P.at[0][m]) : (C)0;
    e[1][m] = (C)0;
    fv[0][m] = P.on(0, m, 2) ? St<T>::ld(f, P.at[0][m]) : (C)0;
    fv[1][m] = P.on(1, m, 3) ? St<T>::ld(f, P.at[1][m]) : (C)0;
  }
  if constexpr (VB) {
#pragma unroll
    for (int m = 0; m < 2; m++) {
      if (P.on(0, m, 2) || P.on(1, m, 3)) {
        TCoef<C> q[2];
        tcoef_pair<C>(L, P.s[0] ? P.i[1] : P.i[0], P.j, P.k[m], q);
#pragma unroll
        for (int c = 0; c < 2; c++) k[c][m] = P.s[c] ? q[1] : q[0];
      }
    }
  }
  __syncthreads();
  int X0, X1, Y0, Y1;
  pcells(Cl.per[0], Cl.n[0], o[0] - HB + 2 * (t & 7) + P.s[0], X0, X1);
  pcells(Cl.per[1], Cl.n[1], o[1] - HB + P.ly, Y0, Y1);
#pragma unroll
  for (int m = 0; m < 2; m++) {
    if (P.on(0, m, 4)) {
      int Z0, Z1;
      pcells(Cl.per[2], Cl.n[2], o[2] - HB + P.z(m), Z0, Z1);
      C acc = (C)0;
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) {
          const C* r = cs + (((a ? Z1 : Z0) - b0[2]) * CW + ((b ? Y1 : Y0) - b0[1])) * CW - b0[0];
          const double wzy = (a ? 0.25 : 0.75) * (b ? 0.25 : 0.75);
          acc += (C)(wzy * 0.75) * r[X0];
          acc += (C)(wzy * 0.25) * r[X1];
        }
      e[0][m] = (C)stored_value<T>((double)(e[0][m] + acc));
    }
    E[0][P.p(m)] = e[0][m];
    E[1][P.p(m)] = (C)0;
  }
  __syncthreads();
  half_sweep<T, RCP, VB, C>(L, K, P, 1, 3, e, fv, k, E);
  half_sweep<T, RCP, VB, C>(L, K, P, 0, 2, e, fv, k, E);
  half_sweep<T, RCP, VB, C>(L, K, P, 1, 1, e, fv, k, E);
#pragma unroll
  for (int m = 0; m < 2; m++) {
    if (P.own(L, o, 0, m)) {
      const TCoef<C> a = K.at(L, P.i[0], P.j, P.k[m], k[0][VB ? m : 0]);
      St<T>::st(eo, P.at[0][m], t_div<RCP>(fv[0][m] + nbsum<C>(a, P.p(m), P.s[0], e[1][m], E[1]), a.diag));
    }
    if (P.own(L, o, 1, m)) St<T>::st(eo, P.at[1][m], e[1][m]);
  }
}

dim3 tile_grid(const Lv& L) {
  return dim3((unsigned)((L.n[0] + TL - 1) / TL), (unsigned)((L.n[1] + TL - 1) / TL),
              (unsigned)((L.n[2] + TL - 1) / TL));
}

}  // namespace

// An iteration of the PCG with the level's half V-cycles by the tiles against by the
// row kernels: uniform 32^3 BF16 51 us against 87, 64^3 BF16 80 against 94, FP32 76
// against 91, FP64 87 against 90, 128x64x64 FP32 109 against 106, FP64 130 against 111;
// variable 64x32x32 FP32 60 against 87, 128x64x32 FP32 88 against 94, BF16 92 against
// 94, 128x64x64 FP32 136 against 113; variable FP64 64x64x32 74 against 90, 96x48x40 99
// against 98, 128x64x32 98 against 96. Past the limits the halo's work outweighs the
// launches.
template <typename T>
bool mg_tile_applies(const Lv& L) {
  const size_t cells = (size_t)L.n[0] * L.n[1] * L.n[2];
  return cells <= (L.b[0] && sizeof(T) == 8 ? MG_TILE_CELLS / 2 : MG_TILE_CELLS);
}

#define SMAC_TILE_V(K, R, ...)                                                                  \
  do {                                                                                          \
    if (F.b[0]) hipLaunchKernelGGL((K<T, true, R>), tile_grid(F), dim3(TT), 0, st, __VA_ARGS__); \
    else hipLaunchKernelGGL((K<T, false, R>), tile_grid(F), dim3(TT), 0, st, __VA_ARGS__);       \
  } while (0)
#define SMAC_TILE(K, ...)                               \
  do {                                                  \
    if constexpr (sizeof(typename St<T>::C) == 4) {     \
      if (rcp) SMAC_TILE_V(K, true, __VA_ARGS__);       \
      else SMAC_TILE_V(K, false, __VA_ARGS__);          \
    } else {                                            \
      SMAC_TILE_V(K, false, __VA_ARGS__);               \
    }                                                   \
  } while (0)

template <typename T>
void launch_mg_down(const Lv& F, const Lv& C, const T* f, T* ep, T* fc, int rcp, hipStream_t st) {
  (void)rcp;
  SMAC_TILE(k_mg_down, F, C, f, ep, fc);
}
template <typename T>
void launch_mg_up(const Lv& C, const Lv& F, const T* ec, const T* ep, const T* f, T* e, int rcp, hipStream_t st) {
  (void)rcp;
  SMAC_TILE(k_mg_up, C, F, ec, ep, f, e);
}
#undef SMAC_TILE
#undef SMAC_TILE_V

#define SMAC_INST_TILE(T)                                                                                        \
  template bool mg_tile_applies<T>(const Lv&);                                                                   \
  template void launch_mg_down<T>(const Lv&, const Lv&, const T*, T*, T*, int, hipStream_t);                     \
  template void launch_mg_up<T>(const Lv&, const Lv&, const T*, const T*, const T*, T*, int, hipStream_t);
SMAC_INST_TILE(double)
SMAC_INST_TILE(float)
SMAC_INST_TILE(bf16s)

}  // namespace smac
