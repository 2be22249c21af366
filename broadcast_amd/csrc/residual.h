// The residual (T = double) and its tangent (T = Dual<1>) in one kernel: state
// in, residu out, everything between in LDS.
//
// A workgroup takes 15 x 15 cells and the 16 x 16 faces of either direction
// around them.  Its 8 waves load the cells those faces read (16 + ORD of them a
// row), form their primitives, then the velocity gradients' dissipation sensor
// and the along-face sums of the compact viscous stencil, each once; then 4
// waves take the i-faces and 4 the j-faces, and the balance adds the fluxes up.
//
// What bounds it: FP64 instructions, about 900 a cell at order 5 (a third of
// what planes of primitives, gradients and fluxes between five kernels took: the
// Roe weights and the Ducros sensor once per cell, one logistic function and
// three divisions a face in the place of two tanh and seven, the square roots of
// the face's normal once, the viscous sums shared by the faces of a row) at two
// workgroups a CU (LDS, and 128 VGPRs).  A cell's primitives are formed 1.96
// times (441 loaded for 225 kept) and 14 % of the faces twice, which costs less
// than the 26 planes written and read between the passes.  16 x 16: 64 x 8 has
// the same halo and waste, and fills less of the chip on a small mesh.
//
// With the boundary conditions before it: residual 2048 x 1024 625 -> 192 us,
// 96 x 64 38.6 -> 18.7 us, order 7 on a 383 x 255 O-mesh 80 -> 44 us; tangent on
// a 509 x 381 O-mesh 93 -> 50 us.  The distance from an 80-bit evaluation is
// 0.79 to 0.96 of the former kernels' (2-norm; flat plate 96 x 64 and 131 x 67,
// O-mesh 28 x 12 and 128 x 90).
#pragma once
#include "bcs.h"
#include "faces.h"

namespace bca {

constexpr int TILE = 16;              // faces a side
constexpr int TILE_CELLS = TILE - 1;  // cells a side
constexpr int TILE_THREADS = 2 * TILE * TILE;
enum { Q_RO = 0, Q_RU, Q_RV, Q_RW, Q_RE, Q_U, Q_V, Q_W, Q_T, Q_P, Q_MU, Q_H, NQ };

// the scheme's coefficients; the off-centred Euler weights of the rows next to
// the wall on cell rows 1 .. NW
template <int ORD>
struct NearWall {
  static constexpr int RC = (ORD + 3) / 2;  // first row with the centred flux
  static constexpr int NW = ORD == 3 ? 2 : ORD == 5 ? 5 : ORD == 7 ? 9 : 11;
  double w[(RC - 2) * NW];  // rows 2 .. RC - 1
  constexpr NearWall() : w() {
    for (int row = 2; row < RC; ++row)
      for (int t = 0; t < NW; ++t) w[(row - 2) * NW + t] = off(row, t);
  }
  // centred Euler flux, k = 0 the innermost pair
  static constexpr double centred(int k) {
    if constexpr (ORD == 3) return k == 0 ? Coef3::c1 : Coef3::c2;
    else if constexpr (ORD == 5) return k == 0 ? Coef::c1 : k == 1 ? Coef::c2 : Coef::c3;
    else return CoefHi<ORD>::c(k);
  }
  // predictor, k = 0 the innermost pair; signs alternate outwards
  static constexpr double pred(int k) {
    if constexpr (ORD == 3) return k == 0 ? Coef3::d1 : Coef3::d2;
    else if constexpr (ORD == 5) return k == 0 ? Coef::d1 : k == 1 ? Coef::d2 : Coef::d3;
    else return CoefHi<ORD>::d(k);
  }
  static constexpr double grad(int k) {
    if constexpr (ORD == 3) return Coef3::b1;
    else if constexpr (ORD == 5) return k == 0 ? Coef::b1 : Coef::b2;
    else return CoefHi<ORD>::b(k);
  }
  static constexpr double off(int row, int t) {
    if constexpr (ORD == 3) return 0.5;  // nearbndfluxes3demi_5p.F
    else if constexpr (ORD == 5) {
      // the off-centred faces 3/2 and 5/2 (flux_num_dnc5.F90:164-196)
      constexpr double k3[5] = {12.0, 77.0, -43.0, 17.0, -3.0}, k5[5] = {-3.0, 27.0, 47.0, -13.0, 2.0};
      return (row == 2 ? k3[t] : k5[t]) / 60.0;
    } else return CoefHi<ORD>::w(row, t);
  }
};
template <int ORD>
__device__ const NearWall<ORD> near_wall{};

// the scheme's constants, formed once on the host
struct ResPhys {
  double gm1, cvm1, betas, s_suth, gr, sqgr, cpp, k2, k4;
};
__host__ inline ResPhys res_phys(const Phys& p) {
  ResPhys r;
  r.gm1 = p.gam - 1.0;
  r.cvm1 = 1.0 / p.cv;
  r.betas = p.muref * (p.tref + p.cs) / (sqrt(p.tref) * p.tref);
  r.s_suth = p.s_suth;
  r.gr = p.gam * p.rgaz;
  r.sqgr = sqrt(r.gr);
  r.cpp = p.cp / p.prandtl;
  r.k2 = p.k2;
  r.k4 = p.k4;
  return r;
}

// 0.5 (1 - tanh x) as the logistic function it is
__device__ inline double dswitch(double x) { return 1.0 / (1.0 + exp(2.0 * x)); }
template <int N> __device__ inline Dual<N> dswitch(const Dual<N>& x) {
  Dual<N> r(dswitch(x.v));
  const double g = -2.0 * r.v * (1.0 - r.v);
#pragma unroll
  for (int k = 0; k < N; ++k) r.d[k] = x.d[k] * g;
  return r;
}

// Where the residual goes: residu, and of a Dual residud too (either may be
// null there; ghosts untouched).
struct ResOut {
  double* res;
  double* resd;
};

template <class T, int ORD>
struct Tile {
  static constexpr int L = (ORD + 1) / 2, R = (ORD - 1) / 2, S = TILE + L + R, SS = S * S;
  static constexpr int A = TILE + 1;  // cells -1 .. 15, the two sides of every face
  // the along-face sums are kept where they leave two workgroups of double a
  // CU's LDS (and one of Dual)
  static constexpr bool SUMS = ORD == 5 || ORD == 7;
  static constexpr int NROWS = TILE + 4;
  static_assert(NQ * SS >= 10 * TILE * TILE, "the fluxes take the cells' place");
  T q[NQ * SS];
  T sr[A * A], c[A * A], duc[A * A], vd[A * A];  // sqrt(rho), speed of sound, Ducros sensor, 10 vol div
  T rows[2][4][SUMS ? NROWS * TILE : 1];         // -f(-2) + 9 f(-1) + 9 f(0) - f(1) along the faces, of u, v, w, T
  double wt[sizeof(NearWall<ORD>) / sizeof(double)];
};

// the metrics of one face: normal, and the raw terms of its contour
struct FaceMetric {
  double nx, ny, vf;
  double px[6], py[6];  // +1, -1 along; the two halves of the cross sides + and -
};
template <bool J>
__device__ inline FaceMetric face_metric(const Mesh& m, const Metric& g, int i, int j) {
  constexpr int D = J ? 1 : 0;
  FaceMetric f;
  const long n0 = nidx(m, i, j), si = 1, sj = m.ni + 1;
  const long along = J ? sj : si, cross = J ? si : sj;
  const long pd = (long)D * m.nnode, pc = (long)(1 - D) * m.nnode;
  f.nx = g.nx[n0 + pd], f.ny = g.ny[n0 + pd];
  f.vf = g.volf[cidx(m, i, j) + (long)D * m.ncell];
  const long o[6] = {n0 + along + pd, n0 - along + pd, n0 - along + cross + pc, n0 + cross + pc, n0 - along + pc, n0 + pc};
#pragma unroll
  for (int k = 0; k < 6; ++k) f.px[k] = g.nx[o[k]], f.py[k] = g.ny[o[k]];
  return f;
}

template <class T>
struct Flux {
  T h0, h1, h2, h3, h4;
};

// hn = Euler - dissipation - viscous of one face.  NEAR: a tile at the wall,
// whose rows differ (the wall face, the off-centred rows, the 2nd-order viscous
// flux of rows 1 and 2): weights by row, in the place of a variant a row.
template <class T, int ORD, bool J, bool NEAR>
__device__ inline Flux<T> tile_face(const Tile<T, ORD>& s, const ResPhys& ph, const FaceMetric& fm, int tx, int ty,
                                    int j) {
  using TL = Tile<T, ORD>;
  using C = NearWall<ORD>;
  constexpr int S = TL::S, SS = TL::SS, sa = J ? S : 1, sc = J ? 1 : S;
  const int b = (ty + TL::L) * S + tx + TL::L;
  auto Q = [&](int pl, int off) -> T { return s.q[pl * SS + b + off]; };
  if constexpr (NEAR && J) {
    if (j <= 1) {
      // adiabatic no-slip wall (fluxwall.F)
      const double nx = fm.nx, ny = fm.ny, vf = fm.vf;
      T pw = 1.125 * Q(Q_P, 0) - 0.125 * Q(Q_P, sa);
      T mmu = Q(Q_MU, 0), u = Q(Q_U, 0), v = Q(Q_V, 0), ww = Q(Q_W, 0);
      T ux = 2.0 * u * nx * vf, vx = 2.0 * v * nx * vf, wx = 2.0 * ww * nx * vf;
      T uy = 2.0 * u * ny * vf, vy = 2.0 * v * ny * vf, wy = 2.0 * ww * ny * vf;
      T sh = mmu * (uy + vx);
      Flux<T> h;
      h.h0 = T(0.0);
      h.h1 = pw * nx - (Coef::twothird * mmu * (2.0 * ux - vy) * nx + sh * ny);
      h.h2 = pw * ny - (sh * nx + Coef::twothird * mmu * (2.0 * vy - ux) * ny);
      h.h3 = -(mmu * wx * nx + mmu * wy * ny);
      h.h4 = T(0.0);
      return h;
    }
  }
  Flux<T> h;
  const double nx = fm.nx, ny = fm.ny;
  // ---- dissipation scalars: Roe-weighted spectral radius, eps2 and eps4
  T rspec, eps2(0.0), eps4;
  {
    const int r0 = (ty + 1) * TL::A + tx + 1, r1 = r0 - (J ? TL::A : 1);
    const double n2 = nx * nx + ny * ny;
    const T s0 = s.sr[r0], s1 = s.sr[r1];
    const T iw = 1.0 / (s0 + s1);
    const T un = (nx * (Q(Q_U, -sa) * s1 + Q(Q_U, 0) * s0) + ny * (Q(Q_V, -sa) * s1 + Q(Q_V, 0) * s0)) * iw;
    const T c2 = ph.gr * ((Q(Q_T, -sa) * s1 + Q(Q_T, 0) * s0) * iw);
    rspec = dabs(un) + dsqrt(c2 * n2);
    if (ph.k2 != 0.0) {
      const T pm2 = Q(Q_P, -2 * sa), pm1 = Q(Q_P, -sa), p0 = Q(Q_P, 0), pp1 = Q(Q_P, sa);
      // the larger of each pair of ratios, compared by cross products
      T kn = dabs(pm1 - 2.0 * p0 + pp1), kd = dabs(pm1 + 2.0 * p0 + pp1);
      const T kn2 = dabs(pm2 - 2.0 * pm1 + p0), kd2 = dabs(pm2 + 2.0 * pm1 + p0);
      if (val(kn) * val(kd2) < val(kn2) * val(kd)) kn = kn2, kd = kd2;
      const double sn = sqrt(n2);
      T vn = s.vd[r0], vdn = s.c[r0] * sn + 1e-15;
      const T vn2 = s.vd[r1], vdn2 = s.c[r1] * sn + 1e-15;
      if (val(vn2) * val(vdn) < val(vn) * val(vdn2)) vn = vn2, vdn = vdn2;
      const T duc = dmax(s.duc[r0], s.duc[r1]);
      eps2 = ph.k2 * (kn / kd * duc * dswitch(2.5 + vn / vdn));
    }
    eps4 = ph.k4 - eps2 * 12.0;
    if (!(0.0 < val(eps4))) eps4 = T(0.0);
  }
  __builtin_amdgcn_sched_barrier(0);
  // ---- viscous flux
  T v1, v2;
  {
    // rows 1 and 2 take the 2nd-order flux, and so does order 3 throughout
    const bool o4 = ORD != 3 && (!NEAR || j >= 3);
    const double al = (o4 ? Coef::r24 : 1.0) * fm.vf * 0.5, ac = (o4 ? Coef::cross : 0.25) * fm.vf * 0.5;
    const double cx[4] = {(fm.px[0] + nx) * al, -(fm.px[1] + nx) * al, (fm.px[2] + fm.px[3]) * ac,
                          -(fm.px[4] + fm.px[5]) * ac};
    const double cy[4] = {(fm.py[0] + ny) * al, -(fm.py[1] + ny) * al, (fm.py[2] + fm.py[3]) * ac,
                          -(fm.py[4] + fm.py[5]) * ac};
    constexpr int ra = J ? TL::NROWS : 1, rc = J ? 1 : TILE;
    const int rb = (J ? ty : tx) * ra + ((J ? tx : ty) + 2) * rc;
    // the values around the face (along +, -; across +, -) and on it
    struct Around { T p, m, cp, cm, f; };
    auto around = [&](int k) {
      const int pl = k == 3 ? Q_T : Q_U + k;
      Around r;
      const T f0 = Q(pl, 0), f1 = Q(pl, -sa);
      if (o4) {
        if constexpr (ORD != 3) {
          auto row = [&](int n) -> T {
            if constexpr (TL::SUMS) return s.rows[J][k][rb + n * rc];
            else return 9.0 * (Q(pl, n * sc - sa) + Q(pl, n * sc)) - (Q(pl, n * sc - 2 * sa) + Q(pl, n * sc + sa));
          };
          const T m1 = row(-1), z = row(0), p1 = row(1);
          r.p = 26.0 * f0 - (Q(pl, sa) + f1);
          r.m = 26.0 * f1 - (f0 + Q(pl, -2 * sa));
          r.cp = 7.0 * (z + p1) - (m1 + row(2));
          r.cm = 7.0 * (m1 + z) - (row(-2) + p1);
          r.f = 0.0625 * z;
        }
      } else {
        const T fs = f0 + f1;
        r.p = f0;
        r.m = f1;
        r.cp = fs + (Q(pl, sc) + Q(pl, sc - sa));
        r.cm = fs + (Q(pl, -sc) + Q(pl, -sc - sa));
        r.f = 0.5 * fs;
      }
      return r;
    };
    auto dot = [](const Around& a, const double c[4]) { return a.p * c[0] + a.m * c[1] + a.cp * c[2] + a.cm * c[3]; };
    const T mmu = o4 ? 0.0625 * (9.0 * (Q(Q_MU, 0) + Q(Q_MU, -sa)) - (Q(Q_MU, sa) + Q(Q_MU, -2 * sa)))
                     : 0.5 * (Q(Q_MU, 0) + Q(Q_MU, -sa));
    const Around u = around(0), v = around(1);
    const T ux = dot(u, cx), uy = dot(u, cy), vx = dot(v, cx), vy = dot(v, cy);
    const T sh = uy + vx;
    const T f1 = mmu * ((Coef::twothird * nx) * (2.0 * ux - vy) + ny * sh);
    const T f2 = mmu * (nx * sh + (Coef::twothird * ny) * (2.0 * vy - ux));
    double cn[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) cn[k] = nx * cx[k] + ny * cy[k];
    const Around w = around(2);
    const T f3 = mmu * dot(w, cn);
    const T f4 = mmu * ph.cpp * dot(around(3), cn) + u.f * f1 + v.f * f2 + w.f * f3;
    h.h0 = T(0.0);
    v1 = f1, v2 = f2;
    h.h3 = -f3, h.h4 = -f4;
  }
  __builtin_amdgcn_sched_barrier(0);
  // ---- Euler flux and dissipation, pair by pair
  // (the momentum as it is stored: rho times the rounded velocity would carry
  // a rounding more into the mass flux; the momentum fluxes as x and y sums with
  // the pressure inside, the order that keeps the rounding of the pressure, the
  // largest term at a low Mach number, where the scheme's own statement has it)
  T xx(0.0), xy(0.0), yy(0.0), d1(0.0), d2(0.0);
  sfor<0, TL::L>([&](auto K) {
    // the second pair first: its small product takes the rounding that the
    // largest one's would
    constexpr int k = decltype(K)::value < 2 ? 1 - decltype(K)::value : decltype(K)::value;
    constexpr int o0 = k * sa, o1 = -(k + 1) * sa;
    const T d = k == 0 ? 0.5 * eps2 + C::pred(0) * eps4 : (k % 2 ? -C::pred(k) : C::pred(k)) * eps4;
    const T rd = rspec * d;
    h.h0 = h.h0 - rd * (Q(Q_RO, o0) - Q(Q_RO, o1));
    d1 = d1 + d * (Q(Q_RU, o0) - Q(Q_RU, o1));
    d2 = d2 + d * (Q(Q_RV, o0) - Q(Q_RV, o1));
    h.h3 = h.h3 - rd * (Q(Q_RW, o0) - Q(Q_RW, o1));
    h.h4 = h.h4 - rd * (Q(Q_RE, o0) - Q(Q_RE, o1));
    if (!(NEAR && J) || j >= C::RC) {
      constexpr double c = C::centred(k);
      const T q0 = nx * Q(Q_RU, o0) + ny * Q(Q_RV, o0), q1 = nx * Q(Q_RU, o1) + ny * Q(Q_RV, o1);
      h.h0 = h.h0 + c * (q0 + q1);
      xx = xx + c * ((Q(Q_RU, o0) * Q(Q_U, o0) + Q(Q_P, o0)) + (Q(Q_RU, o1) * Q(Q_U, o1) + Q(Q_P, o1)));
      xy = xy + c * (Q(Q_RU, o0) * Q(Q_V, o0) + Q(Q_RU, o1) * Q(Q_V, o1));
      yy = yy + c * ((Q(Q_RV, o0) * Q(Q_V, o0) + Q(Q_P, o0)) + (Q(Q_RV, o1) * Q(Q_V, o1) + Q(Q_P, o1)));
      h.h3 = h.h3 + c * (q0 * Q(Q_W, o0) + q1 * Q(Q_W, o1));
      h.h4 = h.h4 + c * (q0 * Q(Q_H, o0) + q1 * Q(Q_H, o1));
    }
  });
  if (NEAR && J && j < C::RC) {
    // cell rows 1 .. NW
    const double* wt = s.wt + (j - 2) * C::NW;
    const int o = (1 - j) * sa;
#pragma unroll
    for (int t = 0; t < C::NW; ++t) {
      const double c = wt[t];
      const int off = o + t * sa;
      const T q = c * (nx * Q(Q_RU, off) + ny * Q(Q_RV, off));
      h.h0 = h.h0 + q;
      xx = xx + c * (Q(Q_RU, off) * Q(Q_U, off) + Q(Q_P, off));
      xy = xy + c * (Q(Q_RU, off) * Q(Q_V, off));
      yy = yy + c * (Q(Q_RV, off) * Q(Q_V, off) + Q(Q_P, off));
      h.h3 = h.h3 + q * Q(Q_W, off);
      h.h4 = h.h4 + q * Q(Q_H, off);
    }
  }
  h.h1 = xx * nx + xy * ny - rspec * d1 - v1;
  h.h2 = xy * nx + yy * ny - rspec * d2 - v2;
  return h;
}

// One tile: the cells [x0, x0 + 14] x [y0, y0 + 14] of the interior.
// V: StateView<double> or PairView; NEAR: the tiles at the wall.
template <class V, int ORD, bool NOWALL, bool NEAR>
__device__ inline void residual_tile(Tile<typename V::Scalar, ORD>& s, const V& w, const ResPhys& ph, const Metric& g,
                                     const ResOut& out, int bx, int by) {
  using T = typename V::Scalar;
  using TL = Tile<T, ORD>;
  using C = NearWall<ORD>;
  constexpr int S = TL::S, SS = TL::SS, L = TL::L, A = TL::A;
  const Mesh& m = w.m;
  const int tid = threadIdx.x, x0 = 1 + bx * TILE_CELLS, y0 = 1 + by * TILE_CELLS;
  const int half = tid / (TILE * TILE), t = tid % (TILE * TILE), tx = t % TILE, ty = t / TILE;
  // the face's metrics, on their way while the cells are loaded (lanes past
  // the last face take its)
  const int fi = min(x0 + tx, m.im + 1), fj = min(y0 + ty, m.jm + 1);
  const FaceMetric fm = half ? face_metric<true>(m, g, fi, fj) : face_metric<false>(m, g, fi, fj);
  if (NEAR)
    for (int k = tid; k < (C::RC - 2) * C::NW; k += TILE_THREADS) s.wt[k] = near_wall<ORD>.w[k];
  // ---- cells and their primitives (primvisc.F)
  for (int x = tid; x < SS; x += TILE_THREADS) {
    const int li = x % S, lj = x / S, i = x0 - L + li, j = y0 - L + lj;
    // (i, j) >= 1 - L >= 1 - gh
    if (i > m.im + m.gh || j > m.jm + m.gh) continue;
    T c[5];
#pragma unroll
    for (int e = 0; e < 5; ++e) c[e] = w(i, j, e);
    const T rom1 = 1.0 / c[0];
    const T u = c[1] * rom1, v = c[2] * rom1, ww = c[3] * rom1;
    const T ec = 0.5 * (u * u + v * v + ww * ww);
    const T e = (c[4] - ec * c[0]) * rom1;
    const T tt = e * ph.cvm1;
    const T st = dsqrt(tt);
#pragma unroll
    for (int k = 0; k < 5; ++k) s.q[(Q_RO + k) * SS + x] = c[k];
    s.q[Q_U * SS + x] = u;
    s.q[Q_V * SS + x] = v;
    s.q[Q_W * SS + x] = ww;
    s.q[Q_T * SS + x] = tt;
    const T p = ph.gm1 * c[0] * e;
    s.q[Q_P * SS + x] = p;
    s.q[Q_H * SS + x] = (c[4] + p) * rom1;
    s.q[Q_MU * SS + x] = ph.betas / (tt + ph.s_suth) * st * tt;
    const int ai = li - L + 1, aj = lj - L + 1;
    if (ai >= 0 && ai < A && aj >= 0 && aj < A) {
      s.sr[aj * A + ai] = dsqrt(c[0]);
      s.c[aj * A + ai] = ph.sqgr * st;
    }
  }
  __syncthreads();
  // ---- sensor: gradop_*pi/j.F, gradient.F; a ghost cell's gradients are
  // extrapolated from the two interior cells beside it (gradveloingh.F:
  // 2 g(1) - g(2))
  if (ph.k2 != 0.0 && tid < A * A) {
    const int ai = tid % A, aj = tid / A, i = x0 - 1 + ai, j = y0 - 1 + aj;
    const int di = i < 1 ? 1 : i > m.im ? -1 : 0, dj = j < 1 ? 1 : j > m.jm ? -1 : 0;
    if (i <= m.im + 1 && j <= m.jm + 1 && (di == 0 || dj == 0) && (NOWALL || j >= 1)) {
      const int n = di | dj ? 2 : 1;
      T gr[4] = {T(0.0), T(0.0), T(0.0), T(0.0)};
      for (int k = 0; k < n; ++k) {
        // the cell itself, or the first and second inner neighbour
        const int o = n == 1 ? 0 : k + 1, ci = i + o * di, cj = j + o * dj;
        const int b = (cj - y0 + L) * S + ci - x0 + L;
        T gi[2], gj[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const T* f = s.q + (Q_U + q) * SS + b;
          gi[q] = C::grad(0) * (f[1] - f[-1]);
          gj[q] = C::grad(0) * (f[S] - f[-S]);
#pragma unroll
          for (int d = 1; d < TL::R; ++d) {
            gi[q] = gi[q] + C::grad(d) * (f[d + 1] - f[-d - 1]);
            gj[q] = gj[q] + C::grad(d) * (f[(d + 1) * S] - f[-(d + 1) * S]);
          }
        }
        const long n0 = nidx(m, ci, cj), nn = m.nnode, up = m.ni + 1;
        const double vm = 0.5 / g.vol[cidx(m, ci, cj)];
        const double dx1 = (g.nx[n0] + g.nx[n0 + 1]) * vm, dx2 = (g.nx[n0 + nn] + g.nx[n0 + up + nn]) * vm;
        const double dy1 = (g.ny[n0] + g.ny[n0 + 1]) * vm, dy2 = (g.ny[n0 + nn] + g.ny[n0 + up + nn]) * vm;
        const double sg = n == 1 ? 1.0 : k ? -1.0 : 2.0;
        gr[G_UX] = gr[G_UX] + sg * (dx1 * gi[0] + dx2 * gj[0]);
        gr[G_UY] = gr[G_UY] + sg * (dy1 * gi[0] + dy2 * gj[0]);
        gr[G_VX] = gr[G_VX] + sg * (dx1 * gi[1] + dx2 * gj[1]);
        gr[G_VY] = gr[G_VY] + sg * (dy1 * gi[1] + dy2 * gj[1]);
      }
      const T div = gr[G_UX] + gr[G_VY], rot = gr[G_VX] - gr[G_UY], div2 = div * div;
      s.duc[tid] = div2 / (div2 + rot * rot + 1e-15);
      s.vd[tid] = 10.0 * g.vol[cidx(m, i, j)] * div;
    }
  }
  if constexpr (TL::SUMS) {
    // ---- along-face sums of the compact viscous flux, both directions
    constexpr int NR = TL::NROWS * TILE;
    for (int x = tid; x < 8 * NR; x += TILE_THREADS) {
      const int dir = x / (4 * NR), k = x / NR % 4, y = x % NR;
      // y = across, along (i-faces) or along, across (j-faces): lanes along i
      const int li = dir ? y % TL::NROWS - 2 : y % TILE, lj = dir ? y / TL::NROWS : y / TILE - 2;
      const int sa = dir ? S : 1;
      const T* f = s.q + (k == 3 ? Q_T : Q_U + k) * SS + (lj + L) * S + li + L;
      s.rows[dir][k][y] = 9.0 * (f[-sa] + f[0]) - (f[-2 * sa] + f[sa]);
    }
  }
  __syncthreads();
  // ---- faces
  Flux<T> h;
  if (half == 0) h = tile_face<T, ORD, false, NEAR>(s, ph, fm, tx, ty, y0 + ty);
  else h = tile_face<T, ORD, true, NEAR>(s, ph, fm, tx, ty, y0 + ty);
  __syncthreads();
  // ---- balance (balanceloop.F)
  constexpr int F = TILE * TILE;
  T* hq = s.q + half * 5 * F + t;
  hq[0] = h.h0, hq[F] = h.h1, hq[2 * F] = h.h2, hq[3 * F] = h.h3, hq[4 * F] = h.h4;
  __syncthreads();
  const int i = x0 + tx, j = y0 + ty;
  if (tx < TILE_CELLS && ty < TILE_CELLS && i <= m.im && j <= m.jm) {
    const long c = cidx(m, i, j);
    for (int e = half; e < 5; e += 2) {
      const T* hi = s.q + e * F + t;
      const T* hj = s.q + (5 + e) * F + t;
      const T r = -(hi[1] - hi[0]) - (hj[TILE] - hj[0]);
      if constexpr (std::is_same<T, double>::value) {
        out.res[c + (long)e * m.ncell] = r;
      } else {
        if (out.res) out.res[c + (long)e * m.ncell] = r.v;
        if (out.resd) out.resd[c + (long)e * m.ncell] = r.d[0];
      }
    }
  }
}

template <class V, int ORD, bool NOWALL>
__global__ void __launch_bounds__(TILE_THREADS, sizeof(typename V::Scalar) > 8 ? 2 : 4)
    k_residual(V w, ResPhys ph, Metric g, ResOut out) {
  using TL = Tile<typename V::Scalar, ORD>;
  __shared__ __align__(16) unsigned char mem[sizeof(TL)];
  TL& s = *reinterpret_cast<TL*>(mem);
  int bx, by;
  xcd_block(bx, by);
  // (two whole tiles: one with both kinds of faces in it spills registers for
  // the sake of the few that stand at the wall)
  if (!NOWALL && by == 0) residual_tile<V, ORD, NOWALL, true>(s, w, ph, g, out, bx, by);
  else residual_tile<V, ORD, NOWALL, false>(s, w, ph, g, out, bx, by);
}

// The interior of 5 planes, from one array to another.
__global__ void k_store_interior(Mesh m, const double* __restrict__ from, double* __restrict__ to) {
  const int i = 1 + blockIdx.x * blockDim.x + threadIdx.x;
  const int j = 1 + blockIdx.y * blockDim.y + threadIdx.y;
  if (i > m.im || j > m.jm) return;
  const long c = cidx(m, i, j);
#pragma unroll
  for (int e = 0; e < 5; ++e) to[c + e * m.ncell] = from[c + e * m.ncell];
}

}  // namespace bca
