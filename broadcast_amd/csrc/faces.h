// The stencils of the DNC5 face fluxes written against an accessor whose cell
// offsets are compile-time constants, for the face adjoints (adjface.h) and the
// Jacobian's face blocks (fwdface.h, blockskern.h):
//
//   PlainAcc<double>    a face's primal values
//   SeededAcc<SI, SJ>   block of the wall face      (only the cell at offset
//                       d hn(face) / d w(cell)       (SI, SJ) carries a 5-way
//                                                     tangent; all else double)
//
// (the residual itself: residual.h).
//
// Formulas: srcfv/rhs/flux_num_dnc5.F90 (expanded srcfv/prepro/flux_num_dnc5.f90)
//   Euler        euler_o6_i.F / nearbndfluxes{3,5}demi_7p.F (coefnearbnd_7p.F)
//   dissipation  predictor_7p_i.F, spectralradius_i.F, ducrosfordnc_i.F
//   viscous      flux_visqueux_o4_i.F, flux_visqueux_o2_i.F, fluxwall.F
#pragma once
#include <type_traits>

#include "scheme.h"

namespace bca {

template <int B, int E, class F>
__device__ inline void sfor(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    sfor<B + 1, E>(f);
  }
}

// primitives of one cell from its 5 conservative values (primvisc.F)
template <class T>
__device__ inline void prim_of(const Phys& ph, const T& ro, const T& ru, const T& rv, const T& rw,
                               const T& re, T out[NPRIM]) {
  const double cvm1 = 1.0 / ph.cv;
  const double betas = ph.muref * (ph.tref + ph.cs) / (sqrt(ph.tref) * ph.tref);
  T rom1 = 1.0 / ro;
  T u = ru * rom1, v = rv * rom1, ww = rw * rom1;
  T ec = 0.5 * (u * u + v * v + ww * ww);
  T e = (re - ec * ro) * rom1;
  T t = e * cvm1;
  T p = (ph.gam - 1.0) * ro * e;
  out[P_U] = u;
  out[P_V] = v;
  out[P_W] = ww;
  out[P_T] = t;
  out[P_P] = p;
  out[P_H] = (re + p) * rom1;
  out[P_MU] = betas / (t + ph.s_suth) * dsqrt(t) * t;
}

// ------------------------------------------------------------ accessors
// Common part: position of the face's right cell (i, j) and metrics.
struct AccBase {
  Mesh m;
  Phys ph;
  Metric g;
  int i, j;
  __device__ double NX(int di, int dj, int d) const { return g.nx[nidx(m, i + di, j + dj) + (long)d * m.nnode]; }
  __device__ double NY(int di, int dj, int d) const { return g.ny[nidx(m, i + di, j + dj) + (long)d * m.nnode]; }
  __device__ double VOL(int di, int dj) const { return g.vol[cidx(m, i + di, j + dj)]; }
  __device__ double VOLF(int di, int dj, int d) const { return g.volf[cidx(m, i + di, j + dj) + (long)d * m.ncell]; }
};

// Every cell value read from planes of T (T = double or Dual<N>).
template <class T>
struct PlainAcc : AccBase {
  using Out = T;
  template <int DI, int DJ> using CT = T;
  const T* w;
  const T* prim;
  const T* grad;
  template <int DI, int DJ> __device__ T W(int e) const { return w[cidx(m, i + DI, j + DJ) + (long)e * m.ncell]; }
  template <int DI, int DJ> __device__ T P(int k) const { return prim[cidx(m, i + DI, j + DJ) + (long)k * m.ncell]; }
  template <int DI, int DJ> __device__ T G(int k) const { return grad[cidx(m, i + DI, j + DJ) + (long)k * m.ncell]; }
};

// Unit 5-way tangent on the cell at offset (SI, SJ) (the 5 conservative
// variables of that cell), FP64 everywhere else.
template <int SI, int SJ>
struct SeededAcc : AccBase {
  using Out = Dual<5>;
  template <int DI, int DJ> using CT = std::conditional_t<(DI == SI && DJ == SJ), Dual<5>, double>;
  const double* w;
  const double* prim;
  const double* grad;
  Dual<5> sw[5];      // seeded cell state
  Dual<5> sp[NPRIM];  // its primitives

  __device__ void seed() {
    const long c = cidx(m, i + SI, j + SJ);
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      sw[e] = Dual<5>(w[c + (long)e * m.ncell]);
      sw[e].d[e] = 1.0;
    }
    prim_of(ph, sw[0], sw[1], sw[2], sw[3], sw[4], sp);
  }
  template <int DI, int DJ> __device__ CT<DI, DJ> W(int e) const {
    if constexpr (DI == SI && DJ == SJ) return sw[e];
    else return w[cidx(m, i + DI, j + DJ) + (long)e * m.ncell];
  }
  template <int DI, int DJ> __device__ CT<DI, DJ> P(int k) const {
    if constexpr (DI == SI && DJ == SJ) return sp[k];
    else return prim[cidx(m, i + DI, j + DJ) + (long)k * m.ncell];
  }
};

// ------------------------------------------------------------ building blocks
// contour-integral face gradient of primitive k from the four staggered values
struct Contour {
  double nxN, nxS, nxO, nxE, nyN, nyS, nyO, nyE, vf;
};
template <class VN, class VS, class VO, class VE>
__device__ inline auto cgx(const Contour& c, const VN& vN, const VS& vS, const VO& vO, const VE& vE) {
  return (vN * c.nxN + vS * c.nxS + vO * c.nxO + vE * c.nxE) * c.vf;
}
template <class VN, class VS, class VO, class VE>
__device__ inline auto cgy(const Contour& c, const VN& vN, const VS& vS, const VO& vO, const VE& vE) {
  return (vN * c.nyN + vS * c.nyS + vO * c.nyO + vE * c.nyE) * c.vf;
}

// ---------------------------------------------------------------- i-faces
template <class A>
__device__ inline Contour contour_i(const A& a) {
  Contour c;
  c.vf = a.VOLF(0, 0, 0);
  c.nxN = 0.5 * (a.NX(1, 0, 0) + a.NX(0, 0, 0));
  c.nxS = -(0.5 * (a.NX(-1, 0, 0) + a.NX(0, 0, 0)));
  c.nxO = 0.5 * (a.NX(-1, 1, 1) + a.NX(0, 1, 1));
  c.nxE = -(0.5 * (a.NX(-1, 0, 1) + a.NX(0, 0, 1)));
  c.nyN = 0.5 * (a.NY(1, 0, 0) + a.NY(0, 0, 0));
  c.nyS = -(0.5 * (a.NY(-1, 0, 0) + a.NY(0, 0, 0)));
  c.nyO = 0.5 * (a.NY(-1, 1, 1) + a.NY(0, 1, 1));
  c.nyE = -(0.5 * (a.NY(-1, 0, 1) + a.NY(0, 0, 1)));
  return c;
}

// staggered values of primitive k around the i-face, compact 4th order
template <class A>
__device__ inline auto ivals_o4(const A& a, int k) {
  auto row = [&](auto JJ) {
    constexpr int jj = decltype(JJ)::value;
    return -a.template P<-2, jj>(k) + 9.0 * a.template P<-1, jj>(k) + 9.0 * a.template P<0, jj>(k) -
           a.template P<1, jj>(k);
  };
  auto r0 = row(std::integral_constant<int, -2>{});
  auto r1 = row(std::integral_constant<int, -1>{});
  auto r2 = row(std::integral_constant<int, 0>{});
  auto r3 = row(std::integral_constant<int, 1>{});
  auto r4 = row(std::integral_constant<int, 2>{});
  auto vN = Coef::r24 * (-a.template P<1, 0>(k) + 26.0 * a.template P<0, 0>(k) - a.template P<-1, 0>(k));
  auto vS = Coef::r24 * (-a.template P<0, 0>(k) + 26.0 * a.template P<-1, 0>(k) - a.template P<-2, 0>(k));
  auto vE = Coef::cross * (-r0 + 7.0 * r1 + 7.0 * r2 - r3);
  auto vO = Coef::cross * (-r1 + 7.0 * r2 + 7.0 * r3 - r4);
  struct Q { decltype(vN) N; decltype(vS) S; decltype(vO) O; decltype(vE) E; };
  return Q{vN, vS, vO, vE};
}
template <class A>
__device__ inline auto ivals_o2(const A& a, int k) {
  auto vN = a.template P<0, 0>(k);
  auto vS = a.template P<-1, 0>(k);
  auto vE = 0.25 * (a.template P<0, 0>(k) + a.template P<0, -1>(k) + a.template P<-1, 0>(k) +
                    a.template P<-1, -1>(k));
  auto vO = 0.25 * (a.template P<0, 0>(k) + a.template P<0, 1>(k) + a.template P<-1, 0>(k) +
                    a.template P<-1, 1>(k));
  struct Q { decltype(vN) N; decltype(vS) S; decltype(vO) O; decltype(vE) E; };
  return Q{vN, vS, vO, vE};
}

// predictor of a face whose right cell is offset (0, 0) and left cell
// (-DX, -DY): 6 points for ORD 5 (predictor_7p_i.F)
template <int DX, int DY, class A>
__device__ inline auto predictor(const A& a, int e) {
  return -(Coef::d3 * a.template W<-3 * DX, -3 * DY>(e)) + Coef::d2 * a.template W<-2 * DX, -2 * DY>(e) -
         Coef::d1 * a.template W<-DX, -DY>(e) + Coef::d1 * a.template W<0, 0>(e) -
         Coef::d2 * a.template W<DX, DY>(e) + Coef::d3 * a.template W<2 * DX, 2 * DY>(e);
}

// ---------------------------------------------------------------- j-faces
template <class A>
__device__ inline Contour contour_j(const A& a) {
  Contour c;
  c.vf = a.VOLF(0, 0, 1);
  c.nxN = 0.5 * (a.NX(1, -1, 0) + a.NX(1, 0, 0));
  c.nxS = -(0.5 * (a.NX(0, -1, 0) + a.NX(0, 0, 0)));
  c.nxO = 0.5 * (a.NX(0, 1, 1) + a.NX(0, 0, 1));
  c.nxE = -(0.5 * (a.NX(0, -1, 1) + a.NX(0, 0, 1)));
  c.nyN = 0.5 * (a.NY(1, -1, 0) + a.NY(1, 0, 0));
  c.nyS = -(0.5 * (a.NY(0, -1, 0) + a.NY(0, 0, 0)));
  c.nyO = 0.5 * (a.NY(0, 1, 1) + a.NY(0, 0, 1));
  c.nyE = -(0.5 * (a.NY(0, -1, 1) + a.NY(0, 0, 1)));
  return c;
}

template <class A>
__device__ inline auto jvals_o4(const A& a, int k) {
  auto col = [&](auto II) {
    constexpr int ii = decltype(II)::value;
    return -a.template P<ii, -2>(k) + 9.0 * a.template P<ii, -1>(k) + 9.0 * a.template P<ii, 0>(k) -
           a.template P<ii, 1>(k);
  };
  auto c0 = col(std::integral_constant<int, -2>{});
  auto c1 = col(std::integral_constant<int, -1>{});
  auto c2 = col(std::integral_constant<int, 0>{});
  auto c3 = col(std::integral_constant<int, 1>{});
  auto c4 = col(std::integral_constant<int, 2>{});
  auto vN = Coef::cross * (-c1 + 7.0 * c2 + 7.0 * c3 - c4);
  auto vS = Coef::cross * (-c0 + 7.0 * c1 + 7.0 * c2 - c3);
  auto vE = Coef::r24 * (-a.template P<0, 0>(k) + 26.0 * a.template P<0, -1>(k) - a.template P<0, -2>(k));
  auto vO = Coef::r24 * (-a.template P<0, 1>(k) + 26.0 * a.template P<0, 0>(k) - a.template P<0, -1>(k));
  struct Q { decltype(vN) N; decltype(vS) S; decltype(vO) O; decltype(vE) E; };
  return Q{vN, vS, vO, vE};
}
template <class A>
__device__ inline auto jvals_o2(const A& a, int k) {
  auto vN = 0.25 * (a.template P<0, 0>(k) + a.template P<1, 0>(k) + a.template P<0, -1>(k) +
                    a.template P<1, -1>(k));
  auto vS = 0.25 * (a.template P<0, 0>(k) + a.template P<-1, 0>(k) + a.template P<0, -1>(k) +
                    a.template P<-1, -1>(k));
  auto vO = a.template P<0, 0>(k);
  auto vE = a.template P<0, -1>(k);
  struct Q { decltype(vN) N; decltype(vS) S; decltype(vO) O; decltype(vE) E; };
  return Q{vN, vS, vO, vE};
}

// adiabatic no-slip wall j-face at j = 1 (fluxwall.F)
template <class A>
__device__ inline void jface_wall(const A& a, typename A::Out hn[5]) {
  using Out = typename A::Out;
  const double n2x = a.NX(0, 0, 1), n2y = a.NY(0, 0, 1), vf = a.VOLF(0, 0, 1);
  auto pw = 1.125 * a.template P<0, 0>(P_P) - 0.125 * a.template P<0, 1>(P_P);
  auto mmu = a.template P<0, 0>(P_MU);
  auto u = a.template P<0, 0>(P_U), v = a.template P<0, 0>(P_V), ww = a.template P<0, 0>(P_W);
  auto ux = 2.0 * u * n2x * vf, vx = 2.0 * v * n2x * vf, wx = 2.0 * ww * n2x * vf;
  auto uy = 2.0 * u * n2y * vf, vy = 2.0 * v * n2y * vf, wy = 2.0 * ww * n2y * vf;
  auto fu = Coef::twothird * mmu * (2.0 * ux - vy);
  auto fvv = mmu * (uy + vx);
  auto fw = mmu * wx;
  auto gu = mmu * (uy + vx);
  auto gvv = Coef::twothird * mmu * (-ux + 2.0 * vy);
  auto gw = mmu * wy;
  hn[0] = Out(0.0);
  hn[1] = Out(pw * n2x - (fu * n2x + gu * n2y));
  hn[2] = Out(pw * n2y - (fvv * n2x + gvv * n2y));
  hn[3] = Out(-(fw * n2x + gw * n2y));
  hn[4] = Out(0.0);
}

}  // namespace bca
