// Face-local Jacobian blocks by hand-derived forward differentiation (phase 1
// of the colored Jacobian): B(face, o) = d hn(face) / d w(face + o) for the 24
// stencil offsets of every face above the wall row, all of them by one thread.
//
// hn = Euler - dissipation - viscous depends on a stencil cell through its own
// Euler flux (a fixed coefficient), through the jump and predictor (fixed
// coefficients), through the dissipation scalars rspec and eps2 (two gradients
// of the face, formed once by the reverse of diss_primal) and through the
// linear stencils of the viscous flux (a face gradient weight per direction
// and a face-value weight).  So after one primal pass of the face a block is a
// few products of face-level numbers with the cell's d prim / d w:
//
//   B = c dF/dw - (A (x) drspec + E (x) deps2 + s I) - V dprim/dw
//
// with A_e = eps2 jump_e + eps4 pred_e, E_e = rspec (jump_e - 12 pred_e)
// (eps4 = max(0, k4 - 12 eps2)), s = rspec (eps2 cj + eps4 cp), V the 4 x 5
// matrix of the stresses by (u, v, w, T, mu).  The conventions at abs / max /
// sqrt are Dual's, by diss_adjoint.
//
// What bounds it: the 600 values a face stores (1.9 GB at 512 x 384 for both
// families, 0.4 ms at the card's copy rate), at one wave per SIMD (256 VGPRs).
// 512 x 384: i-faces 0.29 ms, j-faces 0.21 ms beside the ghost tangents, where
// 24 seeded passes per face (each recomputing the face's primal, a launch per
// offset) took 1.1 ms.  131 x 67: 47 + 50 us for the interior families and
// 21-27 us for the rows next to the wall, where the seeded passes took 48
// launches of 21 us and 260-356 us for each of those rows (24 offsets in one
// thread, 0.7 KB of scratch): three Newton Jacobians 4.76 -> 1.95 ms.
#pragma once
#include "adjface.h"
#include "blocks.h"

namespace bca {

// The face-level numbers of the blocks.
struct FaceLin {
  double nx, ny;
  Contour c;
  double mmu, lam, uu, vv, ww, s1, s2, s3, s4;  // face values; stresses / mmu, heat flux / lam
  double A[5], E[5], rspec, eps2, eps4;
  double rw0[3], rw1[3], rt0, rt1;              // d rspec: rho, rho u, rho v and T of cells 0, -1
  double ep[4], et0, et1;                       // d eps2: p of cells -2 .. 1, T of cells 0, -1
  GradW gw[4];                                  // d eps2: u, v along i, j of the gradient cells -2 .. 1
};

template <bool J, bool O4>
__device__ inline void face_linearise(const PlainAcc<double>& a, FaceLin& f) {
  constexpr int DX = J ? 0 : 1, DY = J ? 1 : 0, D = J ? 1 : 0;
  const Phys& ph = a.ph;
  f.nx = a.NX(0, 0, D), f.ny = a.NY(0, 0, D);
  const DissPrim ds = diss_primal<DX, DY>(a, D);
  f.rspec = ds.rspec, f.eps2 = ds.eps2, f.eps4 = ds.eps4;
  const double act = 0.0 < ph.k4 - ds.eps2 * 12.0 ? 12.0 : 0.0;
#pragma unroll
  for (int e = 0; e < 5; ++e) {
    const double jp = 0.5 * (a.template W<0, 0>(e) - a.template W<-DX, -DY>(e));
    const double pr = predictor<DX, DY>(a, e);
    f.A[e] = ds.eps2 * jp + ds.eps4 * pr;
    f.E[e] = ds.rspec * (jp - act * pr);
  }
  {
    // k2 = 0 in these constants: the spectral radius alone
    Phys p0 = ph;
    p0.k2 = 0.0;
    const DissAdj r = diss_adjoint(ds, p0, 1.0, 0.0, 0.0);
#pragma unroll
    for (int q = 0; q < 3; ++q) f.rw0[q] = r.w0[q], f.rw1[q] = r.w1[q];
    f.rt0 = r.t0, f.rt1 = r.t1;
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) f.ep[k] = 0.0, f.gw[k] = GradW{0.0, 0.0, 0.0, 0.0};
  f.et0 = f.et1 = 0.0;
  if (ph.k2 != 0.0) {
    const DissAdj r = diss_adjoint(ds, ph, 0.0, 1.0, 0.0);
#pragma unroll
    for (int k = 0; k < 4; ++k) f.ep[k] = r.p[k];
    f.et0 = r.t0, f.et1 = r.t1;
    // the gradients' adjoints on the four cells along the normal whose
    // 4th-order gradients they reach (an extrapolated ghost gradient is
    // 2 g(a) - g(b))
    const bool ext0 = J ? a.j == a.m.jm + 1 : a.i == a.m.im + 1;  // cell 0 a ghost layer
    const bool ext1 = !J && a.i == 1;                             // cell -1 a ghost layer
    double gbp[4][NGRAD];
#pragma unroll
    for (int n = 0; n < NGRAD; ++n) {
      gbp[0][n] = ext0 ? -r.g0[n] : 0.0;
      gbp[1][n] = (ext0 ? 2.0 * r.g0[n] : 0.0) + (ext1 ? 0.0 : r.g1[n]);
      gbp[2][n] = (ext0 ? 0.0 : r.g0[n]) + (ext1 ? 2.0 * r.g1[n] : 0.0);
      gbp[3][n] = ext1 ? -r.g1[n] : 0.0;
    }
    sfor<0, 4>([&](auto K) {
      constexpr int k = decltype(K)::value;
      // only the cells a gradient of this face uses (the others may lie
      // beyond the ghost frame)
      const bool used = k == 2 ? !ext0 || ext1 : k == 1 ? !ext1 || ext0 : k == 0 ? ext0 : ext1;
      if (used) f.gw[k] = grad_weights<(k - 2) * DX, (k - 2) * DY>(a, gbp[k]);
    });
  }
  const ViscPrimal v = visc_primal<J, O4>(a);
  constexpr double tt = Coef::twothird;
  f.c = v.c;
  f.mmu = v.mmu, f.lam = v.lam, f.uu = v.uu, f.vv = v.vv, f.ww = v.ww;
  f.s1 = f.nx * (tt * (2.0 * v.ux - v.vy)) + f.ny * (v.uy + v.vx);
  f.s2 = f.nx * (v.uy + v.vx) + f.ny * (tt * (2.0 * v.vy - v.ux));
  f.s3 = f.nx * v.wx + f.ny * v.wy;
  f.s4 = f.nx * v.tx + f.ny * v.ty;
}

// The block of offset (SI, SJ).
template <bool J, bool O4, int ROW, int SI, int SJ>
__device__ inline void face_block(const PlainAcc<double>& a, const FaceLin& f, const double* cellx, double* out,
                                  long nf) {
  constexpr int DX = J ? 0 : 1, DY = J ? 1 : 0;
  constexpr int along = J ? SJ : SI, across = J ? SI : SJ;
  const Phys& ph = a.ph;
  const double g1 = ph.gam - 1.0, cvm1 = 1.0 / ph.cv;
  const long c = cidx(a.m, a.i + SI, a.j + SJ);
  const double rm = cellx[c + X_RM * a.m.ncell], dmu = cellx[c + X_DMU * a.m.ncell];
  const double u = a.template P<SI, SJ>(P_U), v = a.template P<SI, SJ>(P_V), w = a.template P<SI, SJ>(P_W);
  const double t = a.template P<SI, SJ>(P_T);
  const double ec = 0.5 * (u * u + v * v + w * w), ei = t * ph.cv;
  // d prim / d w: u by (-u, 1, 0, 0, 0) / rho, likewise v, w; T, p
  const double du0 = -u * rm, dv0 = -v * rm, dw0 = -w * rm;
  const double tr = cvm1 * rm;
  const double dt[5] = {tr * (ec - ei), -tr * u, -tr * v, -tr * w, tr};
  const double dp[5] = {g1 * ec, -g1 * u, -g1 * v, -g1 * w, g1};
  double B[5][5];
#pragma unroll
  for (int e = 0; e < 5; ++e)
#pragma unroll
    for (int q = 0; q < 5; ++q) B[e][q] = 0.0;
  // Euler flux of the cell
  if constexpr (across == 0 && euler_coef<ROW>(along) != 0.0) {
    constexpr double ce = euler_coef<ROW>(along);
    const double h = a.template P<SI, SJ>(P_H);
    const double nx = ce * f.nx, ny = ce * f.ny;
    const double qn = nx * a.template W<SI, SJ>(1) + ny * a.template W<SI, SJ>(2);
    const double qr = qn * rm;
    B[0][1] = nx;
    B[0][2] = ny;
#pragma unroll
    for (int q = 0; q < 5; ++q) {
      B[1][q] = nx * dp[q];
      B[2][q] = ny * dp[q];
      B[4][q] = qr * dp[q];
    }
    B[1][0] -= qr * u;
    B[1][1] += nx * u + qr;
    B[1][2] += ny * u;
    B[2][0] -= qr * v;
    B[2][1] += nx * v;
    B[2][2] += ny * v + qr;
    B[3][0] = -qr * w;
    B[3][1] = nx * w;
    B[3][2] = ny * w;
    B[3][3] = qr;
    B[4][0] -= qr * h;
    B[4][1] += nx * h;
    B[4][2] += ny * h;
    B[4][4] += qr;
  }
  IndAcc<SI, SJ> ind;
  ind.m = a.m; ind.ph = ph; ind.g = a.g; ind.i = a.i; ind.j = a.j;
  // jump and predictor
  if constexpr (across == 0) {
    const double cj = 0.5 * (ind.template W<0, 0>(0) - ind.template W<-DX, -DY>(0));
    const double cp = predictor<DX, DY>(ind, 0);
    const double s = f.rspec * (f.eps2 * cj + f.eps4 * cp);
#pragma unroll
    for (int e = 0; e < 5; ++e) B[e][e] -= s;
  }
  // spectral radius of cells 0 and -1
  if constexpr (across == 0 && (along == 0 || along == -1)) {
    const double* rw = along == 0 ? f.rw0 : f.rw1;
    const double rt = along == 0 ? f.rt0 : f.rt1;
    double r[5];
#pragma unroll
    for (int q = 0; q < 5; ++q) r[q] = rt * dt[q] + (q < 3 ? rw[q < 3 ? q : 0] : 0.0);
#pragma unroll
    for (int e = 0; e < 5; ++e)
#pragma unroll
      for (int q = 0; q < 5; ++q) B[e][q] -= f.A[e] * r[q];
  }
  // eps2: p of cells -2 .. 1, T of cells 0 and -1, u and v of the gradients
  constexpr bool in_p = across == 0 && along >= -2 && along <= 1;
  double gu = 0.0, gv = 0.0;
  bool has_g = false;
  sfor<0, 4>([&](auto K) {
    constexpr int k = decltype(K)::value;
    constexpr double wi = grad_wi(SI - (k - 2) * DX, SJ - (k - 2) * DY);
    constexpr double wj = grad_wj(SI - (k - 2) * DX, SJ - (k - 2) * DY);
    if constexpr (wi != 0.0 || wj != 0.0) {
      gu += f.gw[k].cu_i * wi + f.gw[k].cu_j * wj;
      gv += f.gw[k].cv_i * wi + f.gw[k].cv_j * wj;
      has_g = true;
    }
  });
  if (ph.k2 != 0.0 && (in_p || has_g)) {
    double r[5] = {gu * du0 + gv * dv0, gu * rm, gv * rm, 0.0, 0.0};
    if constexpr (in_p) {
      const double ep = f.ep[along + 2], et = along == 0 ? f.et0 : along == -1 ? f.et1 : 0.0;
#pragma unroll
      for (int q = 0; q < 5; ++q) r[q] += ep * dp[q] + et * dt[q];
    }
#pragma unroll
    for (int e = 0; e < 5; ++e)
#pragma unroll
      for (int q = 0; q < 5; ++q) B[e][q] -= f.E[e] * r[q];
  }
  // viscous flux
  const auto qc = [&] {
    if constexpr (J && O4) return jvals_o4(ind, 0);
    else if constexpr (J) return jvals_o2(ind, 0);
    else if constexpr (O4) return ivals_o4(ind, 0);
    else return ivals_o2(ind, 0);
  }();
  constexpr double cm = mid_coef<J, O4>(SI, SJ);
  constexpr double tt = Coef::twothird;
  const Contour& k = f.c;
  const double cx = (qc.N * k.nxN + qc.S * k.nxS + qc.O * k.nxO + qc.E * k.nxE) * k.vf;
  const double cy = (qc.N * k.nyN + qc.S * k.nyS + qc.O * k.nyO + qc.E * k.nyE) * k.vf;
  const double xx = f.nx * cx, yy = f.ny * cy, xy = f.nx * cy, yx = f.ny * cx;
  const double v1u = f.mmu * (2.0 * tt * xx + yy), v1v = f.mmu * (yx - tt * xy);
  const double v2u = f.mmu * (xy - tt * yx), v2v = f.mmu * (xx + 2.0 * tt * yy);
  const double vn = f.mmu * (xx + yy);
  const double v4t = f.lam * (xx + yy);
  double v4u = f.uu * v1u + f.vv * v2u, v4v = f.uu * v1v + f.vv * v2v, v4w = f.ww * vn;
  if constexpr (cm != 0.0) {
    const double cmu = cm * f.mmu;
    v4u += cmu * f.s1, v4v += cmu * f.s2, v4w += cmu * f.s3;
    // through mu
    const double m0 = cm * dmu, cpp = ph.cp / ph.prandtl;
    const double m1 = m0 * f.s1, m2 = m0 * f.s2, m3 = m0 * f.s3;
    const double m4 = m0 * cpp * f.s4 + f.uu * m1 + f.vv * m2 + f.ww * m3;
#pragma unroll
    for (int q = 0; q < 5; ++q) {
      B[1][q] -= m1 * dt[q];
      B[2][q] -= m2 * dt[q];
      B[3][q] -= m3 * dt[q];
      B[4][q] -= m4 * dt[q];
    }
  }
  B[1][0] -= v1u * du0 + v1v * dv0;
  B[1][1] -= v1u * rm;
  B[1][2] -= v1v * rm;
  B[2][0] -= v2u * du0 + v2v * dv0;
  B[2][1] -= v2u * rm;
  B[2][2] -= v2v * rm;
  B[3][0] -= vn * dw0;
  B[3][3] -= vn * rm;
  B[4][0] -= v4u * du0 + v4v * dv0 + v4w * dw0 + v4t * dt[0];
  B[4][1] -= v4u * rm + v4t * dt[1];
  B[4][2] -= v4v * rm + v4t * dt[2];
  B[4][3] -= v4w * rm + v4t * dt[3];
  B[4][4] -= v4t * dt[4];
#pragma unroll
  for (int e = 0; e < 5; ++e)
#pragma unroll
    for (int q = 0; q < 5; ++q) out[(e * 5 + q) * nf] = B[e][q];
}

// One thread per face of rows [j0, j1]: J = false i-faces (O4: rows j >= 3, the
// compact viscous flux; else rows 1, 2), J = true j-faces (ROW 0: rows j >= 4,
// ROW 3, 2: the off-centred rows; O4 all but row 2).  The two extra offsets
// (ioff_live, joff_live) are stored where they exist.
template <bool J, bool O4, int ROW>
__global__ void __launch_bounds__(256) k_face_blocks(Mesh m, Phys ph, Metric g, const double* __restrict__ w,
                                                     const double* __restrict__ prim,
                                                     const double* __restrict__ grad,
                                                     const double* __restrict__ cellx, double* __restrict__ out,
                                                     int j0, int j1) {
  int bx, by;
  xcd_block(bx, by);
  const int i = 1 + bx * (int)blockDim.x + (int)threadIdx.x;
  const int j = j0 + by * blockDim.y + threadIdx.y;
  if (i > (J ? m.im : m.im + 1) || j > j1) return;
  const long nf = J ? (long)m.im * (m.jm + 1) : (long)(m.im + 1) * m.jm;
  double* o0 = out + (J ? (i - 1) + (long)m.im * (j - 1) : (i - 1) + (long)(m.im + 1) * (j - 1));
  PlainAcc<double> a;
  a.m = m; a.ph = ph; a.g = g; a.i = i; a.j = j;
  a.w = w; a.prim = prim; a.grad = grad;
  FaceLin f;
  face_linearise<J, O4>(a, f);
  sfor<0, NOFF>([&](auto O) {
    constexpr int o = decltype(O)::value;
    constexpr int SI = J ? joff_di(o) : ioff_di(o), SJ = J ? joff_dj(o) : ioff_dj(o);
    if constexpr (o >= 22) {
      if (!(J ? joff_live(m, o, j) : ioff_live(m, o, i))) return;
    }
    face_block<J, O4, ROW, SI, SJ>(a, f, cellx, o0 + (long)o * 25 * nf, nf);
    // one offset at a time: the scheduler would otherwise hoist every
    // offset's loads to the top, far beyond the register file
    __builtin_amdgcn_sched_barrier(0);
  });
}

}  // namespace bca
