// Adjoint (reverse mode) of the ghost-filling boundary conditions, as the
// TAPENADE _b routines of the reference (srcfv/adjoint/bc_supandsubinlet_b.f90,
// bc_no_reflexion_b.f90, bc_extrapolateo2_b.f90, bc_wall_viscous_b.f90,
// jn_match_2d_b.f90): on exit wb(ghosts of the BC) = 0 and every cell the BC
// reads has received (d ghosts / d cell)^T wb(ghosts); w is left as given.
//
// A BC line reads the cells at offsets 0..3 along its inward normal and writes
// its gh ghost layers (deeper layers may read the ones before, which the
// forward-mode line function composes).  So the transpose is formed from the
// tangent line functions: for each offset d, a unit Dual<5> tangent on the
// offset-d cell of the line, the tangent BC applied, and the ghost tangents
// contracted with wb(ghosts) as they are formed: a thread per line and offset,
// nothing of the seeded states in memory.
//
// What bounds it: one thread's chain of Dual<5> operations (an inlet line ~10 us).
// Seeding frames, the BC on them, the contraction and the clearing took four
// launches per operation: adjoint 1024 x 256 662 -> 491 us, 127 x 93 O-mesh 191 ->
// 157 us (the flux adjoint included).
#pragma once
#include "bcs.h"

namespace bca {

constexpr int ADJ_REACH = 4;  // offsets 0..3 along the inward normal

__device__ inline void line_cell(int loc, Box b, int l, int& i, int& j, int& i0, int& j0) {
  const Side s = decode_side(loc, b.imin, b.jmin, b.imax, b.jmax);
  i = b.imin + (l - 1) * s.j0 * s.j0;
  j = b.jmin + (l - 1) * s.i0 * s.i0;
  i0 = s.i0;
  j0 = s.j0;
}

// The state with a unit tangent d[e] on variable e of the cell (ci, cj); what a
// line writes to a ghost is contracted with wb there: acc[q] += d ghost / d w_q wb.
struct AdjView {
  using Scalar = Dual<5>;
  Mesh m;
  const double* w;
  const double* wb;
  int ci, cj;
  double* acc;
  __device__ Dual<5> operator()(int i, int j, int e) const {
    Dual<5> x(w[cidx(m, i, j) + (long)e * m.ncell]);
    const double one = i == ci && j == cj ? 1.0 : 0.0;
#pragma unroll
    for (int q = 0; q < 5; ++q) x.d[q] = q == e ? one : 0.0;
    return x;
  }
  __device__ void put(int i, int j, int e, const Dual<5>& x) const {
    const double y = wb[cidx(m, i, j) + (long)e * m.ncell];
#pragma unroll
    for (int q = 0; q < 5; ++q) acc[q] += x.d[q] * y;
  }
};

constexpr int ADJ_LINES = 64 / ADJ_REACH;  // lines per workgroup (one wave)

// One BC operation: wb(offset-d cell, q) += sum over the line's ghosts g and
// variables e of d ghost(g, e) / d w(offset-d cell, q) wb(g, e), then the line's
// wb(g) = 0.  A line's offset-d cells and ghosts are its own, so only the lanes
// of one line have to wait for each other before its ghosts are cleared.
template <int KIND>
__global__ void __launch_bounds__(64) k_bc_adjoint(Mesh m, const double* __restrict__ w, double* __restrict__ wb,
                                                   BcSeqOp q, const double* __restrict__ nx,
                                                   const double* __restrict__ ny, int lmax) {
  const int l = 1 + blockIdx.x * ADJ_LINES + threadIdx.x % ADJ_LINES, d = threadIdx.x / ADJ_LINES;
  int i, j, i0, j0;
  line_cell(q.loc, q.box, l, i, j, i0, j0);
  if (l <= lmax) {
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    const AdjView v{m, w, wb, i + d * i0, j + d * j0, acc};
    if constexpr (KIND == SEQ_INLET) bc_inlet_line(v, q.loc, q.box, q.data, q.lm, nx, ny, q.gam, l);
    else if constexpr (KIND == SEQ_NOREF) bc_noref_line(v, q.data, q.lm, q.loc, q.box, nx, ny, q.gam, l);
    else if constexpr (KIND == SEQ_EXTRAP2) bc_extrap2_line(v, q.loc, q.box, 5, l);
    else bc_wall_line(v, q.loc, q.box, q.gam, l);
    const long s = cidx(m, i + d * i0, j + d * j0);
#pragma unroll
    for (int e = 0; e < 5; ++e) wb[s + e * m.ncell] += acc[e];
  }
  __syncthreads();
  if (l <= lmax)
    for (int de = d + 1; de <= m.gh; de += ADJ_REACH)
#pragma unroll
      for (int e = 0; e < 5; ++e) wb[cidx(m, i - de * i0, j - de * j0) + e * m.ncell] = 0.0;
}

// In-block join (identity transform, disjoint boxes): the copy wb(prr) <-
// wb(prd) transposed, wb(prd cell) += wb(prr cell), then wb(prr cell) = 0.
__global__ void k_join_adjoint(Mesh m, double* __restrict__ wb, Box prr, Box prd, int em) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int ni_ = prd.imax - prd.imin + 1, nj_ = prd.jmax - prd.jmin + 1;
  if (t >= ni_ * nj_) return;
  const int a = t % ni_, q = t / ni_;
  const long dst = cidx(m, prr.imin + a, prr.jmin + q), src = cidx(m, prd.imin + a, prd.jmin + q);
  for (int e = 0; e < em; ++e) {
    wb[src + e * m.ncell] += wb[dst + e * m.ncell];
    wb[dst + e * m.ncell] = 0.0;
  }
}

}  // namespace bca
