// Cell gather of the residual VJP.  The face kernels leave, per tile of faces,
// what its stencil cells receive (RevTile); the wall faces' kernel leaves 5 values
// per offset in planes.  The adjoint of a cell is the sum over the tiles that hold
// it (at most four of a family) in a fixed order, its primitives' part taken back
// to the state, plus the wall face's.
#pragma once
#include "adjface.h"

namespace bca {

// The tiles of one launch of k_face_reverse.
struct RevSet {
  const double* part;
  int j0, nbx, nby;
};
struct RevSets {
  RevSet i[2], j[3];  // i-faces: rows >= 3, rows 1 and 2; j-faces: rows >= 4, row 3, row 2
};
__host__ __device__ inline long rev_doubles(const RevSet& s) { return (long)s.nbx * s.nby * REV_N; }

template <bool J>
__device__ inline void rev_add(const RevSet& s, int ci, int cj, double pb[NPRIM], double wb[5]) {
  using R = RevTile<J>;
  const int bh = (ci - 1 + R::C4) >> 4, rh = (cj - s.j0 + R::R4) >> 4;
  for (int by = rh - 1; by <= rh; ++by) {
    const int r = cj - s.j0 - by * REV;
    if (by < 0 || by >= s.nby || r + R::R4 >= R::H4) continue;
    for (int bx = bh - 1; bx <= bh; ++bx) {
      const int c = ci - 1 - bx * REV;
      if (bx < 0 || bx >= s.nbx || c + R::C4 >= R::W4) continue;
      const double* p = s.part + (long)(bx + by * s.nbx) * REV_N;
      const double* a = p + (r + R::R4) * R::W4 + c + R::C4;
      constexpr int s4 = R::W4 * R::H4, s8 = R::W8 * R::H8;
      pb[P_U] += a[0];
      pb[P_V] += a[s4];
      pb[P_W] += a[2 * s4];
      pb[P_T] += a[3 * s4];
      const int r8 = r + R::R8, c8 = c + R::C8;
      if (r8 < 0 || r8 >= R::H8 || c8 < 0 || c8 >= R::W8) continue;
      const double* q = p + R::N4 + r8 * R::W8 + c8;
#pragma unroll
      for (int e = 0; e < 5; ++e) wb[e] += q[e * s8];
      pb[P_P] += q[5 * s8];
      pb[P_MU] += q[6 * s8];
      pb[P_H] += q[7 * s8];
    }
  }
}

// Grid over the whole array (ghost frame included): wb is overwritten
// everywhere, as the reference zeroes it before accumulating
// (srcfv/adjoint/flux_num_dnc5_b.f90:834).
__global__ void __launch_bounds__(256) k_vjp_gather(Mesh m, Phys ph, const double* w, RevSets sets,
                                                    const double* __restrict__ cj, double* wb) {
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  const int b = blockIdx.y * blockDim.y + threadIdx.y;
  if (a >= m.ni || b >= m.nj) return;
  const int i = a - m.gh + 1, j = b - m.gh + 1;
  const long c = a + (long)m.ni * b;
  double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, pb[NPRIM];
#pragma unroll
  for (int k = 0; k < NPRIM; ++k) pb[k] = 0.0;
  rev_add<false>(sets.i[0], i, j, pb, acc);
  rev_add<true>(sets.j[0], i, j, pb, acc);
  if (j <= 8) {
    rev_add<false>(sets.i[1], i, j, pb, acc);
    rev_add<true>(sets.j[1], i, j, pb, acc);
    rev_add<true>(sets.j[2], i, j, pb, acc);
  }
  bool any = false;
#pragma unroll
  for (int k = 0; k < NPRIM; ++k) any = any || pb[k] != 0.0;
  // (a ghost that no face reads may hold anything)
  if (any) {
    double wc[5];
#pragma unroll
    for (int q = 0; q < 5; ++q) wc[q] = w[c + (long)q * m.ncell];
    const double cvm1 = 1.0 / ph.cv;
    const double betas = ph.muref * (ph.tref + ph.cs) / (sqrt(ph.tref) * ph.tref);
    prim_reverse(ph, cvm1, betas, wc, cell_prim(ph, cvm1, wc), pb, acc);
  }
  // the wall face (i, 1): cells j = 1, 2
  if (i >= 1 && i <= m.im && (j == 1 || j == 2)) {
    const long nfj = (long)m.im * (m.jm + 1);
    const double* p = cj + (long)(j == 1 ? joff_index(0, 0) : joff_index(0, 1)) * 5 * nfj + (i - 1);
#pragma unroll
    for (int q = 0; q < 5; ++q) acc[q] += p[q * nfj];
  }
#pragma unroll
  for (int q = 0; q < 5; ++q) wb[c + q * m.ncell] = acc[q];
}

// residub is consumed: its interior is zeroed after use
// (srcfv/adjoint/flux_num_dnc5_b.f90:809-829).
__global__ void k_zero_interior(Mesh m, double* __restrict__ r) {
  const int i = 1 + blockIdx.x * blockDim.x + threadIdx.x;
  const int j = 1 + blockIdx.y * blockDim.y + threadIdx.y;
  if (i > m.im || j > m.jm) return;
  const long c = cidx(m, i, j);
#pragma unroll
  for (int e = 0; e < 5; ++e) r[c + e * m.ncell] = 0.0;
}

}  // namespace bca
