// Stencil offsets of the face families, and the kernel of the wall faces'
// blocks B(face, o) = d hn(face) / d w(face + o), by compile-time sparse
// forward mode (SeededAcc; the other faces: fwdface.h).  Two outputs:
//   MODE_BLOCKS  the blocks themselves (phase 1 of the colored assembly);
//   MODE_VJP     hnb(face)^T B(face, o), 5 values per offset, with hnb the
//                face adjoint of residub (the VJP, gathered per cell later).
// Templates only, instantiated in objects of their own (blocks.hip).
#pragma once
#include "faces.h"

namespace bca {

constexpr int NOFF = 24;  // stencil offsets per face family

// i-face (between cells (i-1, j) and (i, j)) stencil, offsets from (i, j):
// row 0: -3..2, rows -2, -1, 1, 2: -2..1, plus (3, 0) and (-4, 0) reached only
// through the extrapolated ghost gradients of the faces i = 1 and i = im+1.
__host__ __device__ constexpr int ioff_di(int o) {
  return o < 6 ? o - 3 : o < 22 ? ((o - 6) % 4) - 2 : (o == 22 ? 3 : -4);
}
__host__ __device__ constexpr int ioff_dj(int o) {
  return o < 6 ? 0 : o < 22 ? ((o - 6) / 4 < 2 ? (o - 6) / 4 - 2 : (o - 6) / 4 - 1) : 0;
}
// j-face (between (i, j-1) and (i, j)): transpose of the above, plus (0, 3)
// (the off-centred Euler flux of row 2) and (0, -4) (ghost gradients of row
// jm+1).
__host__ __device__ constexpr int joff_di(int o) { return ioff_dj(o); }
__host__ __device__ constexpr int joff_dj(int o) { return ioff_di(o); }

// offset -> index lookups (-1: not in the stencil); i-face table over
// di in [-4, 3] x dj in [-2, 2], j-face table over di in [-2, 2] x dj in [-4, 3]
__host__ __device__ inline int ioff_index(int di, int dj) {
  if (dj == 0) {
    if (di >= -3 && di <= 2) return di + 3;
    if (di == 3) return 22;
    if (di == -4) return 23;
    return -1;
  }
  if (dj < -2 || dj > 2 || di < -2 || di > 1) return -1;
  const int r = dj < 0 ? dj + 2 : dj + 1;  // -2,-1,1,2 -> 0,1,2,3
  return 6 + r * 4 + (di + 2);
}
__host__ __device__ inline int joff_index(int di, int dj) { return ioff_index(dj, di); }

// is offset index o of a face at (fi, fj) a stored block?  (the two extra
// offsets exist only on the faces listed in the phase-1 kernels)
__host__ __device__ inline bool ioff_live(const Mesh& m, int o, int fi) {
  return o < 22 || (o == 22 && fi == 1) || (o == 23 && fi == m.im + 1);
}
__host__ __device__ inline bool joff_live(const Mesh& m, int o, int fj) {
  return o < 22 || (o == 22 && fj == 2) || (o == 23 && fj == m.jm + 1);
}

// compact index of a ghost-frame cell given storage coordinates (a, b)
__host__ __device__ inline long ghost_index(const Mesh& m, int a, int b) {
  const int gh = m.gh;
  if (b < gh) return (long)b * m.ni + a;
  if (b >= gh + m.jm) return (long)gh * m.ni + (long)(b - gh - m.jm) * m.ni + a;
  return 2L * gh * m.ni + (long)(b - gh) * 2 * gh + (a < gh ? a : a - m.im);
}
__host__ __device__ inline long ghost_count(const Mesh& m) {
  return 2L * m.gh * m.ni + 2L * m.gh * m.jm;
}

// ------------------------------------------------------------------ phase 1
enum { MODE_BLOCKS = 0, MODE_VJP = 1 };

template <int SI, int SJ>
__device__ inline SeededAcc<SI, SJ> seeded(const Mesh& m, const Phys& ph, const Metric& g,
                                           const double* w, const double* prim, const double* grad,
                                           int i, int j) {
  SeededAcc<SI, SJ> a;
  a.m = m; a.ph = ph; a.g = g; a.i = i; a.j = j;
  a.w = w; a.prim = prim; a.grad = grad;
  a.seed();
  return a;
}

// Output of the seeded pass of offset o at face f.  MODE_BLOCKS: B(face, o)
// in plane o, out[(o * 25 + e * 5 + q) * nf + f]; MODE_VJP: sum_e hb[e]
// B(face, o)[e][q] in out[(o * 5 + q) * nf + f].  Either way a wave
// (consecutive faces, one offset) stores coalesced rows.
template <int MODE>
struct FaceSink {
  double* out;
  long nf, f;
  double hb[5];
  __device__ void put(int o, const Dual<5> hn[5]) const {
    if constexpr (MODE == MODE_BLOCKS) {
      double* p = out + (long)o * 25 * nf + f;
#pragma unroll
      for (int e = 0; e < 5; ++e)
#pragma unroll
        for (int q = 0; q < 5; ++q) p[(e * 5 + q) * nf] = hn[e].d[q];
    } else {
      double* p = out + (long)o * 5 * nf + f;
#pragma unroll
      for (int q = 0; q < 5; ++q) {
        double t = 0.0;
#pragma unroll
        for (int e = 0; e < 5; ++e) t += hb[e] * hn[e].d[q];
        p[q * nf] = t;
      }
    }
  }
};

// Face adjoints of the balance R(i,j) = hn(i) - hn(i+1) + hn(j) - hn(j+1) over
// the interior rows (srcfv/adjoint/flux_num_dnc5_b.f90:800-829).
__device__ inline void face_adjoint(const Mesh& m, const double* resb, int i, int j, int di, int dj,
                                    double hb[5]) {
  const bool lo = (i - di) >= 1 && (j - dj) >= 1, hi = i <= m.im && j <= m.jm;
#pragma unroll
  for (int e = 0; e < 5; ++e) {
    double v = 0.0;
    if (hi) v += resb[cidx(m, i, j) + (long)e * m.ncell];
    if (lo) v -= resb[cidx(m, i - di, j - dj) + (long)e * m.ncell];
    hb[e] = v;
  }
}

// Wall faces (i, 1) (adiabatic no-slip, fluxwall.F): they depend on the cells
// (0, 0) and (0, 1) only; the other blocks are stored as explicit zeros where
// the assembly may look for them.
template <int MODE>
__global__ void __launch_bounds__(256) k_jface_wall_blocks(Mesh m, Phys ph, Metric g, const double* __restrict__ w,
                                                           const double* __restrict__ prim,
                                                           const double* __restrict__ grad,
                                                           double* __restrict__ out,
                                                           const double* __restrict__ resb, int j0, int j1) {
  const int i = 1 + blockIdx.x * (int)blockDim.x + (int)threadIdx.x;
  const int j = j0 + blockIdx.y * blockDim.y + threadIdx.y;
  if (i > m.im || j > j1) return;
  const long nf = (long)m.im * (m.jm + 1);
  FaceSink<MODE> sink{out, nf, (i - 1) + (long)m.im * (j - 1), {}};
  if constexpr (MODE == MODE_VJP) face_adjoint(m, resb, i, j, 0, 1, sink.hb);
  sfor<0, 22>([&](auto O) {
    constexpr int o = decltype(O)::value;
    constexpr int SI = joff_di(o), SJ = joff_dj(o);
    Dual<5> hn[5];
    if constexpr (SI == 0 && (SJ == 0 || SJ == 1)) {
      auto a = seeded<SI, SJ>(m, ph, g, w, prim, grad, i, j);
      jface_wall(a, hn);
    }
    sink.put(o, hn);
  });
}

}  // namespace bca
