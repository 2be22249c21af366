// Host launchers of the face-block kernels (each compiled in its own object).
#pragma once
#include <hip/hip_runtime.h>

#include "scheme.h"

namespace bca {

// Planes of BlockArgs::cellx: 1 / rho and d mu / d T of every cell (k_cellx),
// for the blocks' d prim / d w.
enum { X_RM = 0, X_DMU, NCELLX };

struct BlockArgs {
  Mesh m;
  Phys ph;
  Metric g;
  const double* w;
  const double* prim;
  const double* grad;
  double* out;          // blocks (25 planes per offset) or VJP contributions (5)
  const double* resb;   // residual adjoint (VJP only)
  int j0, j1;
  const double* cellx;  // 1 / rho and d mu / d T (blocks only)
};

void launch_iface_blocks_o4(dim3 gr, dim3 bl, hipStream_t s, const BlockArgs& a);
void launch_iface_blocks_o2(dim3 gr, dim3 bl, hipStream_t s, const BlockArgs& a);
void launch_jface_blocks_c(dim3 gr, dim3 bl, hipStream_t s, const BlockArgs& a);
void launch_jface_blocks_r3(dim3 gr, dim3 bl, hipStream_t s, const BlockArgs& a);
void launch_jface_blocks_r2(dim3 gr, dim3 bl, hipStream_t s, const BlockArgs& a);
void launch_jface_blocks_wall(dim3 gr, dim3 bl, hipStream_t s, const BlockArgs& a);
void launch_jface_vjp_wall(dim3 gr, dim3 bl, hipStream_t s, const BlockArgs& a);
void launch_iface_vjp_rev(dim3 gr, dim3 bl, hipStream_t s, const BlockArgs& a);
void launch_iface_vjp_rev_o2(dim3 gr, dim3 bl, hipStream_t s, const BlockArgs& a);
void launch_jface_vjp_rev(dim3 gr, dim3 bl, hipStream_t s, const BlockArgs& a);
void launch_jface_vjp_rev_r3(dim3 gr, dim3 bl, hipStream_t s, const BlockArgs& a);
void launch_jface_vjp_rev_r2(dim3 gr, dim3 bl, hipStream_t s, const BlockArgs& a);

}  // namespace bca
