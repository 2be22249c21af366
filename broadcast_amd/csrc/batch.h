// Residual (+ JVP) of a batch of meshes of different sizes, one launch per
// stage over all meshes.
//
// Per mesh this is the reference's per-iteration sequence -- the BC calls in
// order (BROADCAST_npz.py:1018-1021 primal, :1079-1082 tangent) then
// flux_num_dnc5_2d[_d] (srcfv/rhs/flux_num_dnc5.F90:7-226,
// srcfv/tangent/flux_num_dnc5_d.f90:15) -- with the same device functions as
// the per-mesh kernels.  A batch of small and uneven meshes would leave most
// of the chip idle under launches of its own per mesh; here the workgroups of
// all meshes make one grid (the mesh of a workgroup found in the stage's prefix
// table):
//
//   bc        k_bc_sequence's workgroups of every mesh (or, where a sequence is
//             not one of its kind, the k-th operation of every mesh in turn)
//   residual  k_residual's tiles of every mesh
//   store     only where an output shares memory with an input: the interiors,
//             from scratch
//
// What bounds it is what bounds k_residual.  Eight meshes of 128..1024 x
// 64..256 with their tangents: 393 -> 176 us (11 launches before).
#pragma once
#include "residual.h"

namespace bca {

constexpr int BATCH_MAX = 16;  // meshes per launch
constexpr int BATCH_OPS = 8;   // BC operations per mesh

struct BatchItem {
  Mesh m;
  ResPhys ph;
  Metric g;
  double* w;      // state, ghost frame filled in place
  double* wd;     // tangent, ghost frame filled in place (null: residual only)
  ResOut out;     // residu, residud or their place in scratch
  ResOut store;   // residu, residud
  BcSeq seq;
  int nops;
  BcSeqOp ops[BATCH_OPS];
};

// Prefix sums of each stage's workgroups (bc: lines) over the meshes.
struct BatchPlan {
  int n;
  int seq[BATCH_MAX + 1];
  int tiles[BATCH_MAX + 1];
  int cells[BATCH_MAX + 1];
  int bc[BATCH_OPS][BATCH_MAX + 1];
};

// mesh of flat item t (pre[0] = 0 <= t < pre[n]); n is small, a linear walk
__device__ inline int batch_which(const int* pre, int n, int t) {
  int k = 0;
  while (k + 1 < n && t >= pre[k + 1]) ++k;
  return k;
}

template <class V>
__device__ inline V batch_view(const BatchItem& it) {
  if constexpr (std::is_same<V, PairView>::value) return PairView{it.m, it.w, it.wd};
  else return V(it.m, it.w);
}

template <class V>
__global__ void __launch_bounds__(BC_SEQ_THREADS) k_batch_bc_sequence(const BatchItem* __restrict__ items,
                                                                      const BatchPlan* __restrict__ plan) {
  const int k = batch_which(plan->seq, plan->n, blockIdx.x);
  const BatchItem& it = items[k];
  bc_sequence(batch_view<V>(it), it.seq, it.g.nx, it.g.ny, (int)blockIdx.x - plan->seq[k]);
}

// operation `op` of every mesh: lines, or cells of a join
template <class V>
__global__ void __launch_bounds__(256) k_batch_bc(const BatchItem* __restrict__ items,
                                                  const BatchPlan* __restrict__ plan, int op) {
  const int* pre = plan->bc[op];
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= pre[plan->n]) return;
  const int k = batch_which(pre, plan->n, t);
  const BatchItem& it = items[k];
  const BcSeqOp& q = it.ops[op];
  int lo, hi;
  bc_seq_range(q, lo, hi);
  const int wd = bc_seq_width(q), x = t - pre[k];
  bc_seq_line(batch_view<V>(it), q, it.g.nx, it.g.ny, lo + x / wd, x % wd);
}

template <class V>
__global__ void __launch_bounds__(TILE_THREADS, sizeof(typename V::Scalar) > 8 ? 2 : 4)
    k_batch_residual(const BatchItem* __restrict__ items, const BatchPlan* __restrict__ plan) {
  using TL = Tile<typename V::Scalar, 5>;
  __shared__ __align__(16) unsigned char mem[sizeof(TL)];
  TL& s = *reinterpret_cast<TL*>(mem);
  int t, zero;
  xcd_block(t, zero);
  const int k = batch_which(plan->tiles, plan->n, t);
  const BatchItem& it = items[k];
  t -= plan->tiles[k];
  const int nbx = (it.m.im + TILE_CELLS - 1) / TILE_CELLS, bx = t % nbx, by = t / nbx;
  const V w = batch_view<V>(it);
  if (by == 0) residual_tile<V, 5, false, true>(s, w, it.ph, it.g, it.out, bx, by);
  else residual_tile<V, 5, false, false>(s, w, it.ph, it.g, it.out, bx, by);
}

__global__ void __launch_bounds__(256) k_batch_store(const BatchItem* __restrict__ items,
                                                     const BatchPlan* __restrict__ plan) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= plan->cells[plan->n]) return;
  const int k = batch_which(plan->cells, plan->n, t);
  const BatchItem& it = items[k];
  const int q = t - plan->cells[k];
  const long c = cidx(it.m, 1 + q % it.m.im, 1 + q / it.m.im);
#pragma unroll
  for (int e = 0; e < 5; ++e) {
    const long ce = c + (long)e * it.m.ncell;
    it.store.res[ce] = it.out.res[ce];
    if (it.wd) it.store.resd[ce] = it.out.resd[ce];
  }
}

}  // namespace bca
