// One family of face kernels per compilation (selected by BCA_VARIANT): their
// per-offset code is large, so the build compiles the variants as separate
// objects in parallel.  Variants 0-3 store Jacobian blocks, 4 those of the wall
// faces and their VJP contributions, 5 the reverse-mode face adjoints.
#include <hip/hip_runtime.h>

#include "adjface.h"
#include "blocks.h"
#include "blockskern.h"
#include "fwdface.h"

namespace bca {

#define BCA_BLOCKS(name, ...)                                                                                \
  void name(dim3 gr, dim3 bl, hipStream_t s, const BlockArgs& a) {                                            \
    k_face_blocks<__VA_ARGS__><<<gr, bl, 0, s>>>(a.m, a.ph, a.g, a.w, a.prim, a.grad, a.cellx, a.out, a.j0, a.j1); \
  }
#define BCA_LAUNCH(name, kern, ...)                                                                          \
  void name(dim3 gr, dim3 bl, hipStream_t s, const BlockArgs& a) {                                            \
    kern<__VA_ARGS__><<<gr, bl, 0, s>>>(a.m, a.ph, a.g, a.w, a.prim, a.grad, a.out, a.resb, a.j0, a.j1);      \
  }

#if BCA_VARIANT == 0
BCA_BLOCKS(launch_iface_blocks_o4, false, true, 0)
#elif BCA_VARIANT == 1
BCA_BLOCKS(launch_iface_blocks_o2, false, false, 0)
BCA_BLOCKS(launch_jface_blocks_r2, true, false, 2)
#elif BCA_VARIANT == 2
BCA_BLOCKS(launch_jface_blocks_c, true, true, 0)
#elif BCA_VARIANT == 3
BCA_BLOCKS(launch_jface_blocks_r3, true, true, 3)
#elif BCA_VARIANT == 4
BCA_LAUNCH(launch_jface_blocks_wall, k_jface_wall_blocks, MODE_BLOCKS)
BCA_LAUNCH(launch_jface_vjp_wall, k_jface_wall_blocks, MODE_VJP)
#elif BCA_VARIANT == 5
BCA_LAUNCH(launch_iface_vjp_rev, k_face_reverse, false, true, 0)
BCA_LAUNCH(launch_iface_vjp_rev_o2, k_face_reverse, false, false, 0)
BCA_LAUNCH(launch_jface_vjp_rev, k_face_reverse, true, true, 0)
BCA_LAUNCH(launch_jface_vjp_rev_r3, k_face_reverse, true, true, 3)
BCA_LAUNCH(launch_jface_vjp_rev_r2, k_face_reverse, true, false, 2)
#else
#error "BCA_VARIANT must be 0..5"
#endif

}  // namespace bca
