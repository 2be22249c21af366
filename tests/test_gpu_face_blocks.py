"""The Jacobian's face blocks (hand-derived forward differentiation, all 24
offsets of a face in one thread) through the CSR product against the tangent
routine (bca_jvp, the scheme on dual numbers): -J v = dR/dw . v with the
linearised boundary conditions, on meshes at the edges of the launch (one block
row, 64 and 65 faces a row, the smallest j ranges of each face variant), with the
shock sensor on and off.

Tolerance: both sum the same ~150 products per row with different roundings;
each product carries at most ~30 roundings, so 1e-12 of the largest value leaves
two orders (the bound the parity tests use)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,im,jm", [("bl", 14, 8), ("bl", 63, 9), ("bl", 64, 12), ("bl", 65, 17), ("cyl", 14, 10),
                                        ("cyl", 64, 9), ("cyl", 71, 23)])
@pytest.mark.parametrize("k2", [0.0, 1.01])
def test_face_blocks_match_the_tangent(kind, im, jm, k2):
    import torch as t
    from broadcast_amd.cases import bl_case, cylinder_case
    from broadcast_amd.flow import Flow, to_device

    print(f"{kind} {im}x{jm} k2 {k2}", flush=True)
    case = (bl_case(im, jm, seed=im, k2=k2, noise=1e-2) if kind == "bl"
            else cylinder_case(im, jm, seed=im, k2=k2, mach=0.3, noise=1e-2))
    f = Flow(case)
    w = to_device(case.w)
    f.apply_bcs(w)
    indptr, indices, data = f.jacobian_csr(w)
    n = 5 * im * jm
    v = np.random.default_rng(im * jm).standard_normal((im, jm, 5))
    wd = np.zeros(f.shape_w, order="F")
    wd[3:-3, 3:-3] = v
    _, resd = f.jvp(w, to_device(wd))
    ref = resd.view(5, f.nj, f.ni)[:, 3:-3, 3:-3].permute(2, 1, 0).reshape(-1)
    A = t.sparse_csr_tensor(indptr.long(), indices.long(), data, size=(n, n))
    got = -(A @ t.from_numpy(v.reshape(-1)).cuda())
    err = (got - ref).view(im, jm, 5).abs().amax((0, 1)) / ref.view(im, jm, 5).abs().amax((0, 1))
    assert float(err.max()) < 1e-12, err
