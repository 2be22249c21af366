"""The residual's adjoint at the edges of its 16 x 16 face tiles: the smallest
mesh, a last tile of one face or one row, several tiles; both kinds of mesh, the
sensor on and off.  Against the oracle's transposed tangent, and twice the same
bits.

Tolerance 1e-12 of the largest value of a variable, the adjoint tests' bound (the
same ~300 products a cell in another order, ~30 roundings each)."""
import numpy as np
import pytest

from golden_util import close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,im,jm", [("bl", 5, 5), ("bl", 15, 18), ("cyl", 16, 19), ("bl", 31, 17), ("cyl", 33, 8)])
@pytest.mark.parametrize("k2", [0.0, 1.01])
def test_adjoint_tiles(kind, im, jm, k2):
    import oracle
    from oracle import driver as D
    from broadcast_amd.cases import bl_case, cylinder_case
    from broadcast_amd.flow import Flow, to_device, to_host

    print(f"{kind} {im}x{jm} k2 {k2}", flush=True)
    case = (bl_case(im, jm, seed=im, k2=k2, noise=1e-2) if kind == "bl"
            else cylinder_case(im, jm, seed=im, k2=k2, mach=0.3, r1=5.0, dr1=0.05, noise=1e-2))
    O = oracle.Oracle()
    g = D.geometry(O, case)
    f = Flow(case)
    w = to_device(case.w)
    f.apply_bcs(w)
    rb = np.zeros(f.shape_w, order="F")
    rb[3:-3, 3:-3] = np.random.default_rng(im).standard_normal((im, jm, 5))
    ref = D.vjp(O, case, g, to_host(w, f.shape_w), rb)
    got = f.vjp(w, to_device(rb))
    a = to_host(got, f.shape_w).copy()
    ok, err = close(a, ref, 1e-12)
    assert ok, err
    assert np.array_equal(a, to_host(f.vjp(w, to_device(rb)), f.shape_w))
