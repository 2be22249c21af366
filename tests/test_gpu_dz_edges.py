"""The colored spanwise operators where their two kernels meet (the two cells next
to each edge, the others): one inner cell, one and two launches' worth of i, and a
state with a spanwise velocity.  Against the oracle's seed loop, bounds as for the
larger meshes: 1e-12 of a row's largest value, indices equal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("im,jm", [(5, 5), (6, 9), (11, 5), (68, 6), (69, 8)])
def test_dz_colored_edges(im, jm):
    import oracle
    from oracle import driver as D
    from broadcast_amd.cases import bl_case
    from broadcast_amd.flow import Flow, to_device

    print(f"{im}x{jm}", flush=True)
    O = oracle.Oracle()
    case = bl_case(im, jm, seed=im, noise=1e-2)
    case.w[..., 3] += 0.05 * case.w[..., 0]
    g = D.geometry(O, case)
    w = np.array(case.w, order="F", copy=True)
    D.apply_bcs(O, case, g, w)
    jdz_o, jdz2_o, ia_o, ja_o = D.dz_colored(O, case, g, w)
    f = Flow(case)
    wg = to_device(case.w)
    f.apply_bcs(wg)
    jdz, jdz2, ia, ja = (x.cpu().numpy() for x in f.dz_colored(wg))
    np.testing.assert_array_equal(ia, ia_o)
    np.testing.assert_array_equal(ja, ja_o)
    for got, ref in ((jdz, jdz_o), (jdz2, jdz2_o)):
        rowmax = np.zeros(5 * im * jm)
        np.maximum.at(rowmax, ia_o, np.abs(ref))
        assert (np.abs(got - ref) <= 1e-12 * np.maximum(rowmax[ia_o], 1e-300)).all()
