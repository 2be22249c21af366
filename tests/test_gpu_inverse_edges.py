"""bca_inv_np at the edges of its panels (32 columns), MFMA pivot groups (4) and
output tiles (64), against torch's inverse in float64.

Tolerance: Gauss-Jordan without pivoting on a diagonally heavy block (condition
below 4) commits at most n rounding errors of 2^-53 per entry; 8 n 2^-53
normwise leaves room for the reciprocals and the growth."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 4, 5, 31, 32, 33, 63, 64, 65, 96, 97, 127, 130, 335])
def test_inverse_at_panel_and_tile_edges(n):
    import torch as t
    from broadcast_amd import _lib

    print(f"n {n}", flush=True)
    g = t.Generator(device="cuda").manual_seed(n)
    A0 = t.randn(n, n, dtype=t.float64, device="cuda", generator=g) + 4 * n ** 0.5 * t.eye(n, dtype=t.float64,
                                                                                     device="cuda")
    big = t.full((n, n + 9), 7.0, dtype=t.float64, device="cuda")
    big[:, 4:4 + n] = A0
    A = big[:, 4:4 + n]
    bad = t.zeros(1, dtype=t.int32, device="cuda")
    work = t.empty(n * n, dtype=t.float64, device="cuda")
    s = C.c_void_p(t.cuda.current_stream().cuda_stream)
    _lib.check(_lib.lib().bca_inv_np(s, C.c_void_p(A.data_ptr()), n, big.stride(0), C.c_void_p(work.data_ptr()), 1e-14,
                                     C.c_void_p(bad.data_ptr())), "bca_inv_np")
    ref = t.linalg.inv(A0)
    assert int(bad.item()) == 0
    assert float((A - ref).norm() / ref.norm()) <= 8 * n * 2.0 ** -53
    assert bool((big[:, :4] == 7.0).all()) and bool((big[:, 4 + n:] == 7.0).all())


@pytest.mark.parametrize("n,where", [(40, 0), (40, 36), (97, 64)])
def test_zero_or_undefined_pivot_is_reported(n, where):
    """A zero pivot, or a NaN entry, sets the flag (no entry of the result is
    used then)."""
    import torch as t
    from broadcast_amd import _lib

    for value in (0.0, float("nan")):
        A = 4.0 * t.eye(n, dtype=t.float64, device="cuda")
        A[where, where] = value
        bad = t.zeros(1, dtype=t.int32, device="cuda")
        work = t.empty(n * n, dtype=t.float64, device="cuda")
        s = C.c_void_p(t.cuda.current_stream().cuda_stream)
        _lib.check(_lib.lib().bca_inv_np(s, C.c_void_p(A.data_ptr()), n, n, C.c_void_p(work.data_ptr()), 1e-14,
                                         C.c_void_p(bad.data_ptr())), "bca_inv_np")
        assert int(bad.item()) == 1
