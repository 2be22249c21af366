"""A block row 0 that reaches beyond the band of the other rows: one block is kept
outside it; farther ones widen the band, since eliminating block 0 fills block
row 1 as far.  On CPU tensors, against a dense solve.

Tolerance: diagonally heavy matrices (condition below 10), 40 n 2^-53."""
import ctypes as C

import pytest


@pytest.mark.parametrize("reach", [1, 2, 3, 4])
@pytest.mark.parametrize("kb", [None, 1])
def test_first_block_row_reaches_farther(reach, kb):
    import torch as t
    from broadcast_amd.newton import BlockBandLU

    im, jm, B = 7, 2, 10
    n = im * B
    t.manual_seed(reach)
    k = t.arange(n) // B
    mask = (k[:, None] - k).abs() <= 1
    mask |= (k[:, None] == 0) & (k <= reach)
    A = t.randn(n, n, dtype=t.float64) * mask + 4 * (3 * B) ** 0.5 * t.eye(n, dtype=t.float64)
    c = A.to_sparse_csr()
    b = t.randn(n, dtype=t.float64)
    lu = BlockBandLU(im, jm, kb=kb).factor(c.crow_indices(), c.col_indices(), c.values())
    ref = t.linalg.solve(A, b)
    assert float((lu.solve(b) - ref).norm()) <= 40 * n * 2.0 ** -53 * float(ref.norm())
    assert lu.kb == max(1, reach - 1) and lu.nfar <= 1


def test_band_factor_refuses_two_far_blocks():
    """(checked before anything else is done with the arguments)"""
    from broadcast_amd import _lib

    p = C.c_void_p(8)
    L = _lib.lib()
    assert L.bca_band_factor((C.c_void_p * 3)(), p, p, 9, 4, 1, 2, 9, p, 1e-14, p) == -1
    assert b"beyond the band" in L.bca_last_error()
