"""bca_inv_np of a block scaled by a power of two: the same bits scaled back, and
the same verdict on its pivots, whether or not the panels (32 columns) and the
pivot groups (4) come out even.  And of a block whose rows lie so far apart that a
tile of 64 rows spans more than 4 GiB: the same bits again."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


def inverse(A, ld=None):
    """The inverse of A and the flag; A in rows ld apart."""
    import torch as t
    from broadcast_amd import _lib

    n = A.shape[0]
    ld = ld or n
    A = t.zeros((n - 1) * ld + n, dtype=t.float64, device="cuda").as_strided((n, n), (ld, 1)).copy_(A)
    bad = t.zeros(1, dtype=t.int32, device="cuda")
    work = t.empty(n * n, dtype=t.float64, device="cuda")
    s = C.c_void_p(t.cuda.current_stream().cuda_stream)
    _lib.check(_lib.lib().bca_inv_np(s, C.c_void_p(A.data_ptr()), n, ld, C.c_void_p(work.data_ptr()), 1e-14,
                                     C.c_void_p(bad.data_ptr())), "bca_inv_np")
    return A, int(bad.item())


@pytest.mark.parametrize("n", [1, 2, 3, 31, 33, 40, 65, 97, 130])
@pytest.mark.parametrize("power", [53, -53, 310, -310, 700, -700])
def test_inverse_of_a_scaled_block(n, power):
    import torch as t

    A = t.randn(n, n, dtype=t.float64, device="cuda", generator=t.Generator(device="cuda").manual_seed(n))
    A += 4 * n ** 0.5 * t.eye(n, dtype=t.float64, device="cuda")
    ref, bad = inverse(A)
    assert bad == 0
    got, bad = inverse(A * 2.0 ** power)
    assert bad == 0
    assert t.equal(got * 2.0 ** power, ref)


@pytest.mark.parametrize("n,ld", [(20, 9_000_001), (70, 9_000_001)])
def test_inverse_of_a_block_with_rows_far_apart(n, ld):
    import torch as t

    assert 64 * ld * 8 >= 2 ** 32
    A = t.randn(n, n, dtype=t.float64, device="cuda", generator=t.Generator(device="cuda").manual_seed(n))
    A += 4 * n ** 0.5 * t.eye(n, dtype=t.float64, device="cuda")
    ref, bad = inverse(A)
    got, bad2 = inverse(A, ld)
    assert bad == bad2 == 0
    assert t.equal(got, ref)
