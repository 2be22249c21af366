"""bca_band_factor / bca_band_solve on dense random bands against torch's dense
solve in float64: all downwards and from both ends, one stream and three, block
sizes on both sides of the kernels' tiles (32, 64) and K slices (16, 32), with
far blocks of block row 0.

Tolerance: the bands are diagonally heavy (condition below 10), so a backward
stable elimination of N unknowns solves to about N 2^-53; 4 N 2^-53 for the
growth without pivoting."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,B,kb,nfar", [(1, 20, 0, 0), (4, 33, 1, 0), (9, 15, 1, 1), (11, 64, 2, 0), (13, 65, 3, 1),
                                          (12, 97, 3, 0), (20, 160, 3, 1)])
@pytest.mark.parametrize("both", [False, True])
@pytest.mark.parametrize("streams", [1, 3])
def test_band_solve_matches_dense(nb, B, kb, nfar, both, streams):
    import torch as t
    from broadcast_amd import _lib

    mid = nb // 2 - kb if both else nb
    if both and mid < kb + nfar + 1:
        pytest.skip("too few block rows for two ends")
    print(f"nb {nb} B {B} kb {kb} nfar {nfar} mid {mid} streams {streams}", flush=True)
    g = t.Generator(device="cuda").manual_seed(nb * 1000 + B)
    n, W = nb * B, (2 * kb + 1) * B
    A = t.zeros(n, n, dtype=t.float64, device="cuda")
    R = t.zeros(nb, B, W, dtype=t.float64, device="cuda")
    F = t.zeros(B, max(nfar, 1) * B, dtype=t.float64, device="cuda")
    for K in range(nb):
        for J in range(max(0, K - kb), min(nb, K + kb + 1 + (nfar if K == 0 else 0))):
            blk = t.randn(B, B, dtype=t.float64, device="cuda", generator=g)
            if J == K:
                blk += 4 * W ** 0.5 * t.eye(B, dtype=t.float64, device="cuda")
            A[K * B:(K + 1) * B, J * B:(J + 1) * B] = blk
            if J - K <= kb:
                R[K, :, (J - K + kb) * B:(J - K + kb + 1) * B] = blk
            else:
                F[:, (J - kb - 1) * B:(J - kb) * B] = blk
    b = t.randn(n, dtype=t.float64, device="cuda", generator=g)
    ref = t.linalg.solve(A, b)
    scratch = t.empty(2 * (1 + kb + nfar) * B * B, dtype=t.float64, device="cuda")
    bad = t.zeros(1, dtype=t.int32, device="cuda")
    cur = t.cuda.current_stream()
    st = [cur, cur, cur] if streams == 1 else [cur, t.cuda.Stream(), t.cuda.Stream()]
    p = lambda a: C.c_void_p(a.data_ptr())  # noqa: E731
    L = _lib.lib()
    _lib.check(L.bca_band_factor((C.c_void_p * 3)(*[s.cuda_stream for s in st]), p(R), p(F) if nfar else None, nb, B,
                                 kb, nfar, mid, p(scratch), 1e-14, p(bad)), "bca_band_factor")
    y, z = b.clone(), t.empty_like(b)
    _lib.check(L.bca_band_solve(C.c_void_p(cur.cuda_stream), p(R), p(F) if nfar else None, nb, B, kb, nfar, mid, p(y),
                                p(z)), "bca_band_solve")
    t.cuda.synchronize()
    assert int(bad.item()) == 0
    assert float((z - ref).norm() / ref.norm()) <= 4 * n * 2.0 ** -53


def test_solve_keeps_its_matrix():
    """The solve's correction uses the matrix that was factored, also after the
    caller's CSR arrays have been rewritten."""
    import torch as t
    from broadcast_amd.cases import bl_case
    from broadcast_amd.flow import Flow, to_device
    from broadcast_amd.newton import BlockBandLU, csr_residual

    case = bl_case(40, 24, seed=5)
    f = Flow(case)
    w = to_device(case.w)
    f.apply_bcs(w)
    cd = t.full((case.im * case.jm,), 1e-3, dtype=t.float64, device="cuda")
    csr = f.jacobian_csr(w, coefdiag=cd)
    kept = tuple(a.clone() for a in csr)
    lu = BlockBandLU(case.im, case.jm).factor(*csr)
    for a in csr:
        a.zero_()
    b = t.ones(5 * case.im * case.jm, dtype=t.float64, device="cuda")
    assert float(csr_residual(kept, lu.solve(b), b).norm() / b.norm()) < 1e-12
