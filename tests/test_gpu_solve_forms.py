"""BlockBandLU.solve and csr_residual take what torch takes: right-hand sides of
any stride, any integer index type.  The same kernels on the same values, so the same bits as for
contiguous int32 arrays."""
import pytest

pytestmark = pytest.mark.gpu


def system(kind="bl"):
    """Small relaxed Newton matrix: (case, outer, csr, right-hand side)."""
    import torch as t
    from broadcast_amd.cases import bl_case, cylinder_case
    from broadcast_amd.flow import Flow, to_device

    case = bl_case(24, 16, seed=5) if kind == "bl" else cylinder_case(21, 16, seed=5)
    f = Flow(case)
    w = to_device(case.w)
    f.apply_bcs(w)
    n = 5 * case.im * case.jm
    cd = t.full((case.im * case.jm,), 1e-3, dtype=t.float64, device="cuda")
    b = t.randn(n, dtype=t.float64, device="cuda", generator=t.Generator("cuda").manual_seed(1))
    return case, "i" if kind == "bl" else "j", tuple(a.clone() for a in f.jacobian_csr(w, coefdiag=cd)), b


@pytest.mark.parametrize("kind", ["bl", "cyl"])
def test_solve_right_hand_side_of_any_stride(kind):
    import torch as t
    from broadcast_amd.newton import BlockBandLU, csr_residual

    case, outer, csr, b = system(kind)
    lu = BlockBandLU(case.im, case.jm, outer=outer).factor(*csr)
    x = lu.solve(b)
    column = t.stack((b, b + 1.0), 1)[:, 0]
    assert not column.is_contiguous()
    assert t.equal(lu.solve(column), x)
    assert t.equal(csr_residual(csr, t.stack((x, b), 1)[:, 0], column), csr_residual(csr, x, b))
    one = t.ones(1, dtype=t.float64, device="cuda").expand(b.numel())
    assert t.equal(lu.solve(one), lu.solve(one.clone()))
    assert t.equal(lu.solve(b.reshape(-1, 1)), x)


def test_solve_index_types():
    import torch as t
    from broadcast_amd.newton import BlockBandLU, csr_residual

    case, outer, csr, b = system()
    x = BlockBandLU(case.im, case.jm, outer=outer).factor(*csr).solve(b)
    indptr, indices, data = csr
    forms = {"int64": (indptr.long(), indices.long(), data),
             "strided": tuple(t.stack((a, a), 1)[:, 0] for a in (indptr, indices, data))}
    for name, form in forms.items():
        print(name, flush=True)
        assert t.equal(BlockBandLU(case.im, case.jm, outer=outer).factor(*form).solve(b), x)
        assert t.equal(csr_residual(form, x, b), csr_residual(csr, x, b))
    # the rows of a larger matrix: factor counts from the first row start, the
    # product reads at the row starts
    part = (indptr + 7, indices, data)
    assert t.equal(BlockBandLU(case.im, case.jm, outer=outer).factor(*part).solve(b), x)
    whole = (indptr + 7, t.cat((indices[:7], indices)), t.cat((data[:7], data)))
    assert t.equal(csr_residual(whole, x, b), csr_residual(csr, x, b))


def test_solve_refuses_other_types_and_devices():
    """Raised on the host, before any kernel is given an address."""
    import torch as t
    from broadcast_amd.newton import BlockBandLU, csr_residual

    case, outer, csr, b = system()
    lu = BlockBandLU(case.im, case.jm, outer=outer).factor(*csr)
    for wrong in (b.cpu(), b.float(), b.to(t.complex128)):
        with pytest.raises(RuntimeError):
            lu.solve(wrong)
        with pytest.raises(RuntimeError):
            csr_residual(csr, b, wrong)
        with pytest.raises(RuntimeError):
            csr_residual(csr, wrong, b)
    with pytest.raises(RuntimeError):
        csr_residual(tuple(a.cpu() for a in csr), b.cpu(), b.cpu())


def test_factor_is_complete_when_it_returns():
    """Nothing of factor is left on its stream when it returns, so a solve on
    another stream, which waits for nothing, finds the factors and the matrix."""
    import torch as t
    from broadcast_amd.newton import BlockBandLU

    case, outer, csr, b = system()
    x = BlockBandLU(case.im, case.jm, outer=outer).factor(*csr).solve(b)
    t.cuda.synchronize()
    first, second = t.cuda.Stream(), t.cuda.Stream()
    with t.cuda.stream(first):
        lu = BlockBandLU(case.im, case.jm, outer=outer).factor(*csr)
        assert first.query()
    with t.cuda.stream(second):
        y = lu.solve(b)
    t.cuda.synchronize()
    assert t.equal(x, y)


def band(outer, lines, line, kb):
    """A diagonally heavy random band of `lines` blocks of 5 `line` unknowns, kb
    blocks to either side (condition below 10): (im, jm, dense, csr)."""
    import torch as t

    n, B = 5 * lines * line, 5 * line
    A = t.randn(n, n, dtype=t.float64, device="cuda", generator=t.Generator("cuda").manual_seed(n + kb))
    k = t.arange(n, device="cuda") // B
    A *= (k[:, None] - k).abs() <= kb
    A += 4 * ((2 * kb + 1) * B) ** 0.5 * t.eye(n, dtype=t.float64, device="cuda")
    if outer == "j":
        # from j-line blocks to the reference's order
        A = A.reshape(lines, line, 5, lines, line, 5).permute(1, 0, 2, 4, 3, 5).reshape(n, n)
    im, jm = (lines, line) if outer == "i" else (line, lines)
    return im, jm, A, to_csr(A)


@pytest.mark.parametrize("outer", ["i", "j"])
@pytest.mark.parametrize("lines", [5, 12])
def test_derivatives_through_the_solve(outer, lines):
    """torch's derivatives of x = A^-1 b in b, reverse and forward, and its map
    over several b, against dense solves; from one end of the band and from both.
    Tolerance: backward stable solves of n unknowns at condition 10, 40 n 2^-53
    with the growth without pivoting."""
    import torch as t
    from broadcast_amd.newton import BlockBandLU, csr_residual

    im, jm, A, csr = band(outer, lines, 3, 1)
    n = A.shape[0]
    lu = BlockBandLU(im, jm, outer=outer).factor(*csr)
    assert (lu.mid < lu.nb) == (lines == 12)
    b, g = t.randn(2, n, dtype=t.float64, device="cuda", generator=t.Generator("cuda").manual_seed(2))

    def near(a, ref):
        return float((a - ref).norm()) <= 40 * n * 2.0 ** -53 * float(ref.norm())

    ref, refg = t.linalg.solve(A, b), t.linalg.solve(A, g)
    bt = b.clone().requires_grad_()
    x = lu.solve(bt)
    assert near(lu.solve(b), ref) and near(x.detach(), ref)
    x.backward(g)
    assert near(bt.grad, t.linalg.solve(A.T.contiguous(), g))
    assert near(t.func.jvp(lu.solve, (b,), (g,))[1], refg)
    both = t.func.vmap(lu.solve)(t.stack((b, g)))
    assert near(both[0], ref) and near(both[1], refg)
    bt = b.clone().requires_grad_()
    csr_residual(csr, g, bt).backward(g)
    assert t.equal(bt.grad, g)


def weak_schur(A, B, at, to, eps):
    """A(at, at) such that eliminating block `to` leaves it one singular value of
    eps in place of 1: rows of the elimination in that direction grow by 1 / eps,
    though no pivot is below 1e-14 of its tile; the matrix stays well conditioned."""
    import torch as t

    r, c = slice(at * B, (at + 1) * B), slice(to * B, (to + 1) * B)
    g = t.Generator("cuda").manual_seed(7)
    U, V = (t.linalg.qr(t.randn(B, B, dtype=t.float64, device="cuda", generator=g))[0] for _ in range(2))
    s = t.ones(B, dtype=t.float64, device="cuda")
    s[0] = eps
    A[r, r] = A[r, c] @ t.linalg.solve(A[c, c], A[c, r]) + (U * s) @ V


def to_csr(A):
    c = A.to_sparse_csr()
    return c.crow_indices(), c.col_indices(), c.values()


def test_growth_in_the_upward_elimination_is_noticed():
    """A matrix (condition about 1e3) that only the upward elimination is unstable
    for: the solve is downwards then and accurate.  Tolerance: 40 n cond 2^-53."""
    import torch as t
    from broadcast_amd.newton import SOLVE_TOL, BlockBandLU, refine

    im, jm, A, _ = band("i", 12, 4, 1)
    B, n = 5 * jm, A.shape[0]
    weak_schur(A, B, im - 2, im - 1, 1e-11)
    b = t.randn(n, dtype=t.float64, device="cuda", generator=t.Generator("cuda").manual_seed(2))
    lu = BlockBandLU(im, jm).factor(*to_csr(A))
    assert lu.np_lu and lu.mid < lu.nb
    ref, cond = t.linalg.solve(A, b), float(t.linalg.cond(A))
    for _ in range(2):
        x = lu.solve(b)
        assert float((x - ref).norm()) <= 40 * n * cond * 2.0 ** -53 * float(ref.norm())
        assert lu.np_lu and lu.mid == lu.nb
    # left to refine()
    lu = BlockBandLU(im, jm, check=False).factor(*to_csr(A))
    x = lu.solve(b)
    assert not float((x - ref).norm()) <= 1e-6 * float(ref.norm())
    assert refine(lu, to_csr(A), b, x)[1] <= SOLVE_TOL
    assert float((x - ref).norm()) <= 40 * n * cond * 2.0 ** -53 * float(ref.norm())
    assert lu.np_lu and lu.mid == lu.nb


@pytest.mark.parametrize("pivot", [2e-14, 0.0])
def test_growth_inside_a_block_is_pivoted(pivot):
    """A second pivot just above the reported size, or a first one of zero, in
    the first and the last block row: the pivoted LU of the diagonal blocks in
    the end."""
    import torch as t
    from broadcast_amd.newton import BlockBandLU

    im, jm, A, _ = band("i", 12, 4, 1)
    B, n = 5 * jm, A.shape[0]
    for k in (0, n - B):
        m = float(A[k:k + B, k:k + B].abs().max())
        A[k:k + 2, k:k + 2] = m
        A[k + 1, k + 1] += m * pivot
        if pivot == 0.0:
            A[k, k] = 0.0
    b = t.randn(n, dtype=t.float64, device="cuda", generator=t.Generator("cuda").manual_seed(2))
    lu = BlockBandLU(im, jm).factor(*to_csr(A))
    ref, cond = t.linalg.solve(A, b), float(t.linalg.cond(A))
    x = lu.solve(b)
    assert float((x - ref).norm()) <= 40 * n * cond * 2.0 ** -53 * float(ref.norm())
    assert not lu.np_lu


@pytest.mark.parametrize("lines,kb", [(1, 1), (1, 3), (2, 3), (3, 7)])
def test_half_width_beyond_the_matrix(lines, kb):
    """A half-width of the band given by the caller may exceed the block rows.
    Tolerance: 40 n 2^-53, as above."""
    import torch as t
    from broadcast_amd.newton import BlockBandLU

    im, jm, A, csr = band("i", lines, 3, min(kb, lines - 1))
    n = A.shape[0]
    b = t.randn(n, dtype=t.float64, device="cuda", generator=t.Generator("cuda").manual_seed(2))
    lu = BlockBandLU(im, jm, kb=kb).factor(*csr)
    ref = t.linalg.solve(A, b)
    assert lu.np_lu and lu.kb == kb
    assert float((lu.solve(b) - ref).norm()) <= 40 * n * 2.0 ** -53 * float(ref.norm())
