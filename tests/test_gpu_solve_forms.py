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
