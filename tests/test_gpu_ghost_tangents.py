"""The Jacobian's ghost tangents in one launch (every operation of the boundary
sequence once) against the launch per operation (the same sequence with its wall
condition repeated, which changes no ghost and is not one of the one-launch kind):
the same kept pattern, values to the rounding of ~60 operations a line, 1e-12 of
the largest.  Meshes at the edges of the corner workgroups (2 gh + 1 lines each)
and of the 64 lines of the others; one and two zones."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,im,jm", [("bl", 14, 8), ("bl", 72, 14), ("bl", 79, 16), ("cyl", 14, 15), ("cyl", 30, 9),
                                        ("cyl", 75, 72)])
def test_one_launch_is_one_by_one(kind, im, jm):
    import torch as t
    from broadcast_amd import _lib
    from broadcast_amd.cases import bl_case, cylinder_case
    from broadcast_amd.flow import Flow, to_device

    print(f"{kind} {im}x{jm}", flush=True)
    case = (bl_case(im, jm, seed=im, noise=1e-2) if kind == "bl"
            else cylinder_case(im, jm, seed=im, k2=1.01, mach=0.3, noise=1e-2))
    out = []
    for repeat in (False, True):
        f = Flow(case)
        if repeat:
            wall = next(op for op in f.ops if op.kind == _lib.BC_WALL_ADIA)
            k = next(n for n, op in enumerate(f.ops) if op.kind == _lib.BC_WALL_ADIA)
            ops = [_lib.BcOp.from_buffer_copy(op) for op in f.ops]
            ops.insert(k, _lib.BcOp.from_buffer_copy(wall))
            f.ops, f.nops = (_lib.BcOp * len(ops))(*ops), len(ops)
        w = to_device(case.w)
        f.apply_bcs(w)
        out.append([a.clone() for a in f.jacobian_csr(w)])
    (p, q, x), (rp, rq, rx) = out
    assert t.equal(p, rp) and t.equal(q, rq)
    assert float((x - rx).abs().max()) <= 1e-12 * float(rx.abs().max())
