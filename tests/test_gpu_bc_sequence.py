"""A whole boundary-condition sequence in one launch (bca_bc_sequence) against its
operations one after the other (bca_bc_*): the drivers' sequences and random ones
(orders, lines running on into the corners, operations left out) -- whichever of
them the one launch takes -- with and without the tangent, on the smallest meshes,
one line either side of a workgroup's 64, and below the mesh where the corners
would meet (which goes one after the other).

Tolerance: the same expressions per line (~100 operations, layers growing
linearly), so 1e-12 of the largest value leaves two orders."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _one_by_one(f, L, _lib, ops, w, wd):
    from broadcast_amd.flow import _ptr
    h = f.ctx.sync_stream()
    wp, wdp = _ptr(w), _ptr(wd)
    for op in ops:
        box = (C.c_int * 4)(*op.box)
        if op.kind == _lib.BC_INLET:
            rc = L.bca_bc_inlet(h, wp, wdp, op.loc, box, op.data, op.lm, _ptr(f.nx), _ptr(f.ny), op.gam)
        elif op.kind == _lib.BC_NOREF:
            rc = L.bca_bc_noref(h, wp, wdp, op.data, op.lm, op.loc, box, _ptr(f.nx), _ptr(f.ny), op.gam)
        elif op.kind == _lib.BC_EXTRAP2:
            rc = L.bca_bc_extrap2(h, wp, wdp, op.loc, box, 5)
        elif op.kind == _lib.BC_WALL_ADIA:
            rc = L.bca_bc_wall_adia(h, wp, wdp, op.loc, box, op.gam)
        else:
            box2, tr, rc = (C.c_int * 4)(*op.box2), (C.c_int * 2)(*op.tr), 0
            for a in (w, wd):
                if a is not None:
                    rc = rc or L.bca_bc_join(h, _ptr(a), box, box2, tr, 5, f.ni, f.nj)
        assert rc == 0, L.bca_last_error()


def _variant(f, _lib, rng):
    """The sequence reordered, thinned and with some lines run on into the corners."""
    out = []
    for k in rng.permutation(f.nops):
        if rng.random() < 0.15:
            continue
        op = _lib.BcOp.from_buffer_copy(f.ops[k])
        if op.kind in (_lib.BC_EXTRAP2, _lib.BC_WALL_ADIA) and rng.random() < 0.5:
            a, b, n = (1, 3, f.jm) if op.loc < 2 else (0, 2, f.im)
            op.box[a] = int(rng.choice([1 - f.gh, 1, 2]))
            op.box[b] = n + int(rng.choice([-1, 0, f.gh]))
        out.append(op)
    return (_lib.BcOp * len(out))(*out)


@pytest.mark.parametrize("kind,im,jm", [("bl", 14, 8), ("bl", 5, 7), ("bl", 72, 9), ("bl", 73, 17), ("bl", 140, 71),
                                        ("cyl", 14, 10), ("cyl", 73, 9), ("cyl", 71, 72)])
def test_one_launch_is_the_sequence(kind, im, jm):
    import torch as t
    from broadcast_amd import _lib
    from broadcast_amd.cases import bl_case, cylinder_case
    from broadcast_amd.flow import Flow, _ptr, to_device

    print(f"{kind} {im}x{jm}", flush=True)
    f = Flow(bl_case(im, jm, seed=im, noise=1e-2) if kind == "bl"
             else cylinder_case(im, jm, seed=im, mach=0.3, noise=1e-2))
    rng = np.random.default_rng(im * jm)
    # every ghost holds something, so that a line that reads a ghost too early is seen
    w0 = to_device(f.case.w)
    w0 = w0 * t.from_numpy(1.0 + 0.05 * rng.random(w0.numel())).cuda()
    wd0 = t.from_numpy(rng.standard_normal(w0.numel())).cuda()
    for k in range(12):
        ops = f.ops if k == 0 else _variant(f, _lib, rng)
        for tangent in (False, True):
            w, wd = w0.clone(), wd0.clone() if tangent else None
            rw, rwd = w0.clone(), wd0.clone() if tangent else None
            _lib.check(f.L.bca_bc_sequence(f.ctx.sync_stream(), _ptr(w), _ptr(wd), ops, len(ops), _ptr(f.nx),
                                           _ptr(f.ny)), "sequence")
            _one_by_one(f, f.L, _lib, ops, rw, rwd)
            for a, b in ((w, rw), (wd, rwd)):
                if a is None:
                    continue
                ok = b.isfinite()
                assert bool((a.isfinite() == ok).all())
                a, b = (t.where(ok, x, 0.0).view(5, -1) for x in (a, b))
                err = (a - b).abs().amax(1) / b.abs().amax(1).clamp_min(1e-300)
                assert float(err.max()) < 1e-12, (k, tangent, err)
