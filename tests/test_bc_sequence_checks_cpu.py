"""A boundary sequence refuses what its operations' own entries refuse, before any
launch (no GPU needed)."""
import ctypes as C

from broadcast_amd import _lib


def op(kind, loc, box, lm=0):
    o = _lib.BcOp()
    o.kind, o.loc, o.lm, o.gam = kind, loc, lm, 1.4
    o.box[:], o.tr[:] = box, [1, 2]
    o.data = 8
    return o


def test_sequence_refuses_like_the_entries():
    L = _lib.lib()
    ctx = C.c_void_p()
    assert L.bca_ctx_create(C.byref(ctx), 16, 12, 3, None) == 0
    p = C.c_void_p(8)
    bad = [op(_lib.BC_INLET, 0, [1, 1, 1, 12], lm=11),    # profile shorter than the interface
           op(_lib.BC_INLET, 2, [2, 1, 3, 1], lm=2),      # as long as the interface, but not up to it
           op(_lib.BC_INLET, 0, [4, 1, 4, 12], lm=12),    # reads the profile's layers past gh
           op(_lib.BC_NOREF, 3, [1, 12, 16, 12], lm=15),
           op(_lib.BC_EXTRAP2, 1, [17, 1, 17, 12]),
           op(_lib.BC_WALL_ADIA, 2, [1, 1, 20, 1])]
    for o in bad:
        box = (C.c_int * 4)(*o.box)
        one = {_lib.BC_INLET: lambda: L.bca_bc_inlet(ctx, p, None, o.loc, box, p, o.lm, p, p, 1.4),
               _lib.BC_NOREF: lambda: L.bca_bc_noref(ctx, p, None, p, o.lm, o.loc, box, p, p, 1.4),
               _lib.BC_EXTRAP2: lambda: L.bca_bc_extrap2(ctx, p, None, o.loc, box, 5),
               _lib.BC_WALL_ADIA: lambda: L.bca_bc_wall_adia(ctx, p, None, o.loc, box, 1.4)}[o.kind]()
        why = L.bca_last_error()
        assert one == -1
        assert L.bca_bc_sequence(ctx, p, None, (_lib.BcOp * 1)(o), 1, p, p) == -1
        assert L.bca_last_error() == why
    assert L.bca_ctx_destroy(ctx) == 0
