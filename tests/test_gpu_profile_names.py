"""The names that kernel timings are read by: those of the kernels, and the face
kernels' for the residual and tangent kernels that took their place."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


def test_face_names_read_the_residual_kernels():
    import torch as t
    from broadcast_amd import _lib
    from broadcast_amd.cases import bl_case
    from broadcast_amd.flow import Flow, to_device

    f = Flow(bl_case(24, 16, seed=1))
    w = to_device(f.case.w)
    f.apply_bcs(w)
    L = _lib.lib()
    _lib.check(L.bca_profile_enable(f.ctx.sync_stream(), 1), "bca_profile_enable")
    for _ in range(3):
        f.residual(w)
    f.jvp_flux(w, t.ones_like(w))
    ms, n = C.c_double(), C.c_long()
    for name, launches in (("k_residual<f64>", 3), ("k_face<f64>", 3), ("k_residual<dual1>", 1), ("k_face<dual1>", 1),
                           ("k_facets<f64>", 0)):
        _lib.check(L.bca_profile_read(f.ctx.h, name.encode(), C.byref(ms), C.byref(n)), "bca_profile_read")
        assert n.value == launches and (ms.value > 0.0) == (launches > 0), name
    _lib.check(L.bca_profile_enable(f.ctx.h, 0), "bca_profile_enable")
