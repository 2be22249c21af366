"""A Flow's first CSR is a full build, also when a refresh is asked for.

The library takes the refresh route when the arrays it is given are, by their
addresses, those of the last CSR on the context; the context is shared by all
Flows of one mesh size and outlives them, so the new arrays of a later Flow can
have an earlier one's addresses with other contents."""
from types import SimpleNamespace

from broadcast_amd import flow as F


class _Lib:
    def __init__(self):
        self.calls = []

    def bca_jacobian_colored_csr(self, *a):
        self.calls.append("build")
        a[-1]._obj.value = 7
        return 0

    def bca_jacobian_colored_csr_refresh(self, *a):
        self.calls.append("refresh")
        a[-2]._obj.value, a[-1]._obj.value = 7, 0
        return 0


def _stub_flow(lib):
    class Tensors:
        int32 = float64 = None

        @staticmethod
        def empty(n, dtype=None, device=None):
            import torch

            return torch.zeros(n, dtype=torch.float64)

    f = F.Flow.__new__(F.Flow)
    f.t, f.L, f.im, f.jm, f.gh = Tensors, lib, 8, 8, 3
    f.case = SimpleNamespace(kind="bl")
    f.ctx = SimpleNamespace(sync_stream=lambda: None)
    f.phys, f.ops, f.nops, f.metrics = F._lib.Phys(), None, 0, None
    return f


def test_first_refresh_of_a_flow_is_a_full_build():
    import torch

    lib = _Lib()
    w = torch.zeros(1)
    for _ in range(2):  # the second Flow's arrays may have the first one's addresses
        f = _stub_flow(lib)
        f.jacobian_csr(w, refresh=True)
        assert lib.calls.pop() == "build" and f.csr_rebuilt
        f.jacobian_csr(w, refresh=True)
        assert lib.calls.pop() == "refresh" and not f.csr_rebuilt
