"""One batch run on two streams with different arrays: a call starts after the one
before it has used the batch's table and scratch.  The same kernels on the same
values, so the same bits as one call after the other."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tangent", [False, True])
@pytest.mark.parametrize("in_place", [False, True])
def test_calls_on_two_streams(tangent, in_place):
    import torch as t
    from broadcast_amd.batch import UnevenBatch
    from broadcast_amd.cases import bl_case, cylinder_case
    from broadcast_amd.flow import Flow, to_device

    cases = [bl_case(40, 31, seed=1, noise=1e-2), cylinder_case(32, 20, seed=2, mach=0.3, r1=5.0, dr1=0.05, noise=1e-2)]
    flows = [Flow(c) for c in cases]
    ncall = 4

    def arrays(k):
        g = t.Generator("cuda").manual_seed(k)
        ws = [to_device(c.w) * (1.0 + 1e-3 * k) for c in cases]
        return ws, [t.randn(w.numel(), dtype=t.float64, device="cuda", generator=g) for w in ws]

    def run(batch, ws, wds):
        out = (ws, wds) if in_place else (None, None)
        res, resd = batch.run(ws, wds if tangent else None, out[0], out[1] if tangent else None)
        return ws + wds + ([] if in_place else list(res) + list(resd or []))

    ref = []
    for k in range(ncall):
        ref.append(run(UnevenBatch(flows), *arrays(k)))
        t.cuda.synchronize()
    batch = UnevenBatch(flows)
    streams = [t.cuda.Stream(), t.cuda.Stream()]
    big = t.randn(3000, 3000, dtype=t.float64, device="cuda")
    given = [arrays(k) for k in range(ncall)]
    t.cuda.synchronize()
    got = []
    for k in range(ncall):
        with t.cuda.stream(streams[k % 2]):
            if k % 2 == 0:
                for _ in range(3):  # the other stream would be ahead of this one
                    big @ big
            got.append(run(batch, *given[k]))
    t.cuda.synchronize()
    for k in range(ncall):
        print(f"call {k}", flush=True)
        assert len(got[k]) == len(ref[k])
        for a, b in zip(got[k], ref[k]):
            assert t.equal(a.nan_to_num(), b.nan_to_num())
