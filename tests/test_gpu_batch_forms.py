"""The batched residual's less usual calls against one mesh at a time: outputs in
the place of inputs, two meshes on one state, a sequence of boundary conditions
that has to go one operation after the other.

Tolerance: the same device functions per mesh, possibly contracted differently in
the two kernels; 1e-12 of the largest value, the bound of the per-mesh tests."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tangent", [False, True])
@pytest.mark.parametrize("form", ["plain", "in place", "one state", "in turn"])
def test_batch_form(form, tangent):
    import torch as t
    from broadcast_amd import _lib
    from broadcast_amd.batch import UnevenBatch
    from broadcast_amd.cases import bl_case, cylinder_case
    from broadcast_amd.flow import Flow, to_device

    cases = [bl_case(31, 16, seed=1, noise=1e-2), cylinder_case(16, 30, seed=2, mach=0.3, r1=5.0, dr1=0.05, noise=1e-2),
             bl_case(31, 16, seed=1, noise=1e-2, k2=0.0), bl_case(5, 6, seed=3)]
    flows = [Flow(c) for c in cases]
    if form == "in turn":
        # the wall before the outflow that runs on over its ghosts
        f = flows[0]
        ops = [_lib.BcOp.from_buffer_copy(f.ops[k]) for k in (3, 0, 1, 2)]
        ops[3].box[1] = 1 - f.gh
        f.ops = (_lib.BcOp * 4)(*ops)
    ws = [to_device(c.w) for c in cases]
    wds = [t.randn(w.numel(), dtype=t.float64, device="cuda", generator=t.Generator("cuda").manual_seed(k))
           for k, w in enumerate(ws)]
    if form == "one state":
        ws[2] = ws[0]
        wds[2] = wds[0]
    ref = []
    for f, w, wd in zip(flows, ws, wds):
        w, wd = w.clone(), wd.clone()
        if tangent:
            r, rd = f.jvp(w, wd)
        else:
            f.apply_bcs(w)
            r, rd = f.residual(w), None
        ref.append((w, wd, r, rd))
    res = resd = None
    if form == "in place":
        res, resd = list(ws), list(wds)
    res, resd = UnevenBatch(flows).run(ws, wds if tangent else None, res, resd if tangent else None)
    for k, (f, (w, wd, r, rd)) in enumerate(zip(flows, ref)):
        print(form, k, flush=True)
        inner = lambda a: a.view(5, f.nj, f.ni)[:, 3:-3, 3:-3]  # noqa: E731
        pairs = [(inner(res[k]), inner(r))] + ([(inner(resd[k]), inner(rd))] if tangent else [])
        if form != "in place":
            pairs += [(ws[k].view(5, -1), w.view(5, -1))] + ([(wds[k].view(5, -1), wd.view(5, -1))] if tangent else [])
        for a, b in pairs:
            a, b = a.reshape(5, -1), b.reshape(5, -1)
            ok = b.isfinite()
            assert bool((a.isfinite() == ok).all())
            scale = t.where(ok, b, 0.0).abs().amax(1)
            scale[1:4] = scale[1:4].max()
            assert bool((t.where(ok, a - b, 0.0).abs().amax(1) <= 1e-12 * scale).all())
