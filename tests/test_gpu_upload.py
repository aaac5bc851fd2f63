"""Device memory of blocking calls is taken from blocks the context keeps:
results must not depend on what ran before, resident paths and scenes must not
be touched by blocking calls in between, and the plain form's paths (made by
its first render) must be the uploaded ones. Every comparison is bit for bit
with the first run of the same call."""
import numpy as np
import pytest
import torch

import rasterize_amd as rz
from rasterize_amd import FillRule, SignedDifferenceRasterizer, Transform

pytestmark = pytest.mark.gpu

I = Transform.identity()


def mask(dp, w, h):
    out = torch.zeros((h, w), device="cuda")
    torch.cuda.synchronize()
    for _ in range(4):
        dp.mask_device(I, w, h, out.data_ptr(), w)
        try:
            dp.ctx.sync()
            return out.cpu().numpy()
        except rz.RzError as e:
            assert e.status == rz._abi.RZ_E_CAPACITY
    raise AssertionError("no run without a capacity miss")


@pytest.mark.parametrize("sizes", [(3, 200, 5), (60, 1, 60, 400)])
def test_blocking_calls_leave_resident_objects_alone(sizes):
    ctx = rz.Context(0)
    ras = SignedDifferenceRasterizer(ctx=ctx)
    resident = rz.DevicePath(rz.workload_cubics64(1, 200.0).paths[0], ctx)
    first = mask(resident, 200, 200)
    seen = {}
    for _ in range(2):
        for n in sizes:
            ws = rz.workload_scene(n, n, 256.0)
            view = (0.0, 0.0, 256.0, 200.0)
            batched = ws.scene().render(ras, I, view).image
            plain = ws.scene().render(ras, I, view, batched=False).image
            host = ras.mask_f32(ws.paths[0], I, 64, 48, FillRule.EvenOdd)
            lines = rz.flatten(ws.paths[-1], I, ctx=ctx)
            got = (batched, plain, host, lines)
            for a, b in zip(got, seen.setdefault(n, got)):
                assert np.array_equal(a, b), n
            assert np.array_equal(mask(resident, 200, 200), first)


def test_plain_form_keeps_the_uploaded_points():
    """rz_scene_update_device refreshes only the batched form's copy, also
    when the plain form has not run before it."""
    ws = rz.workload_scene(5, 12, 128.0)
    view = (0.0, 0.0, 128.0, 128.0)
    out = torch.zeros((128, 128, 4), device="cuda")
    torch.cuda.synchronize()

    def render(ds, batched):
        for _ in range(4):
            ds.render_device(I, view, out.data_ptr(), 128, batched=batched)
            try:
                ds.ctx.sync()
                return out.cpu().numpy().copy()
            except rz.RzError as e:
                assert e.status == rz._abi.RZ_E_CAPACITY
        raise AssertionError("no run without a capacity miss")

    ref = render(rz.DeviceScene(ws.scene()), False)
    ds = rz.DeviceScene(ws.scene())
    moved = torch.rand((ds.n_points(), 2), dtype=torch.float64, device="cuda") * 128.0
    torch.cuda.synchronize()
    ds.update_device(moved.data_ptr())
    assert not np.array_equal(render(ds, True), ref)
    assert np.array_equal(render(ds, False), ref)
