"""Device memory of blocking calls is taken from blocks the context keeps:
results must not depend on what ran before, resident paths and scenes must not
be touched by blocking calls in between, and the plain form's paths must be
the uploaded ones and be there when rz_scene_upload returns. Every comparison
is bit for bit with the first run of the same call."""
import numpy as np
import pytest
import torch

import rasterize_amd as rz
from rasterize_amd import FillRule, LinColor, PathBuilder, Scene, SignedDifferenceRasterizer, Transform

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


class Hip:
    """Capture of a context's stream through the HIP runtime torch has loaded."""

    def __init__(self, ctx):
        import ctypes as C
        self.C, self.L = C, C.CDLL("libamdhip64.so")
        self.stream = C.c_void_p(rz._abi.lib().rz_stream(ctx.h))

    def check(self, s):
        assert s == 0, s

    def capture(self, call):
        """call() captured and instantiated."""
        C, L = self.C, self.L
        self.check(L.hipStreamBeginCapture(self.stream, 0))
        try:
            call()
        finally:
            g = C.c_void_p()
            s = L.hipStreamEndCapture(self.stream, C.byref(g))
        self.check(s)
        x = C.c_void_p()
        self.check(L.hipGraphInstantiate(C.byref(x), g, None, None, C.c_size_t(0)))
        return g, x

    def launch(self, x):
        self.check(self.L.hipGraphLaunch(x, self.stream))

    def free(self, g, x):
        self.check(self.L.hipGraphExecDestroy(x))
        self.check(self.L.hipGraphDestroy(g))


def test_the_first_plain_render_of_a_scene_can_be_captured():
    """rz_render_device is asynchronous in both forms: with a context whose
    buffers have their size, a scene's first plain render neither allocates nor
    waits."""
    w = h = 160
    rng = np.random.default_rng(3)
    fills = [(PathBuilder().move_to(tuple(rng.uniform(20, 140, 2))).circle(rng.uniform(5, 30)).build(),
              LinColor(*(0.5 * rng.uniform(0, 1, 3)), 0.5)) for _ in range(12)]
    scene = Scene(Scene.GROUP, children=[Scene.fill(*f) for f in fills])
    view = (0.0, 0.0, float(w), float(h))
    out = torch.zeros((h, w, 4), device="cuda")
    torch.cuda.synchronize()
    ctx = rz.Context(0)
    warm = rz.DeviceScene(scene, ctx)
    for _ in range(4):
        warm.render_device(I, view, out.data_ptr(), w, batched=False)
        try:
            ctx.sync()
            break
        except rz.RzError as e:
            assert e.status == rz._abi.RZ_E_CAPACITY
    ref = out.cpu().numpy().copy()
    hip = Hip(ctx)
    fresh = rz.DeviceScene(scene, ctx)
    g, x = hip.capture(lambda: fresh.render_device(I, view, out.data_ptr(), w, batched=False))
    for k in range(3):
        out.fill_(float(k))
        torch.cuda.synchronize()
        hip.launch(x)
        ctx.sync()
        assert np.array_equal(out.cpu().numpy(), ref), k
        ctx.sync()
    hip.free(g, x)
    # a set without paints and rules keeps no copy: refused, and drawn once eager
    paths = [f[0] for f in fills]
    glyphs = rz.DeviceGlyphs(paths, [rz.atlas_slot(0, 0, 1, 1)] * len(paths), ctx)
    bare = lambda: rz.DeviceScene.render_device(glyphs, I, view, out.data_ptr(), w, batched=False)  # noqa: E731
    hip.check(hip.L.hipStreamBeginCapture(hip.stream, 0))
    with pytest.raises(rz.RzError) as e:
        bare()
    gr = hip.C.c_void_p()
    hip.check(hip.L.hipStreamEndCapture(hip.stream, hip.C.byref(gr)))
    assert e.value.status == rz._abi.RZ_E_CAPACITY
    bare()
    ctx.sync()


def test_a_tree_that_misses_capacity_takes_its_layers_once():
    """A cold context's first rz_render_tree misses the line capacity and runs
    again. It must then hold no more device memory than a context whose
    buffers had their size before the call."""
    import ctypes as C
    w, h, n = 1600, 1200, 4000
    rng = np.random.default_rng(7)
    pb = PathBuilder().move_to((0.0, 0.0))
    for _ in range(n):
        pb.cubic_to(*[tuple(p) for p in rng.uniform(0, 1, (3, 2)) * (w, h)])
    sheet = PathBuilder().move_to((0.0, 0.0)).line_to((w, 0.0)).line_to((w, h)).line_to((0.0, h)).close().build()
    group = Scene(Scene.GROUP, children=[Scene.fill(sheet, LinColor(0.1, 0.2, 0.1, 0.5)),
                                         Scene.fill(pb.close().build(), LinColor(0.2, 0.1, 0.0, 0.3))])
    view = (0.0, 0.0, float(w), float(h))
    layer = 16 * w * h  # the window's, and one for the group under the opacity

    def free():
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info()[0]

    def context():
        ctx = rz.Context(0)
        SignedDifferenceRasterizer(ctx=ctx).mask_f32(sheet, Transform.new_scale(0.01, 0.01), 16, 16, 0)
        return ctx
    out = torch.zeros((h, w, 4), device="cuda")
    taken, images = [], []
    for warm in (True, False):
        ctx = context()
        before = free()
        if warm:
            ds = rz.DeviceScene(group, ctx)
            for _ in range(6):
                ds.render_device(I, view, out.data_ptr(), w)
                try:
                    ctx.sync()
                    break
                except rz.RzError as e:
                    assert e.status == rz._abi.RZ_E_CAPACITY
            ds.close()
        images.append(group.with_opacity(0.5).render(SignedDifferenceRasterizer(ctx=ctx), I, view).image)
        taken.append(before - free())
        c = [C.c_size_t() for _ in range(3)]
        ctx.check(rz._abi.lib().rz_last_counts(ctx.h, *[C.byref(v) for v in c]))
        assert c[0].value > max(1 << 16, 16 * (n + 2))  # more lines than a cold context has room for
        ctx.close()
    print(f"taken warm {taken[0] >> 20} MB, cold {taken[1] >> 20} MB, a layer {layer >> 20} MB", flush=True)
    assert np.array_equal(*images)
    assert taken[1] < taken[0] + layer // 2
