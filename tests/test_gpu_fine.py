"""The fine stage's grouping of paths over a tile and its pixel layout, against
the oracle: numbers of paths around the group size and the 64-path batch,
tiles without records, tiles too large for int32 between ordinary ones,
right-edge columns, and image widths and row strides that are no multiple of
four (bars as in test_gpu_scene.py / test_gpu_mask.py: 2^-20 fixed point and
f32 cell coordinates stay far inside them)."""
import numpy as np
import pytest
import torch

import _oracle as O
import rasterize_amd as rz
from rasterize_amd import FillRule, LinColor, PathBuilder, Scene, SignedDifferenceRasterizer, Transform

pytestmark = pytest.mark.gpu

MAX_ABS, MEAN_ABS = 2e-3, 1e-5
I = Transform.identity()


def rect(x0, y0, x1, y1, copies=1):
    pb = PathBuilder()
    for _ in range(copies):
        pb = pb.move_to((x0, y0)).line_to((x1, y0)).line_to((x1, y1)).line_to((x0, y1)).close()
    return pb.build()


def fills(n, w, h, wide_at=()):
    """n small blobs, whole-view rectangles (uniform tiles), shapes over the
    right edge, and at wide_at rectangles of 700 coincident outlines."""
    rng = np.random.default_rng(n)
    out = []
    for k in range(n):
        rule = FillRule.EvenOdd if k % 3 == 1 else FillRule.NonZero
        c = LinColor(*(0.4 * rng.uniform(0, 1, 3)), 0.4)
        if k in wide_at:
            p = rect(*rng.uniform(1, 8, 2), *rng.uniform(12, 30, 2), copies=701)
        elif k % 5 == 4:
            p = rect(-3.0, -3.0, w + 5.0, h + 4.0)
        elif k % 7 == 3:
            p = rect(w - 7.3, 2.2, w + 9.0, h - 3.1)
        else:
            p = PathBuilder().move_to(rng.uniform(4, min(w, h), 2)).circle(rng.uniform(1, 12)).build()
        out.append((p, c, rule))
    return out


@pytest.mark.parametrize("n,wide", [(1, ()), (4, ()), (5, (0,)), (9, (3, 4)), (64, (7,)), (67, (63, 65))])
def test_path_groups(n, wide):
    w, h = 45, 38
    fl = fills(n, w, h, wide)
    view = (0.0, 0.0, float(w), float(h))
    scene = Scene(Scene.GROUP, children=[Scene.fill(*f) for f in fl])
    got = scene.render(SignedDifferenceRasterizer(), I, view, (0.5, 0.4, 0.3, 0.9))
    ref, _ = O.scene_render([(p, c.abi(), r) for p, c, r in fl], I, view, (0.5, 0.4, 0.3, 0.9))
    d = np.abs(got.image.astype(np.float64) - ref)
    print(f"{n} paths: max|d|={d.max():.3e} mean|d|={d.mean():.3e}", flush=True)
    assert d.max() <= MAX_ABS and d.mean() <= MEAN_ABS


# One wave takes a tile's paths in views of more than 8 tiles a CU, four waves
# a quarter of the row's paths each in smaller ones of eight paths and more
# (scene_split): the groups of four, the 64-path batches and the oversized
# tiles at their boundaries, in the waves' shares where there are four.
@pytest.mark.parametrize("n,wide,waves", [
    (8, (), 1), (9, (3, 4), 1), (64, (7,), 1), (67, (63, 65), 1), (131, (0, 64, 127, 128, 130), 1),
    (8, (1, 2), 4), (17, (4, 5, 9), 4), (20, (), 4), (256, (63, 64), 4),
    (270, (0, 63, 65, 67, 68, 131, 133, 269), 4)])
def test_path_groups_of_one_and_four_waves(n, wide, waves):
    w, h = 45, 38
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    W, H = (w, h) if waves == 4 else (16 * (cus + 1), 128)  # 8 rows of tiles: more than 8 a CU
    fl = fills(n, w, h, wide)
    view = (0.0, 0.0, float(W), float(H))
    scene = Scene(Scene.GROUP, children=[Scene.fill(*f) for f in fl])
    got = scene.render(SignedDifferenceRasterizer(), I, view, (0.5, 0.4, 0.3, 0.9))
    ref, _ = O.scene_render([(p, c.abi(), r) for p, c, r in fl], I, view, (0.5, 0.4, 0.3, 0.9))
    d = np.abs(got.image.astype(np.float64) - ref)
    print(f"{n} paths, {waves} waves: max|d|={d.max():.3e} mean|d|={d[:h, :w].mean():.3e}", flush=True)
    assert np.isfinite(got.image).all()
    assert d.max() <= MAX_ABS and d[:h, :w].mean() <= MEAN_ABS


@pytest.mark.parametrize("long", [False, True])
@pytest.mark.parametrize("waves", [1, 4])
def test_queued_tiles(waves, long):
    """The persistent grid gives the image of the plain one bit for bit, for
    one and four waves a tile, every register budget, and the general gradient
    evaluation (more than 64 stops)."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    w, h = (301, 200) if waves == 4 else (16 * (cus + 1), 128)
    fl = fills(60, w, h, (5, 40))
    stops = [(k / 69.0, LinColor(0.3 * (k % 3), 0.2, 0.1 * (k % 7), 0.6)) for k in range(70 if long else 5)]
    fl.append((rect(3.0, 2.0, w - 4.0, h - 3.0),
               rz.GradLinear(stops, start=(0.0, 0.0), end=(0.7 * w, 0.4 * h), spread=rz.GradSpread.Reflect),
               FillRule.NonZero))
    ctx = rz.Context(0)
    ds = rz.DeviceScene(Scene(Scene.GROUP, children=[Scene.fill(*f) for f in fl]), ctx)
    out = torch.zeros((h, w, 4), device="cuda")

    def render():
        out.fill_(-1.0)
        torch.cuda.synchronize()
        for _ in range(5):
            ds.render_device(I, (0.0, 0.0, float(w), float(h)), out.data_ptr(), w)
            try:
                ctx.sync()
                return out.cpu().numpy().copy()
            except rz.RzError as e:
                assert e.status == rz._abi.RZ_E_CAPACITY
    ref = render()
    assert np.isfinite(ref).all()
    for budget in (8, 6, 1):
        ctx.set_param(rz._abi.RZ_PARAM_SCENE_WAVES, budget)
        ctx.set_param(rz._abi.RZ_PARAM_SCENE_QUEUE, 0)
        assert np.array_equal(render(), ref), budget
        ctx.set_param(rz._abi.RZ_PARAM_SCENE_QUEUE, 1)
        for _ in range(3):
            assert np.array_equal(render(), ref), budget
    ctx.set_param(rz._abi.RZ_PARAM_FINE_LDS, 32)  # four times as much for four waves
    assert np.array_equal(render(), ref)
    ds.close()
    ctx.close()


@pytest.mark.parametrize("w,h,pad", [(1, 1, 0), (2, 17, 1), (15, 16, 0), (17, 33, 5), (47, 15, 2), (130, 31, 3)])
def test_mask_rows_of_any_width(w, h, pad):
    """Every pixel of the mask, nothing beside it, from an unaligned start."""
    path = PathBuilder().move_to((0.6 * w, 0.45 * h)).circle(0.5 * max(w, h)).build()
    stride = w + pad
    for rule in (FillRule.NonZero, FillRule.EvenOdd):
        buf = torch.full((1 + stride * h + 4,), -1.0, device="cuda")
        torch.cuda.synchronize()
        dp = rz.DevicePath(path)
        for _ in range(3):
            dp.mask_device(I, w, h, buf.data_ptr() + 4, stride, fill_rule=rule, edge_mode=rz._abi.RZ_EDGE_NONE)
            try:
                dp.ctx.sync()
                break
            except rz.RzError as e:
                assert e.status == rz._abi.RZ_E_CAPACITY
        got = buf.cpu().numpy()
        rows = got[1:1 + stride * h].reshape(h, stride)
        ref = O.ae_mask(path, I, w, h, rule)
        d = np.abs(rows[:, :w] - ref)
        assert d.max() <= MAX_ABS and d.mean() <= MEAN_ABS
        assert got[0] == -1.0 and (rows[:, w:] == -1.0).all() and (got[1 + stride * h:] == -1.0).all()


def on_a_jump(paint, pos, w, h):
    """Pixels whose position in the gradient lies on a jump of its colour, to
    the rounding of its f64 evaluation: on two stops at one position, on the
    wrap of a repeated gradient, or where a radial gradient's roots end."""
    x, y = np.meshgrid(np.arange(w) + 0.5, np.arange(h) + 0.5)
    a, b, c, d, e, f = paint.tr.m
    det = a * e - b * d
    px, py = (e * (x - c) - b * (y - f)) / det, (a * (y - f) - d * (x - c)) / det
    jump = np.zeros(x.shape, bool)
    if isinstance(paint, rz.GradLinear):
        vx, vy = paint.end[0] - paint.start[0], paint.end[1] - paint.start[1]
        t = ((px - paint.start[0]) * vx + (py - paint.start[1]) * vy) / (vx * vx + vy * vy)
    else:
        fc = paint.fcenter if paint.fcenter is not None else paint.center
        cx, cy, rd = paint.center[0] - fc[0], paint.center[1] - fc[1], paint.radius - paint.fradius
        qx, qy = px - fc[0], py - fc[1]
        A = cx * cx + cy * cy - rd * rd
        B = -2.0 * (cx * qx + cy * qy + paint.fradius * rd)
        disc = B * B - 4.0 * A * (qx * qx + qy * qy - paint.fradius ** 2)
        jump |= np.abs(disc) < 1e-9 * B * B
        t = (-B + np.sign(A) * np.sqrt(np.maximum(disc, 0.0))) / (2.0 * A)  # the larger root
    eps = 1e-11 * (1.0 + np.abs(t))
    if paint.spread != rz.GradSpread.Pad:
        if paint.spread == rz.GradSpread.Repeat:
            jump |= np.abs(t - np.round(t)) < eps
            t = t % 1.0
        else:
            t = np.abs((t + 1.0) % 2.0 - 1.0)
    for p in pos[1:][np.diff(pos) == 0.0]:
        jump |= np.abs(t - p) < eps
    return jump


@pytest.mark.parametrize("n", [1, 2, 5, 64, 65])
@pytest.mark.parametrize("spread", [rz.GradSpread.Pad, rz.GradSpread.Repeat, rz.GradSpread.Reflect])
def test_gradient_stops(n, spread):
    """Gradients of few and many stops (65: beyond the wave's lanes), stops at
    equal positions, every spread, linear and sRGB interpolation, focal
    circles inside, on and outside the outer one (no root: transparent).
    Colours are f32 through the same formulas: 2e-5, of pixels whose position
    does not sit on a stop boundary (a jump between equal positions)."""
    w, h = 50, 35
    rng = np.random.default_rng(10 * n + spread)
    pos = np.sort(rng.uniform(0.0, 1.0, n))
    if n >= 5:
        pos[2] = pos[1]
    stops = []
    for p in pos:
        a = rng.uniform(0.2, 1.0)
        stops.append((float(p), LinColor(*(a * rng.uniform(0, 1, 3)), a)))
    common = dict(spread=spread, tr=Transform.new_rotate(0.3).pre_scale(1.1, 0.9))
    paints = [
        rz.GradLinear(stops, linear_colors=False, start=(5.0, 3.0), end=(38.0, 30.0), **common),
        rz.GradLinear(stops, linear_colors=True, start=(30.0, 3.0), end=(12.0, 9.0), **common),
        rz.GradRadial(stops, center=(25.0, 16.0), radius=14.0, **common),
        rz.GradRadial(stops, center=(25.0, 16.0), radius=14.0, fcenter=(20.0, 12.0), fradius=2.0, **common),
        rz.GradRadial(stops, center=(30.0, 16.0), radius=6.0, fcenter=(14.0, 12.0), fradius=3.0, **common),
    ]
    view = (0.0, 0.0, float(w), float(h))
    for k, paint in enumerate(paints):
        fl = [(rect(-2.0, 1.5, 44.25, 33.0), paint, FillRule.NonZero),
              (PathBuilder().move_to((20.0, 18.0)).circle(13.0).build(), paint, FillRule.NonZero)]
        got = Scene(Scene.GROUP, children=[Scene.fill(*f) for f in fl]).render(
            SignedDifferenceRasterizer(), I, view, (0.2, 0.3, 0.4, 1.0))
        ref, _ = O.scene_render([(p, c.abi(), r) for p, c, r in fl], I, view, (0.2, 0.3, 0.4, 1.0))
        d = np.abs(got.image.astype(np.float64) - ref).max(2)
        print(f"{n} stops, spread {spread}, paint {k}: max|d|={d.max():.3e}", flush=True)
        assert np.isfinite(got.image).all(), (n, spread, k)
        assert np.sort(d.ravel())[-4] <= 2e-5, (n, spread, k)  # at most three pixels on a boundary
        assert not ((d > 2e-5) & ~on_a_jump(paint, pos, w, h)).any(), (n, spread, k)
