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
        assert np.sort(d.ravel())[-4] <= 2e-5, (n, spread, k)  # at most three pixels on a boundary
