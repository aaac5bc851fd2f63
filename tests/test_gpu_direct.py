"""Glyphs masked in one workgroup (k_atlas_direct) and through the tile
pipeline, and which of the two a set takes (rz_atlas_set), against the oracle:
mask sizes around 16-pixel columns, one pixel, and the largest the accumulators
hold, next to glyphs that need the tile pipeline (too large, too many
segments), with lines, quads and cubics, long edges, paths crossing every side
of their view, both edge modes and fill rules, more slots than are staged at
once, and a flatness that needs the deepest subdivision.

A pixel sums the deposits of the lines in it, each rounded once to 2^-20, of
coordinates rounded to 2^-20 (heights) and 2^-23 (columns): 2e-5 holds for the
twenty-odd lines a pixel sees here."""
import numpy as np
import pytest
import torch

import _oracle as O
import rasterize_amd as rz
from rasterize_amd import FillRule, PathBuilder, Transform

pytestmark = pytest.mark.gpu

BAR = 2e-5


def blob(rng, w, h, n, kinds="lqc", over=0.0):
    """n segments round the middle of a w x h view, reaching `over` beyond it."""
    c = np.array([0.5 * w, 0.5 * h])
    r = (0.5 + over) * np.array([w, h])
    th = np.sort(rng.uniform(0, 2 * np.pi, n))
    at = lambda t, k: tuple(c + k * r * np.array([np.cos(t), np.sin(t)]))  # noqa: E731
    pb = PathBuilder().move_to(at(th[0], rng.uniform(0.4, 1.0)))
    for k in range(n):
        t = th[(k + 1) % n]
        end = at(t, rng.uniform(0.4, 1.0))
        kind = kinds[int(rng.integers(len(kinds)))]
        if kind == "l":
            pb.line_to(end)
        elif kind == "q":
            pb.quad_to(at(t - 0.1, rng.uniform(0.2, 1.2)), end)
        else:
            pb.cubic_to(at(t - 0.4, rng.uniform(0.2, 1.3)), at(t + 0.3, rng.uniform(0.2, 1.3)), end)
    return pb.close().build()


def check(paths, sizes, rule, mode, trs=None, flatness=0.05, direct=None):
    trs = trs or [Transform.identity()] * len(paths)
    slots, x = [], 3
    for (w, h), tr in zip(sizes, trs):
        slots.append(rz.atlas_slot(x, 2, w, h, tr))
        x += w + 1
    atlas = np.full((max(h for _, h in sizes) + 5, x + 4), -1.0, np.float32)
    inside = np.zeros(atlas.shape, bool)
    rz.mask_atlas(paths, slots, atlas, rule, flatness=flatness, edge_mode=mode)
    if direct is not None:  # glyphs of k_atlas_direct make no records
        assert (last_counts(rz.default_context())[1] == 0) == direct
    worst = 0.0
    for p, s, tr in zip(paths, slots, trs):
        f = O.sd_mask if mode == rz._abi.RZ_EDGE_MASK else O.sd_mask_iter
        ref = f(p, tr, s.width, s.height, rule, flatness)
        got = atlas[s.y:s.y + s.height, s.x:s.x + s.width]
        d = np.abs(got - ref).max()
        worst = max(worst, d)
        assert d <= BAR, (s.width, s.height, d)
        inside[s.y:s.y + s.height, s.x:s.x + s.width] = True
    print(f"{len(paths)} glyphs, rule {rule}, mode {mode}: max|d|={worst:.2e}", flush=True)
    assert (atlas[~inside] == -1.0).all()


@pytest.mark.parametrize("rule", [FillRule.NonZero, FillRule.EvenOdd])
@pytest.mark.parametrize("mode", [rz._abi.RZ_EDGE_MASK, rz._abi.RZ_EDGE_ITER])
def test_sizes_and_sides(rule, mode):
    rng = np.random.default_rng(11)
    sizes = [(1, 1), (2, 5), (15, 16), (16, 17), (17, 33), (31, 1), (64, 64), (65, 3), (128, 128),
             (132, 135), (200, 190), (40, 300)]
    paths = [blob(rng, w, h, int(n), over=o) for (w, h), n, o in
             zip(sizes, [3, 4, 9, 20, 127, 5, 129, 12, 300, 60, 40, 7], [0, .3, 0, .2, .1, .5, 0, .4, .05, .3, .1, 0])]
    check(paths, sizes, rule, mode)


@pytest.mark.parametrize("rule", [FillRule.NonZero, FillRule.EvenOdd])
@pytest.mark.parametrize("mode", [rz._abi.RZ_EDGE_MASK, rz._abi.RZ_EDGE_ITER])
def test_sizes_and_sides_in_one_workgroup(rule, mode):
    """The same without the glyphs that need the tile pipeline, which take the
    small set with them; and long edges under transforms."""
    rng = np.random.default_rng(11)
    sizes = [(1, 1), (2, 5), (15, 16), (16, 17), (17, 33), (31, 1), (64, 64), (65, 3), (128, 128), (132, 135),
             (40, 300), (270, 50)]
    paths = [blob(rng, w, h, int(n), over=o) for (w, h), n, o in
             zip(sizes, [3, 4, 9, 20, 127, 5, 129, 12, 200, 60, 7, 30], [0, .3, 0, .2, .1, .5, 0, .4, .05, .3, 0, .2])]
    check(paths, sizes, rule, mode, direct=True)
    sizes = [(96, 120), (50, 40), (100, 90)]
    paths = [blob(rng, 96, 120, 4, "l", 2.0), blob(rng, 50, 40, 6, "c", 3.0), blob(rng, 100, 90, 30)]
    trs = [Transform.identity(), Transform.new_rotate(0.4),
           Transform.new_translate(20.0, -15.0) * Transform.new_scale(1.7, 0.6)]
    check(paths, sizes, rule, mode, trs, direct=True)


def test_transforms_long_edges_and_many_segments():
    rng = np.random.default_rng(12)
    sizes = [(96, 120), (50, 40), (60, 60), (100, 90)]
    paths = [blob(rng, 96, 120, 4, "l", 2.0), blob(rng, 50, 40, 6, "c", 3.0),
             blob(rng, 60, 60, 1100, "qc", 0.1),  # more crossings than int32 allows for: tile pipeline
             blob(rng, 100, 90, 30)]
    trs = [Transform.identity(), Transform.new_rotate(0.4), Transform.identity(),
           Transform.new_translate(20.0, -15.0) * Transform.new_scale(1.7, 0.6)]
    for rule in (FillRule.NonZero, FillRule.EvenOdd):
        check(paths, sizes, rule, rz._abi.RZ_EDGE_MASK, trs)


@pytest.mark.parametrize("flatness", [1e-4, 0.01, 2.0])
def test_flatness(flatness):
    rng = np.random.default_rng(13)
    check([blob(rng, 60, 50, 12), blob(rng, 30, 30, 5, "qc", 0.5)], [(60, 50), (30, 30)], FillRule.NonZero,
          rz._abi.RZ_EDGE_MASK, flatness=flatness, direct=True)


def test_updated_points_and_not_a_number():
    """Points replaced on the device are masked as they are; a NaN among the
    uploaded ones is reported as the reference reports it."""
    rng = np.random.default_rng(14)
    a = blob(rng, 60, 50, 12, "q")
    moved = a.points.copy().reshape(-1, 3, 2)  # the quads' control points; their ends stay joined
    moved[:, 1] += rng.uniform(-25.0, 25.0, moved[:, 1].shape)
    b = rz.Path(a.kinds, a.point_offsets, moved, a.subpaths, a.closed)
    glyphs = rz.DeviceGlyphs([a], [rz.atlas_slot(0, 0, 60, 50)])
    out = torch.zeros((50, 60), device="cuda")

    def run():
        for _ in range(4):
            glyphs.mask_device(out.data_ptr(), 60)
            try:
                glyphs.ctx.sync()
                return out.cpu().numpy()
            except rz.RzError as e:
                assert e.status == rz._abi.RZ_E_CAPACITY
    torch.cuda.synchronize()
    assert np.abs(run() - O.sd_mask(a, Transform.identity(), 60, 50, 0)).max() <= BAR
    pts = torch.tensor(b.points, device="cuda")
    torch.cuda.synchronize()
    glyphs.ctx.check(rz._abi.lib().rz_scene_update_device(glyphs.ctx.h, glyphs.h, pts.data_ptr(), None))
    assert np.abs(run() - O.sd_mask(b, Transform.identity(), 60, 50, 0)).max() <= BAR
    bad = blob(rng, 60, 50, 12, "q")
    bad.points[7] = np.nan
    with pytest.raises(rz.RzError) as e:
        rz.mask_atlas([a, bad], [rz.atlas_slot(0, 0, 60, 50), rz.atlas_slot(60, 0, 60, 50)],
                      np.zeros((50, 120), np.float32))
    assert e.value.status == rz._abi.RZ_E_NAN


def last_counts(ctx):
    import ctypes as C
    c = [C.c_size_t() for _ in range(3)]
    ctx.check(rz._abi.lib().rz_last_counts(ctx.h, *[C.byref(v) for v in c]))
    return [v.value for v in c]


def route(paths, sizes, rule=FillRule.NonZero, mode=rz._abi.RZ_EDGE_MASK, flatness=0.05):
    """Lines and records of one call over a set of glyphs in rows: glyphs of
    k_atlas_direct make lines only."""
    width = 4096
    slots, x, y, row = [], 0, 0, 0
    for w, h in sizes:
        if x + w > width:
            x, y, row = 0, y + row, 0
        slots.append(rz.atlas_slot(x, y, w, h))
        x, row = x + w, max(row, h)
    ctx = rz.Context(0)
    g = rz.DeviceGlyphs(paths, slots, ctx)
    out = torch.zeros((y + row, width), device="cuda")
    torch.cuda.synchronize()
    for _ in range(6):
        g.mask_device(out.data_ptr(), width, fill_rule=rule, flatness=flatness, edge_mode=mode)
        try:
            ctx.sync()
            break
        except rz.RzError as e:
            assert e.status == rz._abi.RZ_E_CAPACITY
    n_lines, records, _ = last_counts(ctx)
    atlas = out.cpu().numpy()
    g.close()
    ctx.close()
    return n_lines, records, atlas, slots


def of(n, w, h, segs, kinds="q", seed=15):
    """n glyphs of w x h (of a few different paths) and their sizes."""
    rng = np.random.default_rng(seed)
    some = [blob(rng, w, h, segs, kinds) for _ in range(min(n, 8))]
    return [some[k % len(some)] for k in range(n)], [(w, h)] * n


def lines(n, w, h, k, seed=16):
    rng = np.random.default_rng(seed)
    some = []
    for _ in range(8):
        p = rng.uniform(0, 1, (k, 2)) * (w, h)
        pb = PathBuilder().move_to(tuple(p[0]))
        for q in p[1:]:
            pb.line_to(tuple(q))
        some.append(pb.close().build())
    return [some[j % 8] for j in range(n)], [(w, h)] * n


@pytest.mark.parametrize("what,make,direct", [
    ("few small glyphs", lambda: of(1000, 16, 16, 20), True),
    ("many small glyphs", lambda: of(12000, 16, 16, 20), False),
    ("half a CU's LDS and more, few", lambda: of(3, 132, 135, 40), True),
    ("half a CU's LDS and more, many", lambda: of(4000, 132, 135, 40), False),
    ("just below half a CU's LDS, many", lambda: of(3000, 132, 132, 40), True),
    ("beyond the accumulators", lambda: of(3, 132, 137, 40), False),
    ("few long lines", lambda: lines(100, 100, 100, 30), True),
    ("many long lines", lambda: lines(100, 100, 100, 200), False),
    ("many long lines in more glyphs", lambda: lines(400, 100, 100, 200), False),
    ("few segments in few glyphs", lambda: of(20, 64, 64, 100, "lq"), True),
    ("many segments in few glyphs", lambda: of(20, 64, 64, 900, "lq"), False),
    ("many segments in many glyphs", lambda: of(1500, 64, 64, 400, "lq"), True),
    ("long strips", lambda: lines(400, 1500, 10, 30), False),
], ids=lambda v: v.replace(" ", "_").replace("'", "") if isinstance(v, str) else "")
def test_route(what, make, direct):
    """A set goes where direct_cost and DirectSet put it; either way the masks
    are the oracle's (tile pipeline: coordinates within a 16 px tile are rounded
    to 2^-20 in f32 and deposits to 2^-20, of up to 25 lines in a pixel: 5e-5)."""
    paths, sizes = make()
    n_lines, records, atlas, slots = route(paths, sizes)
    assert n_lines and (records == 0) == direct, what
    for p, s in list(zip(paths, slots))[:8]:
        got = atlas[s.y:s.y + s.height, s.x:s.x + s.width]
        d = np.abs(got - O.sd_mask(p, Transform.identity(), s.width, s.height, 0)).max()
        assert d <= (BAR if direct else 5e-5), (what, d)


def test_route_beside_larger_glyphs():
    """One glyph too large for the workgroup's LDS: the others join it in the
    tile pipeline, unless they are enough to pay for a launch of their own."""
    big, size = of(1, 200, 200, 60)
    alone = route(big, size)[1]
    for n, direct in ((400, False), (6000, True)):
        paths, sizes = of(n, 60, 60, 60)
        n_lines, records, atlas, slots = route(paths + big, sizes + size)
        assert (records == alone) == direct and records >= alone
        for p, s in [(paths[0], slots[0]), (paths[n - 1], slots[n - 1]), (big[0], slots[n])]:
            got = atlas[s.y:s.y + s.height, s.x:s.x + s.width]
            d = np.abs(got - O.sd_mask(p, Transform.identity(), s.width, s.height, 0)).max()
            assert d <= 5e-5, d


@pytest.mark.parametrize("rule", [FillRule.NonZero, FillRule.EvenOdd])
@pytest.mark.parametrize("mode", [rz._abi.RZ_EDGE_MASK, rz._abi.RZ_EDGE_ITER])
@pytest.mark.parametrize("oversized", [0, 3])
def test_both_size_classes(rule, mode, oversized):
    """More glyphs than one launch takes: a launch of two waves a glyph for the
    small ones and of four for the others, of lines, quads and cubics, and the
    same beside glyphs that need the tile pipeline."""
    rng = np.random.default_rng(17)
    some = []
    for k in range(64):
        w, h = rng.integers(20, 77, 2) if k % 2 else rng.integers(80, 129, 2)
        some.append((blob(rng, w, h, int(rng.integers(30, 140)), ("q", "lqc", "c", "lq")[k % 4], over=(0.0, 0.3)[k % 3 == 0]),
                     (int(w), int(h))))
    big = [(blob(rng, 150, 160, 50), (150, 160)) for _ in range(oversized)]
    glyphs = [some[k % 64] for k in range(2400)] + big
    n_lines, records, atlas, slots = route([g[0] for g in glyphs], [g[1] for g in glyphs], rule, mode)
    assert n_lines and (records == 0) == (oversized == 0)
    if oversized:
        assert records == route([g[0] for g in big], [g[1] for g in big], rule, mode)[1]
    f = O.sd_mask if mode == rz._abi.RZ_EDGE_MASK else O.sd_mask_iter
    refs = [f(p, Transform.identity(), w, h, rule, 0.05) for p, (w, h) in some + big]
    worst = 0.0
    for k, s in enumerate(slots):
        direct = k < 2400
        ref = refs[k % 64] if direct else refs[64 + k - 2400]
        d = np.abs(atlas[s.y:s.y + s.height, s.x:s.x + s.width] - ref).max()
        worst = max(worst, d)
        assert d <= (BAR if direct else 5e-5), (k, s.width, s.height, d)
    print(f"rule {rule}, mode {mode}, {oversized} oversized: max|d|={worst:.2e}", flush=True)


@pytest.mark.parametrize("mode", [rz._abi.RZ_EDGE_MASK, rz._abi.RZ_EDGE_NONE])
def test_sets_of_the_tile_pipeline(mode):
    """A set of glyphs beyond the accumulators, and small ones under
    ActiveEdgeRasterizer, both of more lines than a cold context has room for
    (the first run misses capacity). Bars as in test_gpu_mask.py."""
    rng = np.random.default_rng(18)
    side, n, flatness = (150, 300, 0.005) if mode == rz._abi.RZ_EDGE_MASK else (40, 900, 0.005)
    some = [blob(rng, side, side, 30, "c", 0.1) for _ in range(10)]
    for rule in (FillRule.NonZero, FillRule.EvenOdd):
        n_lines, records, atlas, slots = route([some[k % 10] for k in range(n)], [(side, side)] * n, rule, mode,
                                               flatness)
        assert n_lines > max(1 << 16, 16 * n * 31) and records
        f = O.sd_mask if mode == rz._abi.RZ_EDGE_MASK else O.ae_mask
        refs = [f(p, Transform.identity(), side, side, rule, flatness) for p in some]
        for k, s in enumerate(slots):
            d = np.abs(atlas[s.y:s.y + s.height, s.x:s.x + s.width] - refs[k % 10])
            assert d.max() <= 2e-3 and d.mean() <= 1e-5, (k, d.max())


def test_a_placement_that_fails_leaves_the_one_before():
    """rz_atlas_set that cannot be done (here: while its stream is being
    captured) must leave the set as it was: the masks are those of the first
    placement, bit for bit."""
    import ctypes as C
    from test_gpu_upload import Hip
    paths, sizes = of(40, 60, 60, 30)
    ctx = rz.Context(0)
    small = [rz.atlas_slot(64 * k, 0, 60, 60) for k in range(40)]
    g = rz.DeviceGlyphs(paths, small, ctx)
    out = torch.zeros((512, 64 * 40), device="cuda")
    torch.cuda.synchronize()

    def run():
        out.fill_(-1.0)
        torch.cuda.synchronize()
        for _ in range(4):
            g.mask_device(out.data_ptr(), 64 * 40)
            try:
                ctx.sync()
                return out.cpu().numpy().copy()
            except rz.RzError as e:
                assert e.status == rz._abi.RZ_E_CAPACITY
    ref = run()
    hip = Hip(ctx)
    # the second placement: larger views, and some beyond the accumulators
    large = (rz._abi.rz_atlas_slot * 40)(*[rz.atlas_slot(64 * k, 0, 60, 500 if k % 2 else 100) for k in range(40)])
    hip.check(hip.L.hipStreamBeginCapture(hip.stream, 0))
    s = rz._abi.lib().rz_atlas_set(ctx.h, g.h, large)
    graph = C.c_void_p()
    hip.check(hip.L.hipStreamEndCapture(hip.stream, C.byref(graph)))
    assert s == rz._abi.RZ_E_HIP
    assert np.array_equal(run(), ref)
    ctx.check(rz._abi.lib().rz_atlas_set(ctx.h, g.h, large))
    again = run()
    assert not np.array_equal(again, ref) and (again[:100, :60] >= 0.0).all()
