"""The work this library is timed on: coverage masks, batched scene renders,
whole-scene renders from host memory, glyph atlases and the differentiable
render, each through its public entry point, from an icon to the largest
configuration of bench.py.

listed() are the fixed cases, draw() makes more of the same ranges, prepare()
builds what a program holds before the call (resident paths, scenes and output
images, buffers sized by one run), run() is one call, and exact() restates the
result in plain torch at 64 bits.
"""
import math

import numpy as np
import torch

import rasterize_amd as rz
from rasterize_amd import _abi

FLATNESS = 0.05  # the library's default, which every case uses
MODES = {"mask": _abi.RZ_EDGE_MASK, "iter": _abi.RZ_EDGE_ITER, "active": _abi.RZ_EDGE_NONE}


def listed():
    return [
        # an icon: one closed path of 64 cubics into a 512x512 mask
        {"name": "mask_icon", "kind": "mask", "path": "cubics", "segments": 64, "width": 512,
         "height": 512, "rule": "nonzero", "mode": "mask"},
        # a thumbnail-sized fill mask of odd size, the smallest call: latency and launches
        {"name": "mask_thumb", "kind": "mask", "path": "walk", "segments": 150, "width": 251,
         "height": 187, "rule": "evenodd", "mode": "iter"},
        # a map layer at screen size, the other rasterizer (ActiveEdgeRasterizer)
        {"name": "mask_map", "kind": "mask", "path": "walk", "segments": 20_000, "width": 1531,
         "height": 1117, "rule": "evenodd", "mode": "active"},
        # the library's headline: a 200k-segment path into a 4096x4096 mask
        {"name": "mask_4k", "kind": "mask", "path": "walk", "segments": 200_000, "width": 4096,
         "height": 4096, "rule": "nonzero", "mode": "mask"},
        # a user interface or small illustration, resident, redrawn into a window of odd size
        {"name": "scene_ui", "kind": "scene", "paths": 240, "scale": 0.5, "width": 601, "height": 455,
         "bg": True},
        # the largest scene: 10,000 shapes with solid and gradient paints at 2048x2048
        {"name": "scene_10k", "kind": "scene", "paths": 10_000, "scale": 1.0, "width": 2048,
         "height": 2048, "bg": False},
        # the reference's own scene benchmark as its users call it: Scene.render from host memory
        {"name": "render_circles", "kind": "circles", "paths": 1024, "size": 1024},
        # a scene tree (transform, opacity, clip) rendered from host memory
        {"name": "render_tree", "kind": "tree", "paths": 48, "width": 397, "height": 301},
        # the glyphs of a page of text into an atlas
        {"name": "atlas_text", "kind": "atlas", "glyphs": 400, "atlas_width": 1024},
        # a large glyph atlas (a CJK font's worth)
        {"name": "atlas_sheet", "kind": "atlas", "glyphs": 16_384, "atlas_width": 8192},
        # differentiable render, forward and backward: a small fit
        {"name": "diff_small", "kind": "diff", "paths": 16, "cubics": 8, "size": 256},
        # differentiable render, forward and backward: the configured size
        {"name": "diff_full", "kind": "diff", "paths": 256, "cubics": 32, "size": 1024},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    u = rng.random()
    if u < 0.4:
        w, h = _log_int(rng, 64, 4096), _log_int(rng, 64, 4096)
        # up to the headline's segments per pixel
        n = max(12, min(200_000, int(w * h * math.exp(rng.uniform(math.log(0.0005), math.log(0.012))))))
        return {"kind": "mask", "path": "walk", "segments": n, "width": w, "height": h,
                "rule": rng.choice(["nonzero", "evenodd"]), "mode": rng.choice(["mask", "iter", "active"])}
    if u < 0.65:
        w = _log_int(rng, 200, 2048)
        return {"kind": "scene", "paths": _log_int(rng, 40, 4000), "scale": rng.choice([0.5, 1.0]),
                "width": w, "height": max(64, int(w * rng.uniform(0.5, 1.0))), "bg": rng.random() < 0.5}
    if u < 0.8:
        return {"kind": "atlas", "glyphs": _log_int(rng, 60, 8000), "atlas_width": rng.choice([1024, 2048, 4096])}
    if u < 0.9:
        return {"kind": "diff", "paths": _log_int(rng, 8, 128), "cubics": rng.randint(4, 24),
                "size": _log_int(rng, 128, 800)}
    if u < 0.95:
        return {"kind": "circles", "paths": _log_int(rng, 64, 1024), "size": _log_int(rng, 256, 1024)}
    return {"kind": "tree", "paths": rng.randint(16, 64), "width": rng.randint(200, 600),
            "height": rng.randint(150, 400)}


def _rule(case):
    return rz.FillRule.EvenOdd if case["rule"] == "evenodd" else rz.FillRule.NonZero


def _settle(ctx, call):
    """Run once and wait, again where the context's buffers grew."""
    for _ in range(6):
        call()
        try:
            ctx.sync()
            return
        except rz.RzError as e:
            if e.status != _abi.RZ_E_CAPACITY:
                raise
    raise RuntimeError("the context's buffers did not settle")


# ---- inputs ---------------------------------------------------------------

def _mask_input(case, seed):
    if case["path"] == "cubics":
        ws = rz.workload_cubics64(seed & 0xffff, float(min(case["width"], case["height"])))
        return ws.paths[0], rz.Transform.identity()
    ws = rz.workload_random_walk(seed & 0xffff, case["segments"], float(max(case["width"], case["height"])))
    tr = ws.transform
    m = 0.5 * max(case["width"], case["height"])  # the walk's centre to the image's centre
    return ws.paths[0], rz.Transform.new_translate(0.5 * case["width"] - m, 0.5 * case["height"] - m) * tr


def _scene_input(case, seed):
    canvas = max(case["width"], case["height"]) / case["scale"]
    ws = rz.workload_scene(seed & 0xffff, case["paths"], canvas)
    return ws, rz.Transform.new_scale(case["scale"], case["scale"])


def _circles_input(case, seed):
    rng = np.random.default_rng(seed)
    fills = []
    for _ in range(case["paths"]):
        x, y = rng.uniform(0.0, case["size"], 2)
        path = rz.PathBuilder().move_to((x, y)).circle(rng.uniform(30.0, 40.0)).build()
        fills.append(rz.Scene.fill(path, rz.LinColor(*rng.uniform(0.0, 1.0, 3), 1.0)))
    return rz.Scene.group(fills)


def _tree_parts(case, seed):
    """The three groups of the tree, their transform, opacity and clip."""
    w, h = case["width"], case["height"]
    ws = rz.workload_scene(seed & 0xffff, case["paths"], float(max(w, h)))
    k = case["paths"] // 3
    fills = list(zip(ws.paths, ws.paints, ws.rules))
    turn = rz.Transform.new_translate(0.1 * w, 0.05 * h) * rz.Transform.new_rotate(0.2)
    clip = rz.PathBuilder().move_to((0.5 * w, 0.5 * h)).circle(0.35 * min(w, h)).build()
    # a shape over the whole window under the clip, so that its layer is the window
    pb = rz.PathBuilder().move_to((0.0, 0.0)).line_to((w, 0.0)).line_to((w, h)).line_to((0.0, h))
    sheet = (pb.close().build(), rz.LinColor(0.2, 0.3, 0.1, 0.5), rz.FillRule.NonZero)
    return fills[:k], turn, fills[k:2 * k], 0.6, [sheet] + fills[2 * k:], clip


def _tree_input(case, seed):
    plain, turn, faded, opacity, clipped, clip = _tree_parts(case, seed)
    group = lambda fl: rz.Scene(rz.Scene.GROUP, children=[rz.Scene.fill(p, q, r) for p, q, r in fl])  # noqa: E731
    return rz.Scene.group([group(plain), group(faded).with_transform(turn).with_opacity(opacity),
                           group(clipped).with_clip(clip)])


def _atlas_size(case, glyphs):
    """One size for the glyphs of every seed: half as much again as they cover
    on average, and two of the tallest rows."""
    w, h = case["atlas_width"], int(1.5 * 6250 * case["glyphs"] / case["atlas_width"]) + 256
    if glyphs.atlas_size[1] > h:
        raise RuntimeError("the glyphs need a taller atlas")
    return w, h


# ---- prepare and run -------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "mask":
        path, tr = _mask_input(case, seed)
        w, h = case["width"], case["height"]
        out = torch.zeros((h, w), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()  # the library works on a stream of its own
        s = {"kind": kind, "path": rz.DevicePath(path), "tr": tr, "out": out, "rule": _rule(case),
             "mode": MODES[case["mode"]]}
        _settle(s["path"].ctx, lambda: run(s))
        return s
    if kind == "scene":
        ws, tr = _scene_input(case, seed)
        w, h = case["width"], case["height"]
        out = torch.zeros((h, w, 4), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        s = {"kind": kind, "scene": rz.DeviceScene(ws.scene()), "tr": tr, "out": out,
             "view": (0.0, 0.0, float(w), float(h)), "bg": (0.9, 0.9, 0.85, 1.0) if case["bg"] else None}
        _settle(s["scene"].ctx, lambda: run(s))
        return s
    if kind == "atlas":
        gs = rz.workload_glyphs(seed & 0xffff, case["glyphs"], case["atlas_width"])
        w, h = _atlas_size(case, gs)
        out = torch.zeros((h, w), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        s = {"kind": kind, "glyphs": rz.DeviceGlyphs(gs.paths, gs.slots), "out": out}
        _settle(s["glyphs"].ctx, lambda: run(s))
        return s
    if kind == "diff":
        ds, tp, tc = rz.workload_diff(seed, case["paths"], case["cubics"], float(case["size"]))
        dev = rz.DeviceScene(ds.scene())
        size = float(case["size"])
        s = {"kind": kind, "scene": dev, "view": (0.0, 0.0, size, size), "tr": rz.Transform.identity(),
             "index": torch.tensor(ds.index, device="cuda"),
             "points": torch.tensor(ds.points, dtype=torch.float32, device="cuda", requires_grad=True),
             "colors": torch.tensor(ds.colors, dtype=torch.float32, device="cuda", requires_grad=True)}
        with torch.no_grad():
            s["target"] = rz.render_torch(
                dev, torch.tensor(tp, device="cuda")[s["index"]],
                torch.tensor(tc, dtype=torch.float32, device="cuda"), s["tr"], s["view"]).clone()
        run(s)  # sizes the backward's buffers
        return s
    if kind == "circles":
        size = float(case["size"])
        return {"kind": kind, "scene": _circles_input(case, seed), "view": (0.0, 0.0, size, size), "bg": None}
    if kind == "tree":
        return {"kind": kind, "scene": _tree_input(case, seed), "bg": (1.0, 1.0, 1.0, 1.0),
                "view": (0.0, 0.0, float(case["width"]), float(case["height"]))}
    raise ValueError(kind)


def run(s):
    kind = s["kind"]
    if kind == "mask":
        out = s["out"]
        s["path"].mask_device(s["tr"], out.shape[1], out.shape[0], out.data_ptr(), out.shape[1],
                              fill_rule=s["rule"], flatness=FLATNESS, edge_mode=s["mode"])
        return out
    if kind == "scene":
        out = s["out"]
        s["scene"].render_device(s["tr"], s["view"], out.data_ptr(), out.shape[1], bg=s["bg"],
                                 flatness=FLATNESS)
        return out
    if kind == "atlas":
        out = s["out"]
        s["glyphs"].mask_device(out.data_ptr(), out.shape[1], flatness=FLATNESS)
        return out
    if kind == "diff":
        s["points"].grad = s["colors"].grad = None
        out = rz.render_torch(s["scene"], s["points"][s["index"]], s["colors"], s["tr"], s["view"],
                              flatness=FLATNESS)
        loss = ((out - s["target"]) ** 2).sum()
        loss.backward()
        return {"layer": out.detach(), "points": s["points"].grad, "colors": s["colors"].grad}
    layer = s["scene"].render(rz.SignedDifferenceRasterizer(FLATNESS), rz.Transform.identity(),
                              s["view"], s["bg"])
    return layer.image


def work(case):
    """Inputs read once and outputs written once (control points at 16 bytes,
    a kind and an offset per segment; f32 masks, RGBA f32 layers)."""
    kind = case["kind"]
    if kind == "mask":
        pts = 4.0 if case["path"] == "cubics" else 3.05  # points per segment
        return {"bytes": 4.0 * case["width"] * case["height"] + case["segments"] * (16 * pts + 5), "flops": 0}
    if kind == "scene":
        # 60 segments in the median, 160 on average, a third each of 2, 3 and 4 points
        return {"bytes": 16.0 * case["width"] * case["height"] + case["paths"] * 160 * (16 * 3 + 5), "flops": 0}
    if kind == "atlas":
        # masks of side U{16..128}: 6250 pixels on average; 104 quads on average
        return {"bytes": case["glyphs"] * (4.0 * 6250 + 104 * (16 * 3 + 5)), "flops": 0}
    if kind == "diff":
        px, n = case["size"] ** 2, case["paths"] * case["cubics"]
        # layer written, its gradient read; points and their gradients twice over (f32 and f64)
        return {"bytes": 32.0 * px + n * (4 * 16 * 2 + 3 * 8 * 2), "flops": 0}
    if kind == "circles":
        return {"bytes": 16.0 * case["size"] ** 2 + case["paths"] * 4 * 69, "flops": 0}
    return {"bytes": 16.0 * case["width"] * case["height"] + case["paths"] * 160 * 53, "flops": 0}


def tolerance(case):
    # measured against exact(): masks and atlases up to 6.4e-7, layers 1.6e-7,
    # gradients 6.8e-7 (and 1.9e-7 between two runs: f32 atomics)
    return {"rel": 6e-6 if case["kind"] == "diff" else 2.5e-6}


# ---- the result in 64 bits ---------------------------------------------------

DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64 = dict(dtype=torch.float64, device=DEV)


def _flatten_segments(ctrl):
    """Leaves of the reference's subdivision (flatness below 16 tol^2, split
    at t = 1/2) of every curve of ctrl (n, K, 2): curve index, t0, t1, lines."""
    fl = 16.0 * FLATNESS * FLATNESS
    n, k = ctrl.shape[0], ctrl.shape[1]
    node, seg = ctrl, torch.arange(n, device=ctrl.device)
    t0, dt = torch.zeros(n, **F64), 1.0
    out = []
    while node.shape[0]:
        if k == 2:
            flat = torch.ones(node.shape[0], dtype=torch.bool, device=ctrl.device)
        elif k == 3:
            d = 2.0 * node[:, 1] - node[:, 0] - node[:, 2]
            flat = (d * d).sum(1) < fl
        else:
            u = 3.0 * node[:, 1] - 2.0 * node[:, 0] - node[:, 3]
            v = 3.0 * node[:, 2] - node[:, 0] - 2.0 * node[:, 3]
            flat = torch.maximum(u * u, v * v).sum(1) < fl
        leaf = node[flat]
        out.append((seg[flat], t0[flat], t0[flat] + dt, torch.cat([leaf[:, 0], leaf[:, -1]], 1)))
        node, seg, t0 = node[~flat], seg[~flat], t0[~flat]
        dt *= 0.5
        # de Casteljau at 1/2: the left and right control points
        left, right, cur = [node[:, 0]], [node[:, -1]], node
        for _ in range(k - 1):
            cur = 0.5 * (cur[:, :-1] + cur[:, 1:])
            left.append(cur[:, 0])
            right.append(cur[:, -1])
        node = torch.cat([torch.stack(left, 1), torch.stack(right[::-1], 1)])
        seg, t0 = torch.cat([seg, seg]), torch.cat([t0, t0 + dt])
    return tuple(torch.cat(p) for p in zip(*out))


def _path_lines(path, tr):
    """(n, 4) lines of a path under tr, closing lines included."""
    m = tr.m
    p = torch.tensor(path.points.reshape(-1, 2), **F64)
    p = torch.stack([p[:, 0] * m[0] + p[:, 1] * m[1] + m[2], p[:, 0] * m[3] + p[:, 1] * m[4] + m[5]], 1)
    kinds, offs = path.kinds.astype(np.int64), path.point_offsets.astype(np.int64)
    lines = []
    for kind in (0, 1, 2):
        first = torch.tensor(offs[:-1][kinds == kind], device=DEV)
        if first.numel():
            ctrl = p[first[:, None] + torch.arange(kind + 2, device=DEV)]
            lines.append(_flatten_segments(ctrl)[3])
    sub = path.subpaths.astype(np.int64)
    if len(sub) > 1:
        a = p[torch.tensor(offs[sub[1:]] - 1, device=DEV)]
        b = p[torch.tensor(offs[sub[:-1]], device=DEV)]
        lines.append(torch.cat([a, b], 1))
    return torch.cat(lines) if lines else torch.zeros((0, 4), **F64)


def _split(L, x):
    """Each line cut where it crosses the abscissa x (two pieces in all cases)."""
    x0, y0, x1, y1 = L.unbind(1)
    cross = (x0 - x) * (x1 - x) < 0
    dx = torch.where(cross, x1 - x0, torch.ones_like(x0))
    t = torch.where(cross, (x - x0) / dx, torch.ones_like(x0))
    xm = torch.where(cross, torch.full_like(x0, float(x)), x1)
    ym = y0 + t * (y1 - y0)
    return torch.cat([torch.stack([x0, y0, xm, ym], 1),
                      torch.stack([xm, ym, x1, y1], 1)[cross]])


def _winding(L, W, H, wc):
    """Box-filtered winding (H, W) of the lines: the reference's signed area
    accumulation; wc: its right clip abscissa (None: ActiveEdgeRasterizer)."""
    acc = torch.zeros(H * (W + 2), **F64)
    for part in torch.split(L, 500_000):
        acc = acc + _deposits(part, W, H, wc)
    return acc.view(H, W + 2).cumsum(1)[:, :W]


def _deposits(L, W, H, wc):
    if wc is not None:
        # a line wholly beyond wc becomes a vertical one at wc - 0.001; the
        # part beyond of a line that crosses wc is dropped
        x0, y0, x1, y1 = L.unbind(1)
        o0, o1 = x0 > wc, x1 > wc
        both, some = o0 & o1, o0 ^ o1
        dx = torch.where(some, x1 - x0, torch.ones_like(x0))
        ym = y0 + (wc - x0) / dx * (y1 - y0)
        far = torch.full_like(x0, wc - 0.001)
        nx0 = torch.where(both, far, torch.where(some & o0, torch.full_like(x0, wc), x0))
        nx1 = torch.where(both, far, torch.where(some & o1, torch.full_like(x0, wc), x1))
        L = torch.stack([nx0, torch.where(some & o0, ym, y0), nx1, torch.where(some & o1, ym, y1)], 1)
    else:
        L = _split(L, float(W))
    L = _split(L, 0.0)
    x0, y0, x1, y1 = L.unbind(1)
    x0, x1 = x0.clamp(0.0, float(W)), x1.clamp(0.0, float(W))
    up = y0 > y1
    xa, ya = torch.where(up, x1, x0), torch.where(up, y1, y0)
    xb, yb = torch.where(up, x0, x1), torch.where(up, y0, y1)
    sign = torch.where(up, -1.0, 1.0).to(torch.float64)
    keep = (yb > ya) & (yb > 0) & (ya < H)
    xa, ya, xb, yb, sign = xa[keep], ya[keep], xb[keep], yb[keep], sign[keep]
    slope = (xb - xa) / (yb - ya)
    lo, hi = ya.clamp(min=0.0), yb.clamp(max=float(H))
    # one piece per pixel row
    r0 = lo.detach().floor()
    n = (hi.detach().ceil() - r0).clamp(min=1).long()
    i = torch.repeat_interleave(torch.arange(n.numel(), device=L.device), n)
    r = r0[i] + (torch.arange(i.numel(), device=L.device) - (n.cumsum(0) - n)[i])
    top, bot = torch.maximum(lo[i], r), torch.minimum(hi[i], r + 1.0)
    d = sign[i] * (bot - top)
    xt, xe = xa[i] + (top - ya[i]) * slope[i], xa[i] + (bot - ya[i]) * slope[i]
    # one part per pixel column
    left, right = torch.minimum(xt, xe), torch.maximum(xt, xe)
    c0 = left.detach().floor()
    m = (right.detach().ceil() - c0).clamp(min=1).long()
    j = torch.repeat_interleave(torch.arange(m.numel(), device=L.device), m)
    c = c0[j] + (torch.arange(j.numel(), device=L.device) - (m.cumsum(0) - m)[j])
    pl, pr = torch.maximum(left[j], c), torch.minimum(right[j], c + 1.0)
    width = right - left
    wide = width > 0
    share = torch.where(wide[j], (pr - pl) / torch.where(wide, width, torch.ones_like(width))[j],
                        torch.ones_like(pl))
    dd, xm = d[j] * share, 0.5 * (pl + pr) - c
    at = (r[j] * (W + 2) + c).long()
    ok = (c >= 0) & (c <= W) & (r[j] >= 0) & (r[j] < H)
    acc = torch.zeros(H * (W + 2), **F64)
    acc = acc.index_add(0, at[ok], (dd * (1.0 - xm))[ok])
    return acc.index_add(0, at[ok] + 1, (dd * xm)[ok])


def _alpha(w, rule):
    if rule == rz.FillRule.NonZero:
        a = w.abs().clamp(max=1.0)
        return torch.where(a < 1e-6, torch.zeros_like(a), a)
    return (torch.remainder(w + 1.0, 2.0) - 1.0).abs()


def _l2s(x):
    x1 = x.sqrt()
    x2 = x1.sqrt()
    x3 = x2.sqrt()
    high = -0.01848558 * x + 0.6445592 * x1 + 0.70994765 * x2 - 0.33605254 * x3
    return torch.where(x <= 0.0031308, x * 12.92, high)


def _s2l(v):
    u = 2.0843103538116825 * v - 1.0843103538116827
    high = 0.23361048543711943 + 0.4665843122387033 * u + 0.26901741378006355 * u * u + \
        0.031661580753065945 * u ** 3
    return torch.where(v <= 0.04045, v * 0.07739938080495357, high)


def _through(c, f):
    """f of the unmultiplied colours, every lane, times alpha."""
    a = c[..., 3:4]
    u = torch.where(a <= 1e-6, torch.zeros_like(c), c / torch.where(a <= 1e-6, torch.ones_like(a), a))
    return f(u) * a


def _paint(paint, tr, xs, ys):
    """Colours (len(ys), len(xs), 4) of a user-space, padded paint at pixel centres."""
    if isinstance(paint, rz.LinColor):
        return torch.tensor(list(paint), **F64).expand(len(ys), len(xs), 4)
    p = paint.p
    if p.kind == _abi.RZ_PAINT_SOLID:
        return torch.tensor(list(p.color), **F64).expand(len(ys), len(xs), 4)
    m = np.array([[tr.m[0], tr.m[1], tr.m[2]], [tr.m[3], tr.m[4], tr.m[5]], [0, 0, 1.0]])
    inv = np.linalg.inv(m)
    X, Y = xs[None, :] + 0.5, ys[:, None] + 0.5
    ux, uy = inv[0, 0] * X + inv[0, 1] * Y + inv[0, 2], inv[1, 0] * X + inv[1, 1] * Y + inv[1, 2]
    if p.kind == _abi.RZ_PAINT_LINEAR:
        dx, dy = p.end[0] - p.start[0], p.end[1] - p.start[1]
        t = ((ux - p.start[0]) * dx + (uy - p.start[1]) * dy) / (dx * dx + dy * dy)
    else:  # the focus at the centre with radius 0
        t = torch.sqrt((ux - p.center[0]) ** 2 + (uy - p.center[1]) ** 2) / p.radius
    pos = torch.tensor(paint.pos, **F64)
    col = _through(torch.tensor(paint.col.reshape(-1, 4), **F64), _l2s)
    k = torch.searchsorted(pos, t.contiguous())  # stops before t
    k0, k1 = (k - 1).clamp(0, len(pos) - 1), k.clamp(0, len(pos) - 1)
    gap = pos[k1] - pos[k0]
    f = torch.where(gap > 0, (t - pos[k0]) / torch.where(gap > 0, gap, torch.ones_like(gap)),
                    torch.zeros_like(t))[..., None]
    return _through(col[k1] * f + col[k0] * (1.0 - f), _s2l)


def _draw_fills(layer, fills, tr):
    """fills (path, paint, rule) over the layer (H, W, 4), in order."""
    H, W = layer.shape[:2]
    for path, paint, rule in fills:
        L = _path_lines(path, tr)
        if not L.numel():
            continue
        lo = torch.minimum(L[:, :2], L[:, 2:]).amin(0).floor().tolist()
        hi = torch.maximum(L[:, :2], L[:, 2:]).amax(0).ceil().tolist()
        x0, y0 = max(0, int(lo[0])), max(0, int(lo[1]))
        x1, y1 = min(W, int(hi[0]) + 1), min(H, int(hi[1]) + 1)
        if x0 >= x1 or y0 >= y1:
            continue
        shift = torch.tensor([x0, y0, x0, y0], **F64)
        a = _alpha(_winding(L - shift, x1 - x0, y1 - y0, float(W - x0)), rule)[..., None]
        c = _paint(paint, tr, torch.arange(x0, x1, **F64), torch.arange(y0, y1, **F64)) * a
        dst = layer[y0:y1, x0:x1]
        layer[y0:y1, x0:x1] = torch.where(a >= 1e-6, c + dst * (1.0 - c[..., 3:4]), dst)
    return layer


def _blank(w, h, bg):
    return torch.tensor(bg or (0.0, 0.0, 0.0, 0.0), dtype=torch.float32).to(**F64).expand(h, w, 4).clone()


def exact(case, seed):
    kind = case["kind"]
    ident = rz.Transform.identity()
    if kind == "mask":
        if case["mode"] == "active":
            # ActiveEdgeRasterizer moves a row's deposits one column right where
            # rounding left an edge a hair left of x = 0: no 64-bit value
            return None
        path, tr = _mask_input(case, seed)
        w, h = case["width"], case["height"]
        wc = float(w - 1) if case["mode"] == "mask" else float(w)
        return _alpha(_winding(_path_lines(path, tr), w, h, wc), _rule(case))
    if kind == "scene":
        if case["paths"] > 1500:
            return None  # minutes
        ws, tr = _scene_input(case, seed)
        layer = _blank(case["width"], case["height"], (0.9, 0.9, 0.85, 1.0) if case["bg"] else None)
        return _draw_fills(layer, zip(ws.paths, ws.paints, ws.rules), tr)
    if kind == "circles":
        layer = _blank(case["size"], case["size"], None)
        return _draw_fills(layer, _circles_input(case, seed).fills(), ident)
    if kind == "tree":
        w, h = case["width"], case["height"]
        plain, turn, faded, opacity, clipped, clip = _tree_parts(case, seed)
        over = lambda dst, src: src + dst * (1.0 - src[..., 3:4])  # noqa: E731
        layer = _draw_fills(_blank(w, h, (1.0, 1.0, 1.0, 1.0)), plain, ident)
        layer = over(layer, _draw_fills(_blank(w, h, None), faded, turn) * opacity)
        # the clip node's layer ends at its path's box, where its right clip is
        lines = _path_lines(clip, ident)
        edge = int(lines[:, ::2].max().ceil())
        mask = _alpha(_winding(lines, edge, h, float(edge - 1)), rz.FillRule.NonZero)
        part = _draw_fills(_blank(edge, h, None), clipped, ident) * mask[..., None]
        layer[:, :edge] = over(layer[:, :edge], part)
        return layer
    if kind == "atlas":
        if case["glyphs"] > 2000:
            return None  # a minute
        gs = rz.workload_glyphs(seed & 0xffff, case["glyphs"], case["atlas_width"])
        w, h = _atlas_size(case, gs)
        out = torch.zeros((h, w), **F64)
        for path, s in zip(gs.paths, gs.slots):
            L = _path_lines(path, ident)
            out[s.y:s.y + s.height, s.x:s.x + s.width] = _alpha(
                _winding(L, s.width, s.height, float(s.width - 1)), rz.FillRule.NonZero)
        return out
    if kind == "diff":
        if case["paths"] * case["size"] ** 2 > 16 * 400 ** 2:
            return None  # autograd's graph would not fit
        return _diff_exact(case, seed)
    return None


def _diff_layer(pts, cols, index, n_cubics, size):
    """The layer of closed cubic paths as a differentiable function of their
    unique points and colours (subdivision parameters held fixed)."""
    stored = pts[index].view(-1, n_cubics, 4, 2)
    layer = torch.zeros((size, size, 4), **F64)
    for k in range(stored.shape[0]):
        c = stored[k]
        seg, t0, t1, _ = _flatten_segments(c.detach())

        def at(t):
            u = 1.0 - t
            w = torch.stack([u ** 3, 3 * t * u * u, 3 * t * t * u, t ** 3], 1)
            return (w[:, :, None] * c[seg]).sum(1)
        a = _alpha(_winding(torch.cat([at(t0), at(t1)], 1), size, size, None), rz.FillRule.NonZero)
        s = cols[k] * a[..., None]
        layer = torch.where(a[..., None] >= 1e-6, s + layer * (1.0 - s[..., 3:4]), layer)
    return layer


def _diff_exact(case, seed):
    ds, tp, tc = rz.workload_diff(seed, case["paths"], case["cubics"], float(case["size"]))
    index = torch.tensor(ds.index, device=DEV)
    args = (index, case["cubics"], case["size"])
    with torch.no_grad():
        target = _diff_layer(torch.tensor(tp, **F64), torch.tensor(np.float32(tc), device=DEV).double(), *args)
    pts = torch.tensor(np.float32(ds.points), device=DEV).double().requires_grad_(True)
    cols = torch.tensor(np.float32(ds.colors), device=DEV).double().requires_grad_(True)
    layer = _diff_layer(pts, cols, *args)
    ((layer - target) ** 2).sum().backward()
    return {"layer": layer.detach(), "points": pts.grad, "colors": cols.grad}
