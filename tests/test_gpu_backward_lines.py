"""The adjoint's line pass: lines of every direction and place against central
differences of the oracle's coverage (a loss linear in it), and the deeper
split that short launches take against the flatten's own."""
import numpy as np
import pytest

import _oracle as O
from _diffscene import blob_scene
from rasterize_amd import DeviceScene, LinColor, Path, Scene, Transform, render_torch, _abi

pytestmark = pytest.mark.gpu
I = Transform.identity()

POLYGONS = {
    # one pixel; within a row; within a column
    "pixel": [(5.2, 7.1), (5.9, 7.3), (5.4, 7.8)],
    "flat": [(2.3, 7.1), (44.7, 7.4), (20.2, 7.9)],
    "thin": [(9.2, 1.1), (9.7, 40.3), (9.4, 22.8)],
    # exactly vertical, and all but
    "vertical": [(5.5, 3.25), (30.5, 3.75), (30.5, 41.5), (5.5, 40.25)],
    "steep": [(5.5, 3.25), (30.5, 3.75), (30.5 + 1e-13, 41.5), (5.5 + 4e-16 * 8, 40.25)],
    # beyond every edge of the image
    "outside": [(-20.3, 10.2), (24.4, -13.7), (77.6, 30.3), (21.9, 66.1)],
    "left": [(-9.7, 4.3), (0.4, 20.6), (-0.3, 44.2)],
    # long shallow lines, both directions
    "shallow": [(1.3, 4.4), (46.2, 9.7), (2.1, 14.9), (45.3, 21.2), (1.7, 30.6)],
}


@pytest.mark.parametrize("name", sorted(POLYGONS))
def test_lines_match_central_differences(name):
    import torch
    W, H = 48, 45
    poly = np.array(POLYGONS[name])
    n = len(poly)
    idx = np.stack([np.arange(n), (np.arange(n) + 1) % n], 1).reshape(-1)

    def path(v):
        return Path(np.zeros(n, np.uint8), 2 * np.arange(n + 1, dtype=np.uint32), v[idx].reshape(-1),
                    np.array([0, n], np.uint32), np.array([1], np.uint8))

    G = np.random.default_rng(3).uniform(-1.0, 1.0, (H, W))

    def loss(v):
        return float((G * O.sd_mask_iter(path(v), I, W, H, 0)).sum())

    h = 1e-5
    fd = np.zeros((n, 2))
    for i in range(n):
        for d in range(2):
            up, um = poly.copy(), poly.copy()
            up[i, d] += h
            um[i, d] -= h
            fd[i, d] = (loss(up) - loss(um)) / (2 * h)

    dev = DeviceScene(Scene.group([Scene.fill(path(poly), LinColor(0.0, 0.0, 0.0, 1.0))]))
    U = torch.tensor(poly, dtype=torch.float64, device="cuda", requires_grad=True)
    c = torch.tensor([[0.0, 0.0, 0.0, 1.0]], device="cuda")
    out = render_torch(dev, U[torch.tensor(idx, device="cuda")], c, I, (0.0, 0.0, float(W), float(H)))
    (out[..., 3] * torch.tensor(G, dtype=torch.float32, device="cuda")).sum().backward()
    # The slope is itself continuous: moving an end by h changes the line's
    # length inside a pixel by at most h * max(1, |dy/dx|), once per column it
    # crosses, and G changes by at most 2 there. Every polygon has at most
    # 2 * 33 * 1 ("left") or 2 * 1 * 48 times h = 1e-5, so under 1e-3; a line
    # beyond the right edge moves the last pixel by 0.001 of its height (the
    # reference's clip at W - 0.001), which the adjoint leaves out; float32 sums
    # and the 2^-20 coverage are below 1e-4.
    assert np.abs(U.grad.cpu().numpy() - fd).max() <= 2e-3 * max(1.0, np.abs(fd).max())


@pytest.mark.parametrize("n_paths,n_cubics", [(1, 2), (3, 9), (1, 700), (40, 16)])
def test_deeper_split_gives_the_same_gradients(n_paths, n_cubics):
    """(1, 2) and (3, 9) are launches of less than a wave per SIMD; the depth
    only decides which lane integrates a line."""
    import torch
    ds = blob_scene(2, n_paths, n_cubics, 160.0)
    idx = torch.tensor(ds.index, device="cuda")
    G = torch.tensor(np.random.default_rng(4).uniform(-1, 1, (160, 160, 4)), dtype=torch.float32, device="cuda")

    def grads(fixed):
        dev = DeviceScene(ds.scene())
        if fixed is not None:
            dev.ctx.set_param(_abi.RZ_PARAM_SPLIT_CUBIC, fixed)  # (turns the choice per call off)
        try:
            U = torch.tensor(ds.points, dtype=torch.float64, device="cuda", requires_grad=True)
            c = torch.tensor(ds.colors, device="cuda")
            out = render_torch(dev, U[idx], c, I, (0.0, 0.0, 160.0, 160.0))
            (out * G).sum().backward()
            return U.grad.cpu().numpy()
        finally:
            if fixed is not None:
                dev.ctx.set_param(_abi.RZ_PARAM_SPLIT_CUBIC, 4)
                dev.ctx.set_param(_abi.RZ_PARAM_SPLIT_AUTO, 1)

    auto = grads(None)
    for fixed in (0, 3):
        g = grads(fixed)
        # the same lines' integrals (G is at most 1, a line's at most its
        # height), summed in float32 over at most 64 lanes a curve in another
        # order
        assert np.abs(g - auto).max() <= 64 * 2.0 ** -23 * max(1.0, np.abs(auto).max())
