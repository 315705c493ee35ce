"""Gradients of the differentiable fill that large ones beside them must not
touch, component by component against FP64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _line_cubics(corners):
    """Control points of a path along straight lines through `corners`."""
    c = np.asarray(corners, np.float64)
    out = [c[:1]]
    for a, b in zip(c[:-1], c[1:]):
        out.append(np.stack([a + (b - a) / 4.0, a + (b - a) * 0.75, b]))
    return np.concatenate(out)


def _grads(w, h, cubics, points, colours, cotangent):
    """d points, d colours on the GPU and in FP64."""
    from footile_amd.diff import DiffRenderer, device_array
    from footile_amd.plotter import DeviceBuffer
    from oracle import pydiff as pd
    image, cubics = np.zeros(len(cubics), np.uint32), np.asarray(cubics, np.uint32)
    points, colours = points.astype(np.float32), np.asarray(colours, np.float32)
    r = DiffRenderer(1, w, h, image, cubics)
    gp, gc = DeviceBuffer(8 * r.n_points), DeviceBuffer(16 * r.n_paths)
    r.backward(device_array(points), device_array(colours), device_array(cotangent), gp, gc)
    _, want_gp, want_gc = pd.Scene(1, w, h, image, cubics).backward(points, colours, grad_canvas=cotangent)
    return (gp.download(dtype=np.float32).reshape(-1, 2), gc.download(dtype=np.float32).reshape(-1, 4), want_gp,
            want_gc)


@pytest.mark.parametrize("size", [1.0e6, np.inf])
# the second figure's left side: right after the first's, at either side of a
# row of 16 and of a chunk of 64 columns, in a later chunk and a later tile
@pytest.mark.parametrize("left", [9, 15, 16, 31, 47, 48, 62, 63, 64, 100, 127, 200, 255, 256, 300])
def test_large_cotangent_left_of_an_edge(oracle, size, left):
    """One path of two figures, joined by horizontal edges (which have no
    pieces).  A large cotangent on a pixel of the first figure's left side, in
    the row of the second figure's top corners, whose y gradients no edge
    beside them cancels; cotangents of 1 in every pixel the second figure
    crosses.  The gradients of the second figure's points are sums of at most
    10 rows of 12 pixels, each of order 1: 1e-5 of the largest, with vertex
    rounding (2^-24 of coordinates up to 320, 2e-5 of a pixel) on top.  FP64
    takes the large pixel as 0: it lies left of them all."""
    w, h = 320, 20
    a, b = left + 0.375, left + 9.75
    corners = [(4.5, 2.0), (4.25, 17.0), (7.5, 17.0), (a + 1.0, 17.0), (b, 17.0), (b - 1.0, 8.25), (a, 8.25),
               (a + 1.0, 17.0), (7.5, 17.0), (7.25, 2.0), (4.5, 2.0)]
    pts = _line_cubics(corners)
    cubics, colours = [len(corners) - 1], [[0.3, 0.2, 0.1, 0.5]]
    cot = np.zeros((1, h, w, 4), np.float32)
    cot[0, 8:17, left:left + 11] = 1.0
    _, _, want, _ = _grads(w, h, cubics, pts, colours, cot)
    cot[0, 8, 4] = size
    with np.errstate(invalid="ignore"):
        gp, _, _, _ = _grads(w, h, cubics, pts, colours, cot)
    # the points of the second figure's cubics: its bottom, right side, top and left side
    own = np.arange(3 * 3 + 1, 3 * 7)
    assert np.isfinite(gp[own]).all()
    assert np.abs(want[own]).max() > 1.0
    assert np.abs(gp[own] - want[own]).max() < 1e-4 * np.abs(want[own]).max()


@pytest.mark.parametrize("x0", [8, 64, 256])  # inside a chunk, at a chunk's and a tile's border
@pytest.mark.parametrize("eps", [2.0 ** -10, 2.0 ** -13, 2.0 ** -14])
@pytest.mark.parametrize("flip", [False, True])
def test_sliver_of_a_pixel_keeps_its_gradient(oracle, x0, eps, flip):
    """A tip that reaches `eps` into the pixel left of column x0 and covers
    0.21 eps^2 of it, down to 7.8e-10 (each of the tip's two edges half of
    that), at either orientation, between a path below and one above it: the
    pixel's value and the gradients of its cotangent, component by component.
    The tip's x is off by at most 2^-21 below column 8 and by less of the
    spacing of float32 right of that (2^-7 of the smallest eps), the coverage
    by twice that: 3 %."""
    w, h = 300, 9
    corners = [(x0 - eps, 4.5), (x0 + 6.0, 5.75), (x0 + 6.0, 3.25), (x0 - eps, 4.5)]
    box = [(x0 - 4.0, 1.5), (x0 - 4.0, 7.5), (x0 + 9.0, 7.5), (x0 + 9.0, 1.5), (x0 - 4.0, 1.5)]
    pts = np.concatenate([_line_cubics(box), _line_cubics(corners[::-1] if flip else corners), _line_cubics(box)])
    cubics, colours = [4, 3, 4], [[0.1, 0.3, 0.2, 0.4], [0.3, 0.2, 0.1, 0.5], [0.2, 0.1, 0.3, 0.6]]
    cot = np.zeros((1, h, w, 4), np.float32)
    cot[0, 4, x0 - 1] = [1.0, 0.5, -0.25, 0.75]
    gp, gc, want_gp, want_gc = _grads(w, h, cubics, pts, colours, cot)
    own = slice(13, 23)
    assert np.abs(want_gp[own]).max() > 0.01 * eps
    assert np.abs(gp[own] - want_gp[own]).max() < 0.03 * np.abs(want_gp[own]).max()
    assert np.abs(gc[1] - want_gc[1]).max() < 0.03 * np.abs(want_gc[1]).max()


@pytest.mark.parametrize("low", [2.0 ** -25, 2.0 ** -30, 2.0 ** -40])
def test_low_pieces_keep_their_gradient(oracle, low):
    """A box that reaches `low` into row 0 from above: the row's pixels are
    covered by that much, and the gradient of the box's lower side is 1 a
    pixel, as far as float32 has such a y.  Beside it a path whose pieces are
    whole.  Components within 1e-5 of the largest (sums of 200 equal terms)."""
    w, h = 260, 3
    box = [(20.0, -2.0), (20.0, low), (220.0, low), (220.0, -2.0), (20.0, -2.0)]
    other = [(5.0, 0.0), (5.0, 3.0), (250.0, 3.0), (250.0, 0.0), (5.0, 0.0)]
    pts = np.concatenate([_line_cubics(other), _line_cubics(box)])
    cot = np.zeros((1, h, w, 4), np.float32)
    cot[0, 0] = [1.0, 0.5, -0.25, 0.75]
    gp, _, want_gp, _ = _grads(w, h, [4, 4], pts, [[0.1, 0.3, 0.2, 0.4], [0.3, 0.2, 0.1, 0.5]], cot)
    own = slice(13, 26)
    assert np.abs(want_gp[own, 1]).max() > 10.0
    assert np.abs(gp[own] - want_gp[own]).max() < 1e-5 * np.abs(want_gp[own]).max()


@pytest.mark.parametrize("paths", [3, 15, 16, 17, 33])
@pytest.mark.parametrize("tips", [1, 2, 3])
def test_many_slivers_in_a_row(oracle, paths, tips):
    """`paths` paths of `tips` tips as above in one row, two tiny shares a tip:
    up to and past the 32 that a round of 16 paths lists.  Each path's
    gradients, component by component (3 %, as above)."""
    w, h, eps = 40, 9, 2.0 ** -13
    corners = []
    for x0 in (8, 16, 24)[:tips]:  # joined by edges along y = 4.5, which have no pieces
        corners += [(x0 - eps, 4.5), (x0 + 6.0, 5.75), (x0 + 6.0, 3.25), (x0 - eps, 4.5)]
    corners.append(corners[0])
    path = _line_cubics(corners)
    g = np.random.default_rng(paths + tips)
    a = g.uniform(0.3, 0.9, (paths, 1))
    colours = np.concatenate([a * g.random((paths, 3)), a], axis=1)
    cot = np.zeros((1, h, w, 4), np.float32)
    cot[0, 4, [7, 15, 23]] = [1.0, 0.5, 0.25, 0.75]
    gp, gc, want_gp, want_gc = _grads(w, h, [len(corners) - 1] * paths, np.tile(path, (paths, 1)), colours, cot)
    got, want = gp.reshape(paths, -1), want_gp.reshape(paths, -1)
    assert (np.abs(want).max(axis=1) > 0.01 * eps).all()
    assert (np.abs(got - want).max(axis=1) < 0.03 * np.abs(want).max(axis=1)).all()
    assert (np.abs(gc - want_gc).max(axis=1) < 0.03 * np.abs(want_gc).max(axis=1)).all()


@pytest.mark.parametrize("x0", [0.004, 0.1, 0.3, 1.3, 60.2])  # column 0, where x is finer than 1 - x, and others
@pytest.mark.parametrize("slope", [1.2e-5, 4.0e-5, 3.0e-4, 5.0e-3])  # ramp width a row; 1e-5 and narrower take the midpoint
def test_near_vertical_edges(oracle, x0, slope):
    """The canvas and the gradients of a figure whose sides lean by `slope` a
    row.  A side's x is rounded at 2^-24 of it, a ramp's width by the same, so
    that the partials of M, about 1/2 each, are off by 2^-23 x0 / slope
    (half of it a side, either way) and by some 2^-22: bounds of 4 times that
    sum, and 2e-5 for the canvas."""
    w, h = 70, 18
    corners = [(x0, 1.5), (x0 + 14 * slope, 15.5), (x0 + 6.0 - 14 * slope, 15.5), (x0 + 6.0, 1.5), (x0, 1.5)]
    pts = _line_cubics(corners).astype(np.float32)
    cubics, colours = [4], np.array([[0.3, 0.2, 0.1, 0.5]], np.float32)
    cot = np.random.default_rng(5).uniform(0.2, 1.0, (1, h, w, 4)).astype(np.float32)
    gp, gc, want_gp, want_gc = _grads(w, h, cubics, pts, colours, cot)
    bound = 4.0 * (2.0 ** -23 * (x0 + 6.0) / slope + 2.0 ** -22)
    assert np.abs(gp - want_gp).max() < bound * np.abs(want_gp).max()
    assert np.abs(gc - want_gc).max() < 1e-5 * np.abs(want_gc).max()
    from footile_amd.diff import DiffRenderer, device_array
    from oracle import pydiff as pd
    image = np.zeros(1, np.uint32)
    r = DiffRenderer(1, w, h, image, np.asarray(cubics, np.uint32))
    canvas = r.new_canvas()
    r.forward(device_array(pts), device_array(colours), canvas)
    _, want = pd.Scene(1, w, h, image, np.asarray(cubics, np.uint32)).forward(pts, colours)
    assert np.abs(canvas.download(dtype=np.float32).reshape(r.canvas_shape) - want).max() < 2e-5
