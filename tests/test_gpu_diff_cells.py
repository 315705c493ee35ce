"""The differentiable fill's cell coverage at the sizes where it can go wrong:
tile and wavefront edges, more paths than one staging round holds, ramps of
one column and of hundreds, rows with more pieces than 32-bit cells take, and
pieces without a number.

Tolerances, before any run: the canvas is float32 within 2e-5 of FP64 for
paths of up to ~10 pieces per row (as in test_gpu_diff.py).  A pixel's
coverage error is the sum of its pieces' vertex rounding (2^-24 of the
coordinate each), so a row of n pieces gets sqrt(n / 10) times that.
Gradients: normwise 1e-4, the differentiable path's bound.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _scene(seed, w, h, paths, cubics, n_images=1, points=None):
    from footile_amd.diffscene import DiffScene
    g = np.random.default_rng(seed)
    image = np.repeat(np.arange(n_images, dtype=np.uint32), paths)
    cub = np.full(len(image), cubics, np.uint32)
    n = int(np.sum(1 + 3 * cub.astype(np.int64)))
    pts = g.uniform(-3.0, [w + 3.0, h + 3.0], size=(n, 2)) if points is None else points(g, n)
    a = g.uniform(0.3, 0.9, size=len(image))
    col = np.stack([a * g.uniform(0, 1, len(image)) for _ in range(3)] + [a], axis=1).astype(np.float32)
    return DiffScene(n_images, w, h, image, cub, pts.astype(np.float32), col)


def _step(sc, target):
    from footile_amd.diff import DiffRenderer, device_array
    from footile_amd.plotter import DeviceBuffer
    r = DiffRenderer.for_scene(sc)
    P, C, T = device_array(sc.points), device_array(sc.colours), device_array(target)
    canvas, gcan = r.new_canvas(), r.new_canvas()
    gp, gc = DeviceBuffer(8 * r.n_points), DeviceBuffer(16 * r.n_paths)
    loss = r.step(P, C, T, canvas, gcan, gp, gc)
    return (loss, canvas.download(dtype=np.float32).reshape(r.canvas_shape),
            gp.download(dtype=np.float32).reshape(-1, 2), gc.download(dtype=np.float32).reshape(-1, 4))


def _rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def _check(sc, pieces=10):
    from oracle import pydiff as pd
    target = np.random.default_rng(1).uniform(0, 1, size=(sc.n_images, sc.height, sc.width, 4)).astype(np.float32)
    o = pd.Scene(sc.n_images, sc.width, sc.height, sc.path_image, sc.path_cubics)
    want_loss, want_gp, want_gc = o.backward(sc.points, sc.colours, target)
    _, want = o.forward(sc.points, sc.colours)
    loss, canvas, gp, gc = _step(sc, target)
    assert np.abs(canvas - want).max() < 2e-5 * np.sqrt(max(pieces, 10) / 10)
    assert abs(loss - want_loss) <= 1e-5 * abs(want_loss)
    assert _rel(gp, want_gp) < 1e-4 and _rel(gc, want_gc) < 1e-4


@pytest.mark.parametrize("w,h,paths,cubics,images", [
    (1, 7, 3, 2, 1), (63, 9, 15, 2, 1), (64, 9, 16, 2, 2), (65, 9, 17, 2, 1), (255, 5, 4, 3, 1), (257, 5, 4, 3, 1),
    (513, 4, 5, 2, 1), (40, 6, 255, 1, 1), (40, 6, 257, 1, 1), (33, 5, 273, 1, 2), (24, 1, 40, 4, 1)])
def test_tile_and_round_edges(oracle, w, h, paths, cubics, images):
    _check(_scene(w + paths, w, h, paths, cubics, images))


@pytest.mark.parametrize("w,h,paths,cubics", [
    (8, 4, 1024, 1), (8, 4, 1025, 1), (8, 3, 2500, 1),  # one and several paths per geometry block
    (4, 255, 3, 2), (4, 257, 3, 2),  # one and two rows per thread
    (20, 10, 3, 127), (20, 10, 3, 128)])  # 2,033 and 2,049 edges: either side of the one-launch limit
def test_geometry_sizes(oracle, w, h, paths, cubics):
    _check(_scene(w + h + paths, w, h, paths, cubics), pieces=0.6 * cubics + 17.0 * cubics / h)


def _canvas(sc):
    from footile_amd.diff import DiffRenderer, device_array
    r = DiffRenderer.for_scene(sc)
    canvas = r.new_canvas()
    r.forward(device_array(sc.points), device_array(sc.colours), canvas)
    return canvas.download(dtype=np.float32).reshape(r.canvas_shape)


def test_geometry_forms_agree(oracle):
    """The one-launch geometry and the general form (images past 8,192 rows,
    paths past 2,048 edges) give the same bytes: coverage does not depend on
    the order of a row's pieces."""
    import dataclasses
    tall = _scene(11, 5, 8192, 6, 3)
    assert np.array_equal(_canvas(tall)[0], _canvas(dataclasses.replace(tall, height=8193))[0, :8192])
    sc = _scene(12, 90, 40, 30, 4)
    # one more path, last, of 2,081 edges and outside the image
    g = np.random.default_rng(13)
    far = g.uniform(200.0, 300.0, size=(1 + 3 * 130, 2)).astype(np.float32)
    more = dataclasses.replace(sc, path_image=np.append(sc.path_image, 0).astype(np.uint32),
                               path_cubics=np.append(sc.path_cubics, 130).astype(np.uint32),
                               points=np.concatenate([sc.points, far]),
                               colours=np.concatenate([sc.colours, sc.colours[:1]]))
    assert np.array_equal(_canvas(sc), _canvas(more))


def test_wide_and_narrow_ramps(oracle):
    """Outlines whose edges cross hundreds of columns in a row or none."""
    def points(g, n):
        x = np.where(np.arange(n) % 4 < 2, g.uniform(-20.0, 700.0, n), g.integers(0, 600, n))
        return np.stack([x, g.uniform(0.2, 5.8, n)], axis=1)
    _check(_scene(5, 600, 6, 12, 2, points=points), pieces=40)


def test_rows_of_many_pieces(oracle):
    """A path with far more pieces in a row than its 32-bit cells take, beside
    light paths, in a tile of one wavefront and of four."""
    for w in (48, 250):
        sc = _scene(9, w, 8, 20, 2)
        sc.path_cubics[[3, 17]] = 130
        g = np.random.default_rng(10)
        n = int(np.sum(1 + 3 * sc.path_cubics.astype(np.int64)))
        sc.points = g.uniform(0.0, [w, 8.0], size=(n, 2)).astype(np.float32)
        _check(sc, pieces=600)


def test_winding_past_the_cell_range(oracle):
    """200 nested turns in one direction: |A| passes 128 windings, coverage
    stays 1 and the light path over it is unchanged."""
    from footile_amd.diff import DiffRenderer, device_array
    from oracle import pydiff as pd
    w, h, turns = 40, 24, 200
    a = np.linspace(0.0, 2.0 * np.pi * turns, 1 + 3 * 4 * turns)
    spiral = np.stack([20.0 + 15.0 * np.cos(a), 12.0 + 9.0 * np.sin(a)], axis=1)
    light = np.array([[2, 2], [30, 3], [38, 12], [20, 20], [8, 22], [1, 14], [2, 2]], float)
    sc = _scene(3, w, h, 2, 2)
    sc.path_cubics[0] = 4 * turns
    sc.points = np.concatenate([spiral, light]).astype(np.float32)
    _, want = pd.Scene(1, w, h, sc.path_image, sc.path_cubics).forward(sc.points, sc.colours)
    r = DiffRenderer.for_scene(sc)
    canvas = r.new_canvas()
    r.forward(device_array(sc.points), device_array(sc.colours), canvas)
    got = canvas.download(dtype=np.float32).reshape(r.canvas_shape)
    # 1,600 pieces in a row: see the module's rule
    assert np.abs(got - want).max() < 2e-5 * np.sqrt(1600 / 10)


def test_pieces_without_a_number(oracle):
    """A NaN control point: the rows its curve crosses count as covered, the
    others and the paths around it stay as they are, and gradients of the
    other paths stay finite."""
    sc = _scene(4, 70, 12, 3, 2)
    sc.points[7:14, 1] = [1.5, 2.5, 4.0, 5.5, 4.5, 3.0, 1.5]  # path 1 between rows 1 and 5
    clean = sc.points.copy()
    sc.points[9, 0] = np.nan
    target = np.full((1, 12, 70, 4), 0.25, np.float32)
    _, got, gp, gc = _step(sc, target)
    sc.points = clean
    _, want, _, _ = _step(sc, target)
    assert np.isfinite(got).all() and np.isfinite(gp[:7]).all() and np.isfinite(gp[14:]).all()
    assert np.array_equal(got[0, 6:], want[0, 6:]) and np.array_equal(got[0, 0], want[0, 0])
    col = sc.colours
    assert np.all(got[0, 3, :, 3] >= col[1, 3] - 1e-6)  # row 3 lies in the broken curve
