"""Scenes of many small figures: a row's rounds hold only the paths that have
pieces in it.  Against the FP64 oracle with test_gpu_diff_cells' bounds, at
the sizes where the rounds (16 paths) and the staging (256 paths) can go
wrong, and against the cost of the same figures without the others."""
import time

import numpy as np
import pytest

from tests.test_gpu_diff_cells import _check, _scene

pytestmark = pytest.mark.gpu


def _local(h, size, rows=None):
    """Points of figures of about `size` pixels; with rows, figure k lies around row rows(k)."""
    def points(g, n):
        per = 1 + 3 * 2  # two cubics a path
        k = n // per
        c = g.uniform(size, [60.0, h - size], (k, 1, 2))
        if rows is not None:
            c[:, 0, 1] = [rows(i) for i in range(k)]
        return (c + g.uniform(-size / 2, size / 2, (k, per, 2))).reshape(-1, 2)
    return points


@pytest.mark.parametrize("paths,images", [
    (40, 1), (63, 1), (64, 2), (65, 1), (127, 1), (129, 1), (193, 1),  # staged 64 at a time
    (255, 1), (257, 2), (530, 1)])
def test_small_figures(oracle, paths, images):
    _check(_scene(paths, 64, 48, paths, 2, images, points=_local(48, 5.0)))


@pytest.mark.parametrize("live", [1, 15, 16, 17, 32, 33])
@pytest.mark.parametrize("stride", [1, 7, 9])  # every stride-th path crosses row 6, the others lie below: 1 to 2 stagings
def test_rounds_of_a_row(oracle, live, stride):
    """`live` paths of all in row 6, spread over the others."""
    def rows(k):
        return 6.5 if k % stride == 0 and k // stride < live else 24.5
    _check(_scene(live + stride, 70, 32, max(live * stride, 20) + 3, 2, points=_local(32, 4.0, rows)))


def test_heavy_and_light_paths_among_empty_ones(oracle):
    """Paths of many pieces in some rows (64-bit cells) between paths without any."""
    sc = _scene(31, 48, 40, 300, 2, points=_local(40, 6.0))
    cubics = sc.path_cubics.copy()
    cubics[[5, 140, 299]] = 130
    g = np.random.default_rng(32)
    n = 1 + 3 * cubics.astype(np.int64)
    c = np.repeat(g.uniform(4.0, [44.0, 36.0], (300, 2)), n, axis=0)
    sc.path_cubics = cubics
    sc.points = (c + g.uniform(-3.0, 3.0, (int(n.sum()), 2))).astype(np.float32)
    _check(sc, pieces=600)


def _median_forward(sc):
    from footile_amd.diff import DiffRenderer, device_array
    r = DiffRenderer.for_scene(sc)
    p, c, canvas = device_array(sc.points), device_array(sc.colours), r.new_canvas()
    times = []
    for k in range(40):
        a = time.perf_counter()
        r.forward(p, c, canvas)
        if k >= 10:
            times.append(time.perf_counter() - a)
    return float(np.median(times))


def test_paths_without_pieces_cost_little():
    """16 figures across a 512x512 image, alone and before 1,008 paths outside
    it: a row's work is that of its own paths.  (Walking all of them took 6
    times as long; staging their counts takes a tenth.)"""
    few = _scene(41, 512, 512, 16, 2)
    more = _scene(41, 512, 512, 1024, 2, points=lambda g, n: g.uniform(600.0, 700.0, (n, 2)))
    more.points[:len(few.points)] = few.points
    assert _median_forward(more) < 2.5 * _median_forward(few)


@pytest.mark.parametrize("h", [8191, 8192, 8193, 16384, 16385, 20000])
def test_tall_images(oracle, h):
    """The one-launch geometry takes 8,192 rows of a path at a time: for figures
    in and across the windows the same canvas bytes as the general form (a path
    of 2,081 edges outside the image sends all paths there), and the same
    gradients but for the order of their float32 sums (at most some 1,000 terms
    of either sign a vertex: 1e-5).  (FP64 says little here: y near 8,192 is
    rounded at 5e-4.)"""
    import dataclasses

    from tests.test_gpu_diff_cells import _rel, _step
    g = np.random.default_rng(h)
    sc = _scene(h, 5, h, 6, 3)
    tall = sc.points.reshape(6, -1, 2)
    tall[2:] = g.uniform(-2.0, 7.0, tall[2:].shape)  # the last four small, around the windows' borders
    tall[2:, :, 1] += np.array([8192.0, 8190.0, min(16384, h) - 3.0, h - 4.0])[:, None]
    far = g.uniform(200.0, 300.0, size=(1 + 3 * 130, 2)).astype(np.float32)
    more = dataclasses.replace(sc, path_image=np.append(sc.path_image, 0).astype(np.uint32),
                               path_cubics=np.append(sc.path_cubics, 130).astype(np.uint32),
                               points=np.concatenate([sc.points, far]),
                               colours=np.concatenate([sc.colours, sc.colours[:1]]))
    target = g.uniform(0, 1, size=(1, h, 5, 4)).astype(np.float32)
    loss, canvas, gp, gc = _step(sc, target)
    want_loss, want, want_gp, want_gc = _step(more, target)
    assert loss == want_loss and np.array_equal(canvas, want) and np.abs(gp).max() > 0.0
    assert _rel(gp, want_gp[:len(gp)]) < 1e-5 and _rel(gc, want_gc[:len(gc)]) < 1e-5
