"""Status and point counts that kernels write to host memory themselves: batches
around the largest path count that does (16), one format and two, and errors
between good runs.  Everything is bytes or whole numbers: equal."""
import numpy as np
import pytest

from footile_amd.path import CLOSE, CUBIC, LINE, MOVE, ops_array
from footile_amd.pixel import MATTE8, RGBA8P

pytestmark = pytest.mark.gpu

NAN = float("nan")


@pytest.fixture(scope="module")
def ft():
    import footile_amd
    return footile_amd

BAD = [(MOVE, (10.0, 20.0)), (CUBIC, (NAN, 24.0, 16.0, 28.0, 19.0, 32.0)), (CLOSE, ())]


def _figure(k, n=1):
    ops = []
    for j in range(n):
        ops += [(MOVE, (4.0 + k, 3.0)), (CUBIC, (40.0, 2.0 + j, 60.0, 30.0 + k, 30.0, 50.0)), (LINE, (2.0, 40.0 - j)),
                (CLOSE, ())]
    return ops


@pytest.mark.parametrize("two_formats", [False, True])
@pytest.mark.parametrize("n", [1, 2, 16, 17])
def test_counts_and_errors_of_batches(ft, oracle, n, two_formats):
    from footile_amd.plotter import Batch, DeviceBuffer, FillDesc
    figs = [ops_array(_figure(k, 1 + k % 3)) for k in range(n)]
    begin = np.concatenate([[0], np.cumsum([len(f) for f in figs])])
    fmt = [RGBA8P if two_formats and k % 2 else MATTE8 for k in range(n)]
    bufs = [DeviceBuffer(64 * 64 * (4 if f == RGBA8P else 1)) for f in fmt]

    def descs():
        return [FillDesc(int(begin[k]), len(figs[k]), bufs[k].ptr, 64, 64, 64 * (4 if fmt[k] == RGBA8P else 1), fmt[k],
                         fresh=True) for k in range(n)]
    want = []
    for k in range(n):
        o = oracle.Plotter(64, 64, fmt[k])
        assert o.fill(0, figs[k]) == 0
        want.append((o.pixels(), o.last_counts()))
    batch = Batch(np.concatenate(figs), descs())
    for launches in (0, 1, 3):  # run, and eager launches before one sync
        for b in bufs:
            b.zero()
        if launches:
            for _ in range(launches):
                batch.launch()
            batch.sync()
        else:
            batch.run()
        offered, stored, _ = batch.counts()
        for k in range(n):
            assert np.array_equal(bufs[k].download(), want[k][0]), k
            assert (offered[k], stored[k]) == want[k][1], k
    # a path that cannot be flattened fails the batch, each time it runs
    bad = np.concatenate(figs)
    bad[begin[n - 1]:begin[n - 1] + 3] = ops_array(BAD)
    failing = Batch(bad, descs())
    for _ in range(2):
        with pytest.raises(ft.FootileError) as e:
            failing.run()
        assert e.value.code == 4
    failing.launch()
    failing.launch()
    with pytest.raises(ft.FootileError) as e:
        failing.sync()
    assert e.value.code == 4


@pytest.mark.parametrize("parts", [1, 120])  # a small figure; the full pipeline (480 ops)
def test_plotter_after_an_error(ft, oracle, parts):
    good = ops_array(_figure(1, parts))
    bad = np.concatenate([good, ops_array(BAD)])
    g, o = ft.Plotter(ft.Raster.with_clear(64, 64, MATTE8)), oracle.Plotter(64, 64, MATTE8)
    for _ in range(2):
        g.fill(0, good)
        assert o.fill(0, good) == 0
        assert g.last_counts() == o.last_counts()
        with pytest.raises(ft.FootileError) as e:
            g.fill(0, bad)
        assert e.value.code == 4
        g.stroke(good)
        assert o.stroke(good) == 0
        assert np.array_equal(g.raster().as_u8_slice(), o.pixels())


def test_diff_runs_after_a_failed_one(oracle):
    """Runs of one handle leave its device state as the next needs it, also
    after a run whose pairs outgrew their list (every edge as tall as the
    image) and was taken again.  The same inputs give the same bytes."""
    from footile_amd.diff import DiffRenderer, device_array
    from footile_amd.plotter import DeviceBuffer
    w, h, paths = 64, 600, 8
    g = np.random.default_rng(5)
    r = DiffRenderer(1, w, h, np.zeros(paths, np.uint32), np.full(paths, 4, np.uint32))
    short = g.uniform(0.0, [w, 40.0], (r.n_points, 2)).astype(np.float32)
    tall = short.copy()
    tall[:, 1] = np.where(np.arange(r.n_points) % 2, -6000.0, 6600.0)
    col = device_array(g.uniform(0.1, 0.9, (paths, 4)))
    cot = device_array(g.normal(size=(1, h, w, 4)))

    def grads(pts):
        gp, gc = DeviceBuffer(8 * r.n_points), DeviceBuffer(16 * paths)
        canvas = r.new_canvas()
        p = device_array(pts)
        r.forward(p, col, canvas)
        r.backward(p, col, cot, gp, gc)
        return canvas.download(), gp.download(dtype=np.float32), gc.download(dtype=np.float32)
    first = grads(short)
    grads(tall)
    again = grads(short)
    assert np.array_equal(first[0], again[0])
    for a, b in zip(first[1:], again[1:]):  # float atomics: any order
        assert np.all(np.isfinite(b)) and np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(a)
