"""Small figures whose closes come after many repeats of one point: the walk
back over the repeats is bounded, past it the kept points come from a running
maximum in the same kernel.  Bytes and counts against the oracle, and the
cost of a call against the same figure without the repeats."""
import time

import numpy as np
import pytest

from footile_amd.path import CLOSE, LINE, MOVE, OP_DTYPE, PEN_WIDTH

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ft():
    import footile_amd
    return footile_amd


def _ops(g, runs, repeats, first=False, side=96):
    """`runs` outlines of 5 points, the last (with `first` the first) repeated
    `repeats` times before each close."""
    rows = [(PEN_WIDTH, [3.0])]
    for _ in range(runs):
        p = g.uniform(4, side - 4, (5, 2))
        rows += [(MOVE, p[0])] + [(LINE, q) for q in p[1:]]
        rows += [(LINE, p[0 if first else 4])] * repeats + [(CLOSE, [])]
    ops = np.zeros(len(rows), OP_DTYPE)
    for i, (t, v) in enumerate(rows):
        ops["tag"][i] = t
        ops["v"][i, :len(v)] = v
    return ops


@pytest.mark.parametrize("stroke", [False, True])
@pytest.mark.parametrize("first", [False, True])  # a last point like the first is popped
# either side of the walk's 32 points, several runs, and the 256 ops of a small figure
@pytest.mark.parametrize("runs,repeats", [(1, 30), (1, 31), (1, 32), (1, 33), (3, 31), (3, 40), (6, 33), (1, 248)])
def test_repeats_before_a_close(ft, oracle, runs, repeats, first, stroke):
    ops = _ops(np.random.default_rng(runs + repeats), runs, repeats, first)
    assert len(ops) <= 256
    g, o = ft.Plotter(ft.Raster.with_clear(96, 96)), oracle.Plotter(96, 96)
    for _ in range(2):
        if stroke:
            g.stroke(ops)
            assert o.stroke(ops) == 0
        else:
            g.fill(ft.FillRule.NonZero, ops)
            assert o.fill(0, ops) == 0
        assert g.last_counts() == o.last_counts()
    assert np.array_equal(np.asarray(g.raster().as_u8_slice()).reshape(-1), np.asarray(o.pixels()).reshape(-1))


def test_repeats_stay_in_the_small_kernels(ft):
    """(Two launches of the full pipeline after the small one: 4 times as long.)"""
    def median(repeats):
        p = ft.Plotter(ft.Raster.with_clear(96, 96))
        ops = _ops(np.random.default_rng(1), 1, repeats)
        t = []
        for k in range(120):
            a = time.perf_counter()
            p.fill(ft.FillRule.NonZero, ops)
            if k >= 20:
                t.append(time.perf_counter() - a)
        return float(np.median(t))
    assert median(40) < 2.0 * median(0)
