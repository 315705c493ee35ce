"""Strokes past the small figures' limits against the oracle, byte for byte:
the outline in one pass at the edges of its blocks, its general form, joins
whose arcs pass the kept points (10) and the kept levels (32 points), several
sub-strokes with and without closes, and more points than a stroke stores."""
import numpy as np
import pytest

from footile_amd.path import CLOSE, CUBIC, LINE, MOVE, OP_DTYPE, PEN_WIDTH
from footile_amd.pixel import MATTE8

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ft():
    import footile_amd
    return footile_amd


def _route(g, n, w, h, step):
    """n points, every turn between 0.2 and 1.2 rad, kept inside."""
    a = np.cumsum(g.uniform(0.2, 1.2, n) * np.where(g.random(n) < 0.7, 1, -1))
    p = np.cumsum(step * np.stack([np.cos(a), np.sin(a)], 1), 0) + (w / 2, h / 2)
    return np.stack([np.abs((p[:, 0] + w) % (2 * w) - w), np.abs((p[:, 1] + h) % (2 * h) - h)], 1)


def _ops(g, n, w, h, step, width, subs=1, curves=0.0, closes=1):
    rows = [(PEN_WIDTH, [width])]
    for k in range(subs):
        pts = _route(g, n // subs + 1, w, h, step)
        rows.append((MOVE, pts[0]))
        for q in pts[1:]:
            if g.random() < curves:
                rows.append((CUBIC, np.concatenate([q + g.normal(0, step, 2), q + g.normal(0, step, 2), q])))
            else:
                rows.append((LINE, q))
        if k % 3 == 1:
            rows.append((PEN_WIDTH, [width * (1 + 0.2 * (k % 4))]))
        rows += [(CLOSE, [])] * (closes if k % 2 == 0 else 0)
    ops = np.zeros(len(rows), OP_DTYPE)
    for i, (t, v) in enumerate(rows):
        ops["tag"][i] = t
        ops["v"][i, :len(v)] = v
    return ops


def _check(ft, oracle, ops, w, h, join, tol=0.3):
    g, o = ft.Plotter(ft.Raster.with_clear(w, h, MATTE8)), oracle.Plotter(w, h, MATTE8)
    g.set_join({0: ft.JoinStyle.Miter(4.0), 1: ft.JoinStyle.Bevel, 2: ft.JoinStyle.Round}[join])
    o.set_join(join, 4.0)
    g.set_tolerance(tol)
    o.set_tolerance(tol)
    for _ in range(2):
        rc = o.stroke(ops)
        if rc:
            with pytest.raises(ft.FootileError) as e:
                g.stroke(ops)
            assert e.value.code == rc
        else:
            g.stroke(ops)
        assert g.last_counts() == o.last_counts() or rc
        assert np.array_equal(g.raster().as_u8_slice(), o.pixels())


@pytest.mark.parametrize("join", [0, 1, 2])
@pytest.mark.parametrize("n", [300, 382, 383, 384, 1023, 3000, 4200, 9000])
def test_lengths(ft, oracle, n, join):
    """Items 2 (n + 2) + 1 around whole blocks of 256; from 4,032 ops on the
    general form."""
    ops = _ops(np.random.default_rng(n), n, 400, 300, 9.0, 3.0)
    _check(ft, oracle, ops, 400, 300, join)


@pytest.mark.parametrize("width,tol", [(3.0, 0.3), (40.0, 0.3), (90.0, 0.02), (200.0, 0.01)])
def test_long_arcs(ft, oracle, width, tol):
    ops = _ops(np.random.default_rng(7), 300, 400, 300, 60.0, width)
    _check(ft, oracle, ops, 400, 300, 2, tol)


@pytest.mark.parametrize("subs,curves,closes", [(2, 0.0, 1), (7, 0.3, 2), (60, 0.2, 1), (60, 0.0, 0), (300, 0.1, 2)])
@pytest.mark.parametrize("join", [0, 2])
def test_sub_strokes(ft, oracle, subs, curves, closes, join):
    ops = _ops(np.random.default_rng(subs), 900, 500, 400, 7.0, 2.5, subs, curves, closes)
    _check(ft, oracle, ops, 500, 400, join)


@pytest.mark.parametrize("last_close", [True, False])
@pytest.mark.parametrize("n,subs", [(65534, 1), (65600, 1), (66000, 9), (70000, 300)])
def test_more_points_than_are_stored(ft, oracle, n, subs, last_close):
    """Around the 65,535 stored points, the events ending in a close or not:
    the last stored sub-stroke takes the last close of all."""
    ops = _ops(np.random.default_rng(n), n, 300, 200, 2.0, 1.0, subs)
    if ops["tag"][-1] == CLOSE and not last_close:
        ops = ops[:-1]
    elif ops["tag"][-1] != CLOSE and last_close:
        ops = np.concatenate([ops, ops[:1]])
        ops["tag"][-1] = CLOSE
    _check(ft, oracle, ops, 300, 200, 1)
