"""The raster geometry that an untuned batch takes from its sizes against a set
one: the same bytes and counts, at the sizes where the rules change (batch
cells around 4 Mi, heights around 1,024, widths whose two rows end at 3,072
and 6,144 cells), and batches launched before any run has grown a list."""
import numpy as np
import pytest

from footile_amd.path import CLOSE, CUBIC, LINE, MOVE, OP_DTYPE
from footile_amd.pixel import BPP, GRAYA8P, MATTE8, RGBA8P

pytestmark = pytest.mark.gpu


def _ops(seed, w, h, n):
    g = np.random.default_rng(seed)
    ops = np.zeros(n + 2, OP_DTYPE)
    ops["tag"][0], ops["tag"][-1] = MOVE, CLOSE
    ops["tag"][1:-1] = np.where(g.random(n) < 0.4, CUBIC, LINE)
    ops["v"] = (g.random((n + 2, 3, 2)) * (w + 8, h + 8) - 4).reshape(-1, 6).astype(np.float32)
    return ops


@pytest.mark.parametrize("w,h,tiles,fmt,fresh", [
    (31, 7, 1, MATTE8, True), (130, 1024, 1, GRAYA8P, False), (130, 1025, 1, GRAYA8P, False),
    (2032, 2059, 1, MATTE8, False), (2032, 2061, 1, MATTE8, False),  # 2,036 cells a row: around 4 Mi
    (1516, 2900, 1, RGBA8P, False), (1533, 2900, 1, RGBA8P, False),  # two rows: 3,048 and 3,080 cells
    (3052, 1400, 1, RGBA8P, True), (3069, 1400, 1, RGBA8P, False),   # 6,136 and 6,168
    (61, 67, 900, MATTE8, True), (61, 67, 1100, MATTE8, True)])
def test_untuned_geometry_equals_a_set_one(w, h, tiles, fmt, fresh):
    from footile_amd.plotter import Batch, DeviceBuffer, FillDesc
    per = _ops(w + h, w, h, 40)
    ops = np.concatenate([per] * tiles)
    size = w * h * BPP[fmt]
    init = np.random.default_rng(1).integers(0, 256, size * tiles).astype(np.uint8)
    got = []
    for tuned in (False, True):
        buf = DeviceBuffer(size * tiles)
        buf.upload(init)
        batch = Batch(ops, [FillDesc(t * len(per), len(per), buf.ptr + t * size, w, h, w * BPP[fmt], fmt, rule=t & 1,
                                     clr=(90, 60, 30, 120), fresh=fresh) for t in range(tiles)])
        if tuned:
            assert batch.tuning() == (16, 4096, True, 0)
            batch.set_tuning(16, 4096)
        batch.launch()  # (no run before it: the first lists are large enough)
        batch.sync()
        offered, stored, edges = batch.counts()
        got.append((buf.download(), offered, stored, edges))
    for a, b in zip(*got):
        assert np.array_equal(a, b)
