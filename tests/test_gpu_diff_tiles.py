"""The differentiable fill either side of the widths whose tiles are 256 pixels
(193 and up, a kernel of its own), and the loss from buffers aligned to 16
bytes and to 4, against the FP64 oracle with test_gpu_diff_cells' bounds."""
import ctypes

import numpy as np
import pytest

from tests.test_gpu_diff_cells import _check, _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,paths,cubics", [(192, 6, 19, 2), (193, 6, 19, 2), (256, 5, 33, 3), (385, 4, 17, 2)])
def test_tile_widths(oracle, w, h, paths, cubics):
    _check(_scene(w + paths, w, h, paths, cubics))


@pytest.mark.parametrize("w,h", [(1, 1), (3, 5), (256, 256), (257, 300)])  # up to more than one round of the grid
@pytest.mark.parametrize("offset", [0, 4, 8])
def test_loss_of_aligned_and_other_buffers(w, h, offset):
    """The mean of squares in FP64 over FP32 differences, to 1e-12; the
    gradient is the FP32 product."""
    from footile_amd._lib import check, lib
    from footile_amd.diff import DiffRenderer
    from footile_amd.plotter import DeviceBuffer
    g = np.random.default_rng(w * h + offset)
    n = 4 * w * h
    r = DiffRenderer(1, w, h, np.zeros(1, np.uint32), np.ones(1, np.uint32))
    c, t = (g.random(n).astype(np.float32) for _ in range(2))
    pad = np.zeros(offset // 4, np.float32)
    bufs = []
    for a in (c, t, np.zeros(n, np.float32)):
        b = DeviceBuffer(4 * n + 16)
        b.upload(np.concatenate([pad, a]))
        bufs.append(b)
    out = ctypes.c_double()
    d = c - t
    for _ in range(2):
        check(lib().ft_diff_loss(ctypes.c_void_p(r._h), *[ctypes.c_void_p(b.ptr + offset) for b in bufs],
                                 ctypes.byref(out)), "loss")
        want = float((d.astype(np.float64) ** 2).sum()) / n
        assert abs(out.value - want) <= 1e-12 * max(want, 1e-30)
        grad = bufs[2].download(4 * n + offset, np.float32)[offset // 4:]
        assert np.array_equal(grad, np.float32(2.0 / n) * d)
