"""Batches without allocation whose few ops become very many events (long
curves, drawn large): the event kernels' grids against the events' number.
Bytes and counts against the allocating batch, which sizes its grids by the
events of the run before."""
import ctypes

import numpy as np
import pytest

from footile_amd.path import CLOSE, CUBIC, MOVE, OP_DTYPE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("paths,curves,scale", [(1, 1, 1.0e3), (2, 2, 1.0e3), (8, 2, 1.0e4), (64, 4, 1.0e3)])
def test_many_events_of_few_ops(paths, curves, scale):
    from footile_amd._lib import check, lib
    from footile_amd.plotter import Batch, DeviceBuffer, FillDesc, FillDescC
    g = np.random.default_rng(paths)
    side, n = 64, curves + 2
    ops = np.zeros(paths * n, OP_DTYPE)
    ops["tag"] = np.tile([MOVE] + [CUBIC] * curves + [CLOSE], paths)
    ops["v"] = g.random((len(ops), 6)) * side
    out = []
    for noalloc in (True, False):
        dst = DeviceBuffer(side * side * paths)
        dst.zero()
        descs = [FillDesc(k * n, n, dst.ptr + k * side * side, side, side, side,
                          transform=(scale, 0, 0, 0, scale, 0), fresh=True) for k in range(paths)]
        offered, stored = np.zeros(paths, np.uint64), np.zeros(paths, np.uint64)
        if noalloc:
            arr = (FillDescC * paths)(*[d.c for d in descs])
            vp = ctypes.c_void_p
            for _ in range(2):
                check(lib().ft_batch_run_noalloc(ops.ctypes.data_as(vp), len(ops), arr, paths, None,
                                                 offered.ctypes.data_as(vp), stored.ctypes.data_as(vp)), "noalloc")
        else:
            b = Batch(ops, descs)
            b.run()
            offered, stored, _ = b.counts()
        out.append((dst.download(), offered, stored))
    assert int(out[0][1].sum()) > 64 * len(ops)  # (16 are taken for granted)
    for a, b in zip(*out):
        assert np.array_equal(a, b)
