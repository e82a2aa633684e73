"""bk_field_stats_noalloc calls that overlap on one GPU, against its contract,
spoil no later call: each one in order gives bk_field_stats' results again."""
import ctypes as C

import numpy as np
import pytest

from bricklib_amd._lib import check, load

pytestmark = pytest.mark.gpu


def _noalloc(g, f, out, stream):
    check(load().bk_field_stats_noalloc(
        f.dtype, C.c_void_p(f.ptr), C.c_size_t(f.step), C.c_void_p(g.d_interior.ptr),
        C.c_uint32(g.interior.size), C.c_size_t(512), C.c_void_p(out.ptr),
        C.c_void_p(stream.handle)))


def test_after_overlapping_calls(gpu):
    bk = gpu
    streams = [bk.Stream() for _ in range(3)]
    sets = []
    for seed, nb in enumerate([(24, 24, 24), (5, 5, 4), (11, 9, 10)]):  # 256, 7 and 62 workgroups
        g = bk.PeriodicGrid(nb, ghost=0)
        f = bk.Brick(g.info, g.field_storage(0), 0)
        g.fill_uniform(f, seed)
        sets.append((g, f, bk.DeviceBuffer(24)))
    bk.device_sync()
    for _ in range(20):
        for (g, f, out), s in zip(sets, streams):
            _noalloc(g, f, out, s)
    bk.device_sync()
    for _ in range(2):
        for g, f, out in sets:
            out.zero()
            bk.device_sync()
            _noalloc(g, f, out, streams[0])
            bk.device_sync()
            assert np.array_equal(out.download(np.float64), g.stats(f))
