"""Requests without a plan whose lists hold ids beyond their own lengths: where
such a request shares bricks with another one, a captured run keeps the order
of ticks, and both leave what an eager run does."""
import ctypes as C

import numpy as np
import pytest

from bricklib_amd import BK_F32, BK_F64, DeviceBuffer
from bricklib_amd.batch import Arena, Batch, Request, ShapeCache
from bricklib_amd.stencils import Stencil

pytestmark = pytest.mark.gpu

BYTES = 512 * 8
# groups of their own, so that a run would go side by side
MORE = [((6, 5, 4), "13pt", BK_F32, 6), ((3, 2, 2), "13pt", BK_F64, 6), ((4, 2, 3), "25pt", BK_F32, 6),
        ((5, 3, 1), "cond", BK_F64, 6), ((7, 2, 2), "cond", BK_F32, 6)]


class At:
    """A field inside another allocation."""

    def __init__(self, ptr):
        self.ptr = ptr

    def free(self):
        pass


def _request(shapes, rid, nb, name, dt, steps, f0=None, arena=None):
    r = Request(rid=rid, nb=nb, stencil=Stencil.make(name, seed=rid), dtype=dt, steps=steps, seed=rid)
    r.allocate(shapes, arena=arena)
    if f0 is not None:
        r.f0 = f0
    r._rec = bytes(r.req_struct(0))
    return r


@pytest.mark.parametrize("memory", ["allocation", "arena"])
def test_upper_part_of_a_grid(gpu, memory):
    """One sweep over the last quarter of a grid's bricks, which another request
    sweeps as a grid of its own and overwrites in its second tick."""
    big, small = (32, 32, 16), (16, 16, 16)
    first = 32 * 32 * 12
    x = np.random.default_rng(3).uniform(-1, 1, 32 * 32 * 16 * 512)
    ids = np.arange(first, 32 * 32 * 16, dtype=np.uint32)
    got = []
    for use_graph in (False, True):
        shapes, arena = ShapeCache(), Arena(slab_bytes=1 << 29)
        block = arena.alloc(x.nbytes) if memory == "arena" else DeviceBuffer(x.nbytes)
        whole = DeviceBuffer.from_array(x)
        gpu._lib.check(gpu.load().bk_memcpy_d2d(C.c_void_p(block.ptr), C.c_void_p(whole.ptr),
                                                C.c_size_t(x.nbytes), None))
        lower = _request(shapes, 0, big, "25pt", BK_F64, 1, At(block.ptr))
        upper = _request(shapes, 1, small, "7pt", BK_F64, 6, At(block.ptr + first * BYTES))
        d_ids = DeviceBuffer.from_array(ids)
        rec = lower.req_struct(0)
        rec.d_list, rec.nlist = d_ids.ptr, ids.size
        lower._rec = bytes(rec)
        more = [_request(shapes, 2 + q, *m, arena=arena) for q, m in enumerate(MORE)]
        reqs = [lower, upper] + more
        gpu.device_sync()
        batch = Batch(max_reqs=8)
        batch.run(reqs, 6, use_graph=use_graph)
        gpu.device_sync()
        out = [np.empty(x.size) for _ in range(2)]
        for o, p in zip(out, (lower.f1.ptr, block.ptr)):
            gpu._lib.check(gpu.load().bk_memcpy_d2h(o.ctypes.data_as(C.c_void_p), C.c_void_p(p),
                                                    C.c_size_t(o.nbytes), None))
        got.append([out[0].reshape(-1, 512)[first:].tobytes(), out[1].tobytes(),
                    upper.result_host().tobytes()]
                   + [r.result_host().tobytes() for r in more])
    assert got[0] == got[1]
