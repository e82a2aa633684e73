"""Python mirror of bricklib's host interface over libbricks.so.

Names follow the reference (CtopCsUtahEdu/bricklib) so code and tests read
like its drivers: ``init_grid`` (bricksetup.h:73-89), ``BrickInfo``
(brick.h:96-127), ``BrickStorage.allocate`` (brick.h:68-75, here resident in
HBM), ``Brick`` (brick.h:353-395, a field view: storage + offset),
``movBrickInfo`` / ``movBrickStorage`` (brick-gpu.h:42-103),
``copyToBrick`` / ``copyFromBrick`` (bricksetup.h:172-221).  Every GPU
operation goes through the C-ABI; nothing here computes on the CPU.
"""
from __future__ import annotations

import ctypes as C
import itertools
import struct
import threading
from dataclasses import dataclass, field

import numpy as np

from . import _lib
from ._lib import (BK_BF16, BK_F32, BK_F64, bk_sweep_desc, check, load, longs)
from .stencils import NCOEFF, Stencil, stencil_id

DTYPE_NP = {BK_F64: np.float64, BK_F32: np.float32, BK_BF16: np.uint16}
DTYPE_SIZE = {BK_F64: 8, BK_F32: 4, BK_BF16: 2}
BRICK_ELEMS = 512  # 8 x 8 x 8


def _vp(x) -> C.c_void_p:
    if x is None:
        return C.c_void_p(None)
    if isinstance(x, int):
        return C.c_void_p(x)
    if isinstance(x, np.ndarray):
        return x.ctypes.data_as(C.c_void_p)
    return C.c_void_p(int(x))


# ---------------------------------------------------------------------------
# device memory, streams, events
# ---------------------------------------------------------------------------
class DeviceBuffer:
    """An HBM allocation owned by Python (freed with the object)."""

    _stamps = itertools.count(1)

    def __init__(self, nbytes: int):
        self.nbytes = int(nbytes)
        p = C.c_void_p()
        check(load().bk_alloc(C.c_size_t(self.nbytes), C.byref(p)))
        self.ptr = p.value or 0
        self.stamp = next(self._stamps)  # of the last upload or clear, among all buffers

    @classmethod
    def from_array(cls, arr: np.ndarray, stream=None) -> "DeviceBuffer":
        arr = np.ascontiguousarray(arr)
        buf = cls(arr.nbytes)
        buf.upload(arr, stream)
        return buf

    def upload(self, arr: np.ndarray, stream=None, offset: int = 0) -> None:
        arr = np.ascontiguousarray(arr)
        if offset + arr.nbytes > self.nbytes:
            raise ValueError("upload past the end of the buffer")
        self.stamp = next(self._stamps)
        check(load().bk_memcpy_h2d(_vp(self.ptr + offset), _vp(arr), C.c_size_t(arr.nbytes),
                                   _vp(stream)))

    def download(self, dtype, count: int | None = None, stream=None, offset: int = 0):
        dtype = np.dtype(dtype)
        if count is None:
            count = (self.nbytes - offset) // dtype.itemsize
        out = np.empty(count, dtype=dtype)
        if offset + out.nbytes > self.nbytes:
            raise ValueError("download past the end of the buffer")
        check(load().bk_memcpy_d2h(_vp(out), _vp(self.ptr + offset), C.c_size_t(out.nbytes),
                                   _vp(stream)))
        return out

    def zero(self, stream=None) -> None:
        self.stamp = next(self._stamps)
        check(load().bk_zero(_vp(self.ptr), C.c_size_t(self.nbytes), _vp(stream)))

    def free(self) -> None:
        if getattr(self, "ptr", 0):
            load().bk_free(_vp(self.ptr))
            self.ptr = 0

    def __del__(self):
        try:
            self.free()
        except Exception:
            pass


class Stream:
    """A non-blocking HIP stream (default priority)."""

    def __init__(self):
        h = C.c_void_p()
        check(load().bk_stream_create(C.byref(h)))
        self.handle = h.value

    def sync(self) -> None:
        check(load().bk_stream_sync(_vp(self.handle)))

    def __int__(self):
        return int(self.handle or 0)

    def __del__(self):
        try:
            if self.handle:
                load().bk_stream_destroy(_vp(self.handle))
                self.handle = None
        except Exception:
            pass


class Event:
    def __init__(self):
        h = C.c_void_p()
        check(load().bk_event_create(C.byref(h)))
        self.handle = h.value

    def record(self, stream=None) -> None:
        check(load().bk_event_record(_vp(self.handle), _vp(stream)))

    def sync(self) -> None:
        check(load().bk_event_sync(_vp(self.handle)))

    def elapsed_ms(self, end: "Event") -> float:
        ms = C.c_float()
        check(load().bk_event_elapsed_ms(_vp(self.handle), _vp(end.handle), C.byref(ms)))
        return float(ms.value)

    def __del__(self):
        try:
            if self.handle:
                load().bk_event_destroy(_vp(self.handle))
                self.handle = None
        except Exception:
            pass


def device_count() -> int:
    n = C.c_int()
    rc = load().bk_device_count(C.byref(n))
    return n.value if rc == 0 else 0


def device_sync() -> None:
    check(load().bk_device_sync())


def _stream_of(stream):
    if stream is None:
        return None
    return int(stream)


# ---------------------------------------------------------------------------
# BrickInfo / init_grid / BrickStorage / Brick
# ---------------------------------------------------------------------------
class BrickInfo:
    """BrickInfo<3>: the adjacency list adj[nbricks][27] (uint32), on the
    host (``adj``) and, after movBrickInfo, in HBM (``dev``)."""

    def __init__(self, adj: np.ndarray):
        self.adj = np.ascontiguousarray(adj, dtype=np.uint32).reshape(-1, 27)
        self.dev: DeviceBuffer | None = None

    @property
    def nbricks(self) -> int:
        return self.adj.shape[0]

    @property
    def dptr(self) -> int:
        if self.dev is None:
            raise RuntimeError("BrickInfo is not on the device; call movBrickInfo first")
        return self.dev.ptr


def init_grid(dims, periodic: bool = False):
    """init_grid<3>(grid_ptr, dims) -> (grid, BrickInfo).  ``dims`` are brick
    counts contiguous-first (i, j, k); ``grid`` has shape (k, j, i)."""
    dims = [int(d) for d in dims]
    n = dims[0] * dims[1] * dims[2]
    grid = np.empty(n, dtype=np.uint32)
    adj = np.empty(n * 27, dtype=np.uint32)
    check(load().bk_init_grid(longs(dims), int(bool(periodic)),
                              grid.ctypes.data_as(_lib.u32p), adj.ctypes.data_as(_lib.u32p)))
    return grid.reshape(dims[2], dims[1], dims[0]), BrickInfo(adj)


def movBrickInfo(info: BrickInfo, stream=None) -> BrickInfo:
    """Copy the adjacency list into HBM (brick-gpu.h:42-55)."""
    info.dev = DeviceBuffer.from_array(info.adj, _stream_of(stream))
    return info


@dataclass
class BrickStorage:
    """Device-resident BrickStorage: ``chunks`` x ``step`` elements."""

    buf: DeviceBuffer
    chunks: int
    step: int
    dtype: int = BK_F64

    @classmethod
    def allocate(cls, chunks: int, step: int, dtype: int = BK_F64) -> "BrickStorage":
        p = C.c_void_p()
        check(load().bk_storage_alloc(int(dtype), C.c_long(int(chunks)), C.c_size_t(int(step)),
                                      C.byref(p)))
        buf = DeviceBuffer.__new__(DeviceBuffer)
        es = DTYPE_SIZE[dtype]
        buf.nbytes = ((int(chunks) * int(step) * es + 2047) // 2048) * 2048
        buf.ptr = p.value or 0
        buf.stamp = next(buf._stamps)
        return cls(buf, int(chunks), int(step), int(dtype))

    @property
    def dat(self) -> int:
        return self.buf.ptr

    def to_host(self, stream=None) -> np.ndarray:
        """movBrickStorage(..., DeviceToHost) (brick-gpu.h:84-103)."""
        n = self.chunks * self.step
        return self.buf.download(DTYPE_NP[self.dtype], n, _stream_of(stream)).reshape(
            self.chunks, self.step)


def movBrickStorage(host: np.ndarray, dtype: int = BK_F64, stream=None) -> BrickStorage:
    """Copy a host storage array (chunks, step) into a new device
    BrickStorage (brick-gpu.h:84-103)."""
    host = np.ascontiguousarray(host, dtype=DTYPE_NP[dtype])
    chunks, step = host.shape
    st = BrickStorage.allocate(chunks, step, dtype)
    st.buf.upload(host.reshape(-1), _stream_of(stream))
    return st


@dataclass
class Brick:
    """Brick<Dim<8,8,8>,Dim<8,8>>(bInfo, bStorage, offset): one field of a
    storage, ``offset`` elements into each chunk (brick.h:390-394)."""

    info: BrickInfo
    storage: BrickStorage
    offset: int = 0

    @property
    def ptr(self) -> int:
        return self.storage.dat + self.offset * DTYPE_SIZE[self.storage.dtype]

    @property
    def step(self) -> int:
        return self.storage.step

    @property
    def dtype(self) -> int:
        return self.storage.dtype

    def bricks_host(self, stream=None) -> np.ndarray:
        """(chunks, 512) view of this field's bricks, copied to the host."""
        return self.storage.to_host(stream)[:, self.offset:self.offset + BRICK_ELEMS]


def copyToBrick(dimlist, padding, ghost, arr: DeviceBuffer, grid: DeviceBuffer, brick: Brick,
                stream=None) -> None:
    """copyToBrick<3> on the device (bricksetup.h:172-200)."""
    check(load().bk_copy_to_brick(brick.dtype, longs(dimlist), longs(padding), longs(ghost),
                                  _vp(arr.ptr), _vp(grid.ptr), _vp(brick.ptr),
                                  C.c_size_t(brick.step), _vp(_stream_of(stream))))


def copyFromBrick(dimlist, padding, ghost, arr: DeviceBuffer, grid: DeviceBuffer, brick: Brick,
                  stream=None) -> None:
    """copyFromBrick<3> on the device (bricksetup.h:213-221)."""
    check(load().bk_copy_from_brick(brick.dtype, longs(dimlist), longs(padding), longs(ghost),
                                    _vp(arr.ptr), _vp(grid.ptr), _vp(brick.ptr),
                                    C.c_size_t(brick.step), _vp(_stream_of(stream))))


# ---------------------------------------------------------------------------
# execution plans
# ---------------------------------------------------------------------------
PLAN_SHAPES = {"column": _lib.BK_PLAN_COLUMN, "quad": _lib.BK_PLAN_QUAD}


def plan_host(info: BrickInfo, blist: np.ndarray, shape: str, kcol: int) -> dict:
    """The plan's arrays built on the host (bk_plan_build_host)."""
    blist = np.ascontiguousarray(blist, np.uint32)
    lib = load()
    nu, nc = C.c_uint32(), C.c_uint32()
    args = (info.adj.ctypes.data_as(_lib.u32p), info.nbricks, blist.ctypes.data_as(_lib.u32p),
            blist.size, PLAN_SHAPES[shape], int(kcol))
    check(lib.bk_plan_build_host(*args, None, None, None, None, C.byref(nu), C.byref(nc)))
    anchor = np.zeros(nu.value, np.uint32)
    ln = np.zeros(nu.value, np.uint32)
    mask = np.zeros(nu.value * kcol, np.uint32)
    flat = np.zeros(nc.value, np.uint32)
    check(lib.bk_plan_build_host(*args, anchor.ctypes.data_as(_lib.u32p),
                                 ln.ctypes.data_as(_lib.u32p), mask.ctypes.data_as(_lib.u32p),
                                 flat.ctypes.data_as(_lib.u32p), C.byref(nu), C.byref(nc)))
    return {"anchor": anchor, "len": ln, "mask": mask.reshape(-1, kcol), "flat": flat}


class Plan:
    """An execution plan in HBM (bk_plan_create): the listed bricks grouped
    into k-columns ("column") or 2x2 column quads ("quad") of up to kcol
    levels."""

    def __init__(self, info: BrickInfo, blist: np.ndarray, shape: str = "column",
                 kcol: int = 16):
        blist = np.ascontiguousarray(blist, np.uint32)
        h = C.c_void_p()
        check(load().bk_plan_create(info.adj.ctypes.data_as(_lib.u32p), info.nbricks,
                                    blist.ctypes.data_as(_lib.u32p), blist.size,
                                    PLAN_SHAPES[shape], int(kcol), C.byref(h)))
        self.handle = h.value
        self.shape = shape
        self.kcol = int(kcol)
        self.boxed = False  # set_box ran
        self.lock = threading.Lock()  # one declaration at a time
        self.tables: set = set()  # device tables that sequences came with (_declare_box)
        nu, nc = C.c_uint32(), C.c_uint32()
        check(load().bk_plan_query(_vp(self.handle), C.byref(nu), None, None, C.byref(nc)))
        self.nunits = nu.value
        self.ncovered = nc.value

    def set_box(self, info: BrickInfo, nb, ids: np.ndarray, pairs: np.ndarray,
                stream=None) -> None:
        """Declare the plan's bricks a periodic box (bk_plan_set_box): ``ids``
        its nb[0] x nb[1] x nb[2] bricks in grid order (k slowest), ``pairs``
        the (dst, src) ghost pairs, flat.  Sequences of sweeps whose device
        tables are bound to the box (bind_box; ``sweeps`` does it) then read
        the images themselves and may take several sweeps per pass."""
        ids = np.ascontiguousarray(ids, np.uint32)
        pairs = np.ascontiguousarray(pairs, np.uint32)
        check(load().bk_plan_set_box(_vp(self.handle), info.adj.ctypes.data_as(_lib.u32p),
                                     longs(nb), ids.ctypes.data_as(_lib.u32p),
                                     pairs.ctypes.data_as(_lib.u32p), pairs.size // 2,
                                     _stream_of(stream)))
        self.boxed = True

    def bind_box(self, d_adj: int, d_pairs=None, npairs: int = 0, d_img_off=None, d_img=None,
                 stream=None) -> None:
        """Check these device tables against the declared box and let
        sequences that come with them use it (bk_plan_bind_box), until one of
        them is written through the library or freed."""
        check(load().bk_plan_bind_box(_vp(self.handle), _vp(d_adj), _vp(d_pairs), int(npairs),
                                      _vp(d_img_off), _vp(d_img), _stream_of(stream)))

    def unbind_box(self) -> None:
        """End every binding of the plan (bk_plan_unbind_box): sequences
        refresh with their own tables before every sweep again."""
        check(load().bk_plan_unbind_box(_vp(self.handle)))

    def __del__(self):
        try:
            if getattr(self, "handle", None):
                load().bk_plan_destroy(_vp(self.handle))
                self.handle = None
        except Exception:
            pass


# ---------------------------------------------------------------------------
# periodic brick grid with one ghost layer
# ---------------------------------------------------------------------------
# Default schedule per (stencil, dtype): (plan shape, levels), None = one
# brick per wave.  From warmed timings of every schedule at 512^3 on one
# MI355X (ms per step with the refresh fused into the sweep / with a separate
# refresh kernel / kernel alone):
#   stars and cond: 2x2 column quads, whose four waves share one LDS tile
#   of the block, so each wave fetches two of its four in-plane faces --
#   FP64 7-point quad1 0.420 / 0.441 / 0.396 against one brick per wave
#   0.466 / 0.478 / 0.436; 13-point quad1 0.440 / 0.457 against 0.514 /
#   0.516; cond quad1 0.422 / 0.441 against 0.466 / 0.481; 25-point quad2
#   0.505 / 0.510 against k-marching columns of 8 0.598 (separate); FP32
#   7-point quad2 0.235 / 0.241 against 0.257 / 0.269, 13-point and cond
#   quad2, 25-point quad4 0.287 / 0.289 against 0.390 / 0.366.  One level
#   (no k-march) wins for FP64 radius 1-2: four times the units of quad4,
#   and the k-faces a march would save are a quarter of what the shared
#   tile saves.  BF16 (the row-form kernels: 16-byte rows): 7/13-point and
#   cond in 2x2 blocks of 4 levels (kernel alone / with a separate refresh:
#   7-point 0.117 / 0.129 against one brick per wave 0.131 / 0.143 and one
#   level 0.144 / 0.158; 13-point 0.131 / 0.144 against 0.139 / 0.151; cond
#   0.131 / 0.145 against 0.146 / 0.158), the 25-point in blocks of 8
#   levels (0.177-0.180 / 0.183-0.187 against one brick per wave 0.184-0.186
#   / 0.186-0.187).
#   cube: by size (auto_plan); at 512^3 quads of 6 levels (kernel: FP64 0.613 ms against 0.628
#   with 4 levels, 0.646 with 2 and 0.635 with 8; FP32 0.514 against 0.520
#   / 0.521 / 0.540).
DEFAULT_PLANS = {
    (0, BK_F64): ("quad", 1), (1, BK_F64): ("quad", 1), (4, BK_F64): ("quad", 1),
    (2, BK_F64): ("quad", 2),
    (0, BK_F32): ("quad", 2), (1, BK_F32): ("quad", 2), (4, BK_F32): ("quad", 2),
    (2, BK_F32): ("quad", 4),
    (0, BK_BF16): ("quad", 4), (1, BK_BF16): ("quad", 4), (4, BK_BF16): ("quad", 4),
    (2, BK_BF16): ("quad", 8),
    (3, BK_F64): ("quad", 6), (3, BK_F32): ("quad", 6), (3, BK_BF16): ("quad", 6),
}
# Stencils whose sequences may take several sweeps per pass (bk_plan_set_box).
STEP_STENCILS = (_lib.BK_STAR7, _lib.BK_COND7, _lib.BK_STAR13)
# lane_shift of the quad star kernels per (stencil, dtype); absent = 0 (the
# i-taps from the LDS tile).
DEFAULT_LANE_SHIFT: dict = {}


def star_levels(kind: int, dtype: int, n: int, most: int) -> int:
    """Levels a star's quad unit marches on a grid of n bricks.  More levels
    read fewer k-halos, fewer units leave a small device idle.  us a sweep,
    fewer levels / DEFAULT_PLANS': 25-point BF16 20^3 bricks 9.8 (2) / 18.8,
    45x27x33 35.1 (2) / 39.9, 48^3 82.0 (4) / 81.3, FP32 20^3 12.4 (1) / 13.9,
    32^3 35.6 (1) / 38.9, 48^3 103.9 (2) / 104.7, FP64 20^3 20.6 (1) / 21.4,
    45x27x33 83.2 (1) / 81.9; 13-point BF16 20^3 8.0 (1) / 9.7, 45x27x33 25.7
    (2) / 27.6; 7-point FP32 20^3 10.0 (1) / 10.4, 45x27x33 37.1 (1) / 39.0,
    48^3 91.0 (1) / 92.6, 64^3 203.9 (1) / 200.7."""
    wide = kind == _lib.BK_STAR25
    if dtype == BK_F64:
        few = 1 if n <= 12000 else most
    elif dtype == BK_F32:
        few = (1 if n <= 60000 else 2 if n <= 150000 else most) if wide else (
            1 if n <= 120000 else most)
    elif wide:
        few = 2 if n <= 60000 else 4 if n <= 100000 else most
    else:
        few = 1 if n <= 12000 else 2 if n <= 60000 else most
    return min(few, most)


class PeriodicGrid:
    """n = 8*nb interior cells per axis with periodic boundaries, in one of
    two layouts, all tables in HBM:

    ghost=1 (the reference's): an 8-cell (one-brick) ghost zone -- a
      (nb+2)^3 brick grid numbered by init_grid, its adjacency, the interior
      brick list and the periodic ghost pairs a refresh copies before each
      sweep;
    ghost=0: an nb^3 brick grid whose adjacency wraps (init_grid with
      periodic=True); every brick is interior and nothing needs refreshing.
      A sweep reads the periodic image itself where the ghost layout reads
      its copy, so both give the same values, bit for bit.

    layout: the brick shape and vector fold of the grid's fields
    (BK_LAYOUT_8x8x8, BK_LAYOUT_4x8x16 or BK_LAYOUT_4x8x16_F88); nb counts
    bricks of that shape per axis (i, j, k), so the interior holds
    nb[0]*BI x nb[1]*BJ x nb[2]*BK cells.  Each cell gets the same value in
    every layout."""

    def __init__(self, nb, stream=None, ghost: int = 1, tile=(32, 16), layout: int = 0):
        self.nb = tuple(int(x) for x in nb)
        if ghost not in (0, 1):
            raise ValueError("ghost must be 0 or 1")
        ext = (C.c_int * 3)()
        check(load().bk_layout_extents(int(layout), ext))
        self.brick_layout = int(layout)
        self.extents = tuple(int(x) for x in ext)  # (BK, BJ, BI)
        self.ghost = int(ghost)
        self.padded = tuple(x + 2 * self.ghost for x in self.nb)
        self.grid, self.info = init_grid(self.padded, periodic=not self.ghost)
        movBrickInfo(self.info, stream)
        if self.ghost:
            n = C.c_uint32()
            check(load().bk_interior_list(longs(self.nb), None, C.byref(n)))
            self.interior = np.empty(n.value, dtype=np.uint32)
            check(load().bk_interior_list(longs(self.nb), self.interior.ctypes.data_as(_lib.u32p),
                                          C.byref(n)))
            check(load().bk_ghost_pairs(longs(self.nb), None, C.byref(n)))
            self.pairs = np.empty(2 * n.value, dtype=np.uint32)
            check(load().bk_ghost_pairs(longs(self.nb), self.pairs.ctypes.data_as(_lib.u32p),
                                        C.byref(n)))
        else:
            self.interior = np.ascontiguousarray(self.grid.reshape(-1), dtype=np.uint32)
            self.pairs = np.empty(0, dtype=np.uint32)
        self.d_interior = DeviceBuffer.from_array(self.interior, stream)
        self.d_pairs = DeviceBuffer.from_array(self.pairs, stream) if self.pairs.size else None
        # the order the sweeps visit the interior bricks in: grid order (k
        # slowest) with tile=0, or the (i, j) plane cut into Ti x Tj brick
        # tiles (tile=T: T x T), each swept through all k before the next --
        # neighbours in k are then Ti*Tj list positions apart instead of a
        # whole brick plane (T = 32 measured 4-6% faster for the 7-point star
        # at 512^3 than grid order; for the 2x2 block schedules, whose plans
        # follow this order, 32 x 16 is 0-3% ahead of 32 x 32 and 6-10% ahead
        # of whole planes or 8 x 8; 64 x 8, the same 512 bricks per tile
        # plane, ran the radius-1/2 star kernels 0.5-1.3% faster alone but
        # the fused 7-point step 1.9% slower, and 16 x 16, 16 x 8, 32 x 8 and
        # 64 x 4 were 2-8% slower).  Every brick is computed the same way in
        # any order.
        self.tile = (tuple(int(x) for x in tile) if isinstance(tile, (tuple, list))
                     else ((int(tile), int(tile)) if tile else 0))
        self.sweep_list = self.tiled_order(self.tile) if self.tile else self.interior
        self.d_sweep_list = (DeviceBuffer.from_array(self.sweep_list, stream) if self.tile
                             else self.d_interior)
        self.d_grid = DeviceBuffer.from_array(self.grid.reshape(-1), stream)

        self._plans: dict = {}
        self._tuned: dict = {}

    def tiled_order(self, T) -> np.ndarray:
        """Interior bricks tile by tile (bk_tiled_list): Ti x Tj bricks in
        (i, j) (T an int for square tiles or a pair (Ti, Tj)), all k."""
        Ti, Tj = (int(T[0]), int(T[1])) if isinstance(T, (tuple, list)) else (int(T), int(T))
        if Ti < 1 or Tj < 1:
            raise ValueError("tile sides must be positive")
        n = C.c_uint32()
        check(load().bk_tiled_list(longs(self.nb), self.ghost, Ti, Tj, None, C.byref(n)))
        out = np.empty(n.value, dtype=np.uint32)
        check(load().bk_tiled_list(longs(self.nb), self.ghost, Ti, Tj,
                                   out.ctypes.data_as(_lib.u32p), C.byref(n)))
        return out

    def plan(self, shape: str = "column", kcol: int = 16, every: bool = False) -> Plan:
        """A cached plan over the interior bricks in sweep order (every=True:
        over every brick of the padded grid, ghost bricks included)."""
        key = (shape, int(kcol), bool(every))
        if self.brick_layout != 0:
            raise ValueError("plans are built for the 8x8x8 layout only")
        if key not in self._plans:
            blist = np.arange(self.nbricks, dtype=np.uint32) if every else self.sweep_list
            self._plans[key] = Plan(self.info, blist, shape, kcol)
        return self._plans[key]

    def _declare_box(self, plan, stream=None, fused: bool = False) -> None:
        """Ahead of a sequence of sweeps that refresh this grid: declare one
        of its own quad plans a periodic box, once, and bind the tables that
        the sequence comes with."""
        adj, pairs = getattr(self.info, "dev", None), self.d_pairs
        if adj is None:
            return
        off, img = self.ghost_images if fused else (None, None)
        # (a table that was written into is as good as another: its binding ended)
        try:
            tables = ((adj.stamp, pairs and pairs.stamp) if off is None else
                      (adj.stamp, pairs and pairs.stamp, off.stamp, img.stamp))
        except AttributeError:  # memory of the caller's own kind
            tables = tuple(t and getattr(t, "stamp", t.ptr) for t in (adj, pairs, off, img))
        if tables in plan.tables or plan.shape != "quad":
            return
        if not plan.boxed and not any(plan is p for p in list(self._plans.values())):
            return
        with plan.lock:
            if tables in plan.tables:
                return
            try:
                if not plan.boxed:
                    plan.set_box(self.info, self.nb, self.interior, self.pairs, stream)
                plan.bind_box(adj.ptr, pairs and pairs.ptr, self.npairs, off and off.ptr,
                              img and img.ptr, stream=stream)
            except _lib.BrickError as e:
                if e.code == _lib.BK_ERR_NOMEM:
                    return  # one sweep per pass now; the next sequence tries again
                if e.code != _lib.BK_ERR_UNSUPPORTED:
                    raise
                # not a periodic box (changed tables): one sweep per pass with them
            if len(plan.tables) > 64:
                plan.tables.clear()
            plan.tables.add(tables)

    @property
    def ghost_images(self):
        """(d_img_off, d_img): the ghost images of every brick as CSR in HBM
        (bk_ghost_images), for the fused refresh; built on first use."""
        if getattr(self, "_images", None) is None:
            n = C.c_uint32()
            check(load().bk_ghost_images(longs(self.nb), None, None, C.byref(n)))
            off = np.zeros(self.nbricks + 1, np.uint32)
            img = np.zeros(max(1, n.value), np.uint32)
            check(load().bk_ghost_images(longs(self.nb), off.ctypes.data_as(_lib.u32p),
                                         img.ctypes.data_as(_lib.u32p), C.byref(n)))
            self._images = (DeviceBuffer.from_array(off), DeviceBuffer.from_array(img))
        return self._images

    @property
    def d_every(self) -> DeviceBuffer:
        """Every brick of the padded grid in grid order, in HBM (the sweep
        list of brick_stencil(..., skip = 0), weak/main.cpp:26-36)."""
        if getattr(self, "_d_every", None) is None:
            self._d_every = DeviceBuffer.from_array(np.arange(self.nbricks, dtype=np.uint32))
        return self._d_every

    def auto_plan(self, stencil_kind: int, dtype: int = BK_F64):
        """Default schedule per stencil and dtype: the tuned one when tune()
        ran for the stencil on this grid, else DEFAULT_PLANS (measured on
        MI355X at 512^3).  The 4x8x16 layouts always run one brick per
        wave."""
        tuned = self._tuned.get(int(stencil_kind))
        if tuned is not None:
            return None if tuned.plan_shape == 0 else self.plan(
                "quad" if tuned.plan_shape == _lib.BK_PLAN_QUAD else "column", tuned.kcol)
        if self.brick_layout != 0:
            return None
        choice = DEFAULT_PLANS.get((int(stencil_kind), int(dtype)))
        if choice is None:
            return None
        n = self.interior.size
        if int(stencil_kind) == _lib.BK_CUBE125:
            # levels per unit by size: one wave marches a unit, so small grids
            # need short units to fill the device (up to 4500 bricks in FP64 and
            # 130000 in the narrower types the library takes other forms, with
            # any plan).  us a sweep, FP64: 160^3 1 level 32, 2 levels 37, 6
            # levels 91; 176^3 1 level 40, 2 levels 48; 192^3 50 / 49; 256^3 2
            # levels 90, 1 level 99, 4 levels 95, 6 levels 134; 320^3 2 levels
            # 177, 6 levels 189; 384^3 3 levels 283, 4 levels 292, 2 levels
            # 296, 6 levels 310.  1024^3: 4, 5, 6, 8 and 12 levels within
            # 1.5 % on one host, 8 never the slower.
            choice = ("quad", 8 if n > (1 << 20) else 6 if n > 200000 else 3 if n > 80000
                      else 2 if n > 12500 else 1)
        else:
            choice = ("quad", star_levels(int(stencil_kind), int(dtype), n, choice[1]))
        return self.plan(*choice)

    def auto_wg_bricks(self, stencil_kind: int) -> int:
        """Bricks per workgroup of the per-brick kernels: the tuned value,
        else the kernels' default (0)."""
        tuned = self._tuned.get(int(stencil_kind))
        return tuned.wg_bricks if tuned is not None else 0

    def auto_lane_shift(self, stencil_kind: int, dtype: int = BK_F64) -> int:
        """lane_shift of the quad star kernels: the tuned value, else
        DEFAULT_LANE_SHIFT."""
        tuned = self._tuned.get(int(stencil_kind))
        if tuned is not None:
            return int(tuned.lane_shift)
        return DEFAULT_LANE_SHIFT.get((int(stencil_kind), int(dtype)), 0)

    @property
    def cell_extents(self) -> tuple:
        """Interior cells per axis (i, j, k)."""
        BK, BJ, BI = self.extents
        return (self.nb[0] * BI, self.nb[1] * BJ, self.nb[2] * BK)

    def tune(self, st, dtype: int = BK_F64, steps: int = 5, stream=None, rounds: int = 3,
             warm_s: float = 0.3) -> dict:
        """Time every schedule of this grid's layout for stencil `st`
        (bk_tune_sweep on a grid of the same cells and ghost layer: per
        brick with 1/2/4/8 bricks per workgroup, k-columns or column quads)
        and make the fastest this grid's choice for plan="auto".  All
        schedules compute the same bits.  Returns {"best": candidate,
        "ms": {candidate: ms per sweep}} with candidates named by
        cand_name()."""
        res = tune(st, self.cell_extents, dtype, ghost=self.ghost, steps=steps, rounds=rounds,
                   warm_s=warm_s, layouts=(self.brick_layout,), stream=stream)
        self._tuned[int(st.kind)] = res[0]
        return {"best": cand_name(res[0]), "ms": {cand_name(c): round(c.ms, 4) for c in res}}

    @property
    def nbricks(self) -> int:
        return self.info.nbricks

    @property
    def npairs(self) -> int:
        return self.pairs.size // 2

    @property
    def cells(self) -> int:
        return 512 * self.interior.size

    def field_storage(self, dtype: int = BK_F64, fields: int = 1) -> BrickStorage:
        """A storage of ``fields`` interleaved fields per chunk (step
        512*fields), like stencils/3axis.cpp:26-28 when fields == 2."""
        return BrickStorage.allocate(self.nbricks, BRICK_ELEMS * fields, dtype)

    def fill_uniform(self, brick: Brick, seed: int, lo: float = -1.0, hi: float = 1.0,
                     stream=None) -> None:
        check(load().bk_fill_uniform_layout(self.brick_layout, brick.dtype, _vp(brick.ptr),
                                            C.c_size_t(brick.step), longs(self.nb), self.ghost,
                                            C.c_uint64(seed), lo, hi, _vp(_stream_of(stream))))

    def ghost_refresh(self, brick: Brick, stream=None) -> None:
        if not self.npairs:
            return
        check(load().bk_ghost_refresh(brick.dtype, _vp(brick.ptr), C.c_size_t(brick.step),
                                      C.c_size_t(BRICK_ELEMS), _vp(self.d_pairs.ptr),
                                      C.c_uint32(self.npairs), _vp(_stream_of(stream))))

    def stats(self, brick: Brick, stream=None) -> np.ndarray:
        out = np.zeros(3)
        check(load().bk_field_stats(brick.dtype, _vp(brick.ptr), C.c_size_t(brick.step),
                                    _vp(self.d_interior.ptr), C.c_uint32(self.interior.size),
                                    C.c_size_t(BRICK_ELEMS), out.ctypes.data_as(_lib.dblp),
                                    _vp(_stream_of(stream))))
        return out

    def compare(self, a: Brick, ref: Brick, floor: float = 1.0, atol: float = 0.0,
                rtol: float = 0.0, stream=None) -> dict:
        out = np.zeros(5)
        check(load().bk_field_compare(a.dtype, _vp(a.ptr), C.c_size_t(a.step), ref.dtype,
                                      _vp(ref.ptr), C.c_size_t(ref.step),
                                      _vp(self.d_interior.ptr), C.c_uint32(self.interior.size),
                                      C.c_size_t(BRICK_ELEMS), floor, atol, rtol,
                                      out.ctypes.data_as(_lib.dblp), _vp(_stream_of(stream))))
        n = self.cells
        return {"max_abs": out[0], "max_rel": out[1],
                "rms_rel": float(np.sqrt(out[2] / out[3])) if out[3] > 0 else 0.0,
                "rms_abs": float(np.sqrt(out[2] / n)), "bad": int(out[4])}


def _resolve_plan(plan, st: Stencil, grid: PeriodicGrid, dtype: int = BK_F64):
    if plan is None:
        return None
    if isinstance(plan, str):
        if plan == "auto":
            return grid.auto_plan(st.kind, dtype)
        return grid.plan(plan)
    return plan


# bk_sweep_desc's fields in order, padded to its size
_DESC = struct.Struct("@iiPPIPNPNPdiPiii0P")
assert _DESC.size == C.sizeof(bk_sweep_desc)


def _address(a: np.ndarray) -> int:
    """The address of a contiguous array's data (a.ctypes.data takes 1 us)."""
    if a.size and a.flags.writeable:
        return C.addressof(C.c_char.from_buffer(a))
    return a.ctypes.data


def _desc(st: Stencil, out: Brick, inp: Brick, grid: PeriodicGrid, coeff_keep: list,
          blist: DeviceBuffer | None = None, nlist: int | None = None,
          plan=None, wg_bricks=None, lane_shift=None) -> bk_sweep_desc:
    if out.dtype != inp.dtype:
        raise ValueError("input and output fields must share a dtype")
    kind, dtype = st.kind, inp.dtype
    coeff = np.ascontiguousarray(st.coeff, dtype=np.float64)
    if coeff.size != NCOEFF.get(kind, 0):
        raise ValueError(f"stencil {kind} takes {NCOEFF.get(kind, 0)} "
                         f"coefficients, got {coeff.size}")
    coeff_keep.append(coeff)
    pl = _resolve_plan(plan, st, grid, dtype)
    coeff_keep.append(pl)
    if wg_bricks is None:
        wg_bricks = (grid.auto_wg_bricks(kind)
                     if plan == "auto" and hasattr(grid, "auto_wg_bricks") else 0)
    if lane_shift is None:
        # automatic: only where the kernels have it (quad plans of the stars)
        quad_star = pl is not None and pl.shape == "quad" and kind != _lib.BK_CUBE125
        lane_shift = (grid.auto_lane_shift(kind, dtype)
                      if quad_star and hasattr(grid, "auto_lane_shift") else 0)
    # packed at once: field by field, with numpy's data_as for the
    # coefficients, the record took 4.0 us of a small sweep's 7.4, now 2.3 of
    # 6.0
    return bk_sweep_desc.from_buffer_copy(_DESC.pack(
        kind, dtype, grid.info.dptr, (blist or grid.d_sweep_list).ptr or 0,
        grid.interior.size if nlist is None else nlist, inp.ptr or 0, inp.step, out.ptr or 0,
        out.step, _address(coeff), float(st.theta), int(st.cond_mode),
        pl.handle or 0 if pl is not None else 0, getattr(grid, "brick_layout", 0),
        0 if pl is not None else int(wg_bricks), int(lane_shift)))


def sweep(st: Stencil, out: Brick, inp: Brick, grid: PeriodicGrid, stream=None,
          plan="auto", wg_bricks=None, lane_shift=None) -> None:
    """One sweep over the interior bricks: out = stencil(in).  ``plan`` is
    "auto", None (plain brick list, one brick per wave), "column", "quad"
    or a Plan; ``wg_bricks`` the bricks per workgroup of the per-brick
    kernels (None: tuned or default); ``lane_shift`` 1 for the i-taps by
    DPP lane shifts in the quad star kernels (None: tuned or default)."""
    keep: list = []
    d = _desc(st, out, inp, grid, keep, plan=plan, wg_bricks=wg_bricks, lane_shift=lane_shift)
    check(load().bk_sweep(C.byref(d), _stream_of(stream)))


def sweeps(st: Stencil, a: Brick, b: Brick, grid: PeriodicGrid, nsweeps: int,
           use_graph: bool = False, refresh: bool = True, stream=None, plan="auto",
           ghost_iters: int = 1, fused: bool = False, wg_bricks=None,
           lane_shift=None) -> Brick:
    """``nsweeps`` ping-pong sweeps a->b->a..., each preceded by the periodic
    ghost refresh of its input -- or, with ghost_iters > 1, the refresh once
    per ghost_iters sweeps and the sweeps in between over every brick of the
    padded grid (bk_sweeps_deep), or, with fused=True, the refresh folded
    into the sweeps' stores (bk_sweeps_fused; stars and cond, one brick per
    wave or by quad plans).  Same result in every form.  Returns the field
    holding the result."""
    keep: list = []
    if ghost_iters != 1 and lane_shift is None:
        lane_shift = 0  # the sweeps over every brick run without quad plans
    d = _desc(st, b, a, grid, keep, plan=plan, wg_bricks=wg_bricks, lane_shift=lane_shift)
    pairs = grid.d_pairs.ptr if (refresh and grid.d_pairs is not None) else None
    npairs = grid.npairs if refresh else 0
    if (nsweeps > 3 and keep[-1] is not None and ghost_iters == 1
            and (npairs or st.kind in STEP_STENCILS) and hasattr(grid, "_declare_box")
            and npairs == grid.npairs):  # (ghost bricks left alone are boundary values)
        grid._declare_box(keep[-1], stream, fused)
    if fused:
        if ghost_iters != 1:
            raise ValueError("the fused refresh refreshes every sweep (ghost_iters = 1)")
        io, im = grid.ghost_images
        check(load().bk_sweeps_fused(C.byref(d), _vp(io.ptr), _vp(im.ptr), _vp(pairs),
                                     C.c_uint32(npairs), int(nsweeps), int(bool(use_graph)),
                                     _vp(_stream_of(stream))))
    elif ghost_iters == 1:
        check(load().bk_sweeps(C.byref(d), _vp(pairs), C.c_uint32(npairs), int(nsweeps),
                               int(bool(use_graph)), _vp(_stream_of(stream))))
    else:
        # sweeps over every brick: column plans as for the interior; the
        # cube per brick (quad plans cannot take the outer layer of a
        # non-periodic grid, bk_plan_create rejects them)
        ip = _resolve_plan(plan, st, grid, a.dtype)
        ap = (grid.plan(ip.shape, ip.kcol, every=True)
              if ip is not None and ip.shape != "quad" else None)
        keep.append(ap)
        check(load().bk_sweeps_deep(C.byref(d), _vp(grid.d_every.ptr), C.c_uint32(grid.nbricks),
                                    _vp(ap.handle if ap is not None else None), _vp(pairs),
                                    C.c_uint32(npairs), int(nsweeps), int(ghost_iters),
                                    int(bool(use_graph)), _vp(_stream_of(stream))))
    return b if nsweeps % 2 == 1 else a


def sweep_passes(st: Stencil, a: Brick, b: Brick, grid: PeriodicGrid, nsweeps: int,
                 plan="auto", fused: bool = False) -> list:
    """The passes that ``sweeps`` of these arguments takes over the fields, as
    (sweeps, form) pairs (bk_sweeps_passes; forms BK_PASS_*).  The box is
    declared by the first such sequence itself."""
    keep: list = []
    d = _desc(st, b, a, grid, keep, plan=plan)
    images = tuple(_vp(t.ptr) for t in grid.ghost_images) if fused else (None, None)
    pairs = _vp(grid.d_pairs.ptr) if grid.d_pairs is not None else None
    count, cap = C.c_int(), max(int(nsweeps), 1)
    ts, forms = (C.c_int * cap)(), (C.c_int * cap)()
    check(load().bk_sweeps_passes(C.byref(d), *images, pairs, grid.npairs, int(nsweeps), ts, forms,
                                  cap, C.byref(count)))
    return list(zip(ts[:count.value], forms[:count.value]))


def cand_name(c) -> str:
    """A tuner candidate as text: layout, then the schedule."""
    lay = {0: "8x8x8", 1: "4x8x16", 2: "4x8x16/f88"}[c.layout]
    if c.plan_shape == 0:
        return f"{lay} brick wg{c.wg_bricks}"
    shape = "quad" if c.plan_shape == _lib.BK_PLAN_QUAD else "column"
    return f"{lay} {shape}{c.kcol}" + ("+dpp" if c.lane_shift else "")


def tune(st: Stencil, cells, dtype: int = BK_F64, ghost: int = 1, steps: int = 5,
         rounds: int = 3, warm_s: float = 0.3, layouts=(0, 1, 2), batch_only: bool = False,
         stream=None) -> list:
    """bk_tune_sweep: time every (layout, schedule) candidate for stencil
    `st` on a periodic grid of `cells` (i, j, k) and return them fastest
    first (bk_tune_cand records: layout, plan_shape, kcol, wg_bricks,
    lane_shift, ms)."""
    flags = 0
    for lay in layouts:
        flags |= 1 << int(lay)
    if batch_only:
        flags |= _lib.BK_TUNE_BATCH_SCHEDULES
    coeff = np.ascontiguousarray(st.coeff, dtype=np.float64)
    n = C.c_uint32()
    args = (int(st.kind), int(dtype), coeff.ctypes.data_as(_lib.dblp), float(st.theta),
            int(st.cond_mode), longs(cells), int(ghost), int(steps), int(rounds), float(warm_s),
            C.c_uint(flags))
    check(load().bk_tune_sweep(*args, None, 0, C.byref(n), None))
    out = (_lib.bk_tune_cand * n.value)()
    check(load().bk_tune_sweep(*args, out, n.value, C.byref(n), _vp(_stream_of(stream))))
    return list(out[:n.value])


__all__ = [
    "tune", "cand_name", "DeviceBuffer", "Stream", "Event", "BrickInfo", "init_grid", "movBrickInfo",
    "BrickStorage", "movBrickStorage", "Brick", "copyToBrick", "copyFromBrick",
    "PeriodicGrid", "Plan", "plan_host", "sweep", "sweeps", "sweep_passes", "device_count", "device_sync", "DTYPE_NP",
    "DTYPE_SIZE", "BK_F64", "BK_F32", "BK_BF16",
]
