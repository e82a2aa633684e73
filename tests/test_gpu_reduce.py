"""Field statistics and comparison against numpy in FP64: every pair of element
types, brick sizes off the vector width and off the block's chunks, lists
shorter than a block and longer than a pass, zero and positive floors, NaN and
infinite cells, and the counter's return between calls."""
import ctypes as C

import numpy as np
import pytest

from bricklib_amd import _lib
from bricklib_amd._lib import check

pytestmark = pytest.mark.gpu

NP = {0: np.float64, 1: np.float32, 2: np.uint16}


def _wide(x, dt):
    return ((x.astype(np.uint32) << 16).view(np.float32) if dt == 2 else x).astype(np.float64)


def _field(rng, dt, n, step):
    x = rng.uniform(-1, 1, (n, step))
    if dt == 2:
        return (x.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    return x.astype(NP[dt])


def _call(bk, a, dta, r, dtr, lst, elems, floor, atol, rtol):
    lib = bk.load()
    da, dr, dl = (bk.DeviceBuffer.from_array(v) for v in (a, r, lst))
    vp = lambda b: C.c_void_p(b.ptr)  # noqa: E731
    s, c = np.zeros(3), np.zeros(5)
    args = (vp(dl), C.c_uint32(lst.size), C.c_size_t(elems))
    check(lib.bk_field_stats(dta, vp(da), C.c_size_t(a.shape[1]), *args,
                             s.ctypes.data_as(_lib.dblp), None))
    check(lib.bk_field_compare(dta, vp(da), C.c_size_t(a.shape[1]), dtr, vp(dr),
                               C.c_size_t(r.shape[1]), *args, floor, atol, rtol,
                               c.ctypes.data_as(_lib.dblp), None))
    return s, c


def _want(x, y, floor, atol, rtol):
    with np.errstate(all="ignore"):
        d, m = np.abs(x - y), np.abs(y)
        ratio = d / np.maximum(np.where(np.isnan(m), floor, m), floor)
        return (np.array([x.sum(), (x * x).sum(), np.nanmax(np.abs(x), initial=0.0)]),
                np.array([np.nanmax(d, initial=0.0), np.nanmax(ratio, initial=0.0), (d * d).sum(),
                          (y * y).sum(), (d > atol + rtol * m).sum()]))


# sums of n terms of size <= 1 in any order: n * 2^-53 of the sum of absolute
# values; maxima and the count are exact
def _check(got, want, x, y):
    (s, c), (ws, wc) = got, want
    n = max(1, x.size)
    eps = n * 2.0 ** -53
    assert abs(s[0] - ws[0]) <= eps * np.abs(x).sum() and s[2] == ws[2]
    assert abs(s[1] - ws[1]) <= eps * ws[1]
    assert c[0] == wc[0] and c[1] == wc[1] and c[4] == wc[4]
    assert abs(c[2] - wc[2]) <= eps * wc[2] and abs(c[3] - wc[3]) <= eps * wc[3]


@pytest.mark.parametrize("dta", [0, 1, 2], ids=["f64", "f32", "bf16"])
@pytest.mark.parametrize("dtr", [0, 1, 2], ids=["f64", "f32", "bf16"])
@pytest.mark.parametrize("elems,n", [(512, 1), (512, 700), (512, 5000), (64, 3001), (6, 999),
                                     (500, 40), (1, 5), (1000, 33), (4096, 9)])
def test_against_numpy(gpu, dta, dtr, elems, n):
    rng = np.random.default_rng(n + elems)
    a, r = _field(rng, dta, n + 2, elems + 3), _field(rng, dtr, n + 2, elems)
    lst = rng.permutation(n + 2)[:n].astype(np.uint32)
    x, y = _wide(a[lst, :elems], dta), _wide(r[lst, :elems], dtr)
    for floor, atol, rtol in ((1.0, 0.0, 0.0), (1e-3, 0.1, 0.5)):
        _check(_call(gpu, a, dta, r, dtr, lst, elems, floor, atol, rtol),
               _want(x, y, floor, atol, rtol), x, y)


def test_special_values(gpu):
    rng = np.random.default_rng(2)
    a, r = _field(rng, 0, 600, 512), _field(rng, 0, 600, 512)
    lst = np.arange(600, dtype=np.uint32)
    for cells in ((0.0, 0.0), (0.5, 0.0), (5e-324, 1e-310), (1e308, -1e308), (np.inf, 1.0),
                  (np.nan, 1.0), (1.0, np.nan), (1.0, np.inf)):
        u, v = a.copy(), r.copy()
        u[100, 7], v[100, 7] = cells
        for floor in (0.0, 1e-2):
            s, c = _call(gpu, u, 0, v, 0, lst, 512, floor, 0.1, 0.5)
            ws, wc = _want(u, v, floor, 0.1, 0.5)
            assert s[2] == ws[2] and c[0] == wc[0] and c[1] == wc[1] and c[4] == wc[4], cells


def test_empty_list(gpu):
    a = np.ones((2, 512))
    s, c = _call(gpu, a, 0, a, 0, np.zeros(0, np.uint32), 512, 1.0, 0.0, 0.0)
    assert not s.any() and not c.any()
