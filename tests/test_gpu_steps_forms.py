"""Every kernel that takes several sweeps per pass, asked for by name: boxes
that the model of their times sends to it (checked), ragged in every axis, bit
for bit what single sweeps of one brick per wave leave in both fields -- and in
all of their ghost bricks, where the refresh is fused."""
import numpy as np
import pytest

from bricklib_amd._lib import BK_PASS_BLOCKS, BK_PASS_STRIPS
from bricklib_amd.bricks import sweep_passes

pytestmark = pytest.mark.gpu

DT = {"f64": 0, "f32": 1, "bf16": 2}
# name, theta, cond mode: 7-point; cond with values and with clamped values in
# registers; 13-point
STENCILS = {"7pt": ("7pt", None, 0), "raw": ("cond", -0.07, 1), "clamped": ("cond", 0.04, 1),
            "13pt": ("13pt", None, 0)}


def _run(bk, g, st, dt, n, plan, fused):
    a, b = (bk.Brick(g.info, g.field_storage(dt), 0) for _ in range(2))
    for f in (a, b):
        f.storage.buf.zero()
    g.fill_uniform(a, 11)
    bk.sweeps(st, a, b, g, n, plan=plan, fused=fused)
    bk.device_sync()
    out = [f.storage.to_host() for f in (a, b)]
    return [(x if fused else x[g.interior]).view(np.uint8) for x in out], (a, b)


def _check(bk, kind, dtype, nb, n, fused):
    """The passes taken, after a comparison of all they leave."""
    name, theta, mode = STENCILS[kind]
    st = bk.Stencil.make(name, seed=7, cond_mode=mode)
    if theta is not None:
        st.theta = theta
    g = bk.PeriodicGrid(nb, ghost=1)
    got, fields = _run(bk, g, st, DT[dtype], n, "auto", fused)
    want, _ = _run(bk, g, st, DT[dtype], n, None, fused)
    for x, y in zip(got, want):
        assert np.array_equal(x, y)
    return sweep_passes(st, *fields, g, n, fused=fused)


@pytest.mark.parametrize("fused", [False, True], ids=["separate", "fused"])
@pytest.mark.parametrize("kind,dtype,sweeps,nb,n", [
    ("7pt", "f64", 3, (26, 5, 27), 8), ("7pt", "f64", 4, (19, 31, 7), 9),
    ("7pt", "f32", 3, (67, 30, 3), 5), ("7pt", "f32", 4, (28, 39, 6), 9),
    ("7pt", "bf16", 3, (39, 65, 5), 7), ("7pt", "bf16", 4, (20, 31, 52), 9),
    ("raw", "f64", 3, (53, 14, 8), 5), ("raw", "f32", 3, (41, 47, 7), 6),
    ("raw", "f32", 4, (103, 67, 8), 9), ("clamped", "f64", 3, (16, 11, 27), 6),
    ("clamped", "f64", 4, (23, 49, 6), 9), ("clamped", "f32", 3, (43, 39, 7), 5),
    ("clamped", "f32", 4, (35, 62, 18), 9), ("13pt", "f64", 2, (49, 33, 4), 5),
    ("13pt", "f32", 2, (41, 47, 9), 5)])
def test_strips(gpu, kind, dtype, sweeps, nb, n, fused):
    assert (sweeps, BK_PASS_STRIPS) in _check(gpu, kind, dtype, nb, n, fused)


@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("kind", list(STENCILS))
@pytest.mark.parametrize("nb", [(3, 5, 7), (5, 7, 9)], ids=["half", "whole"])
def test_blocks(gpu, nb, kind, dtype):
    passes = []
    for n, fused in ((5, False), (8, True), (9, True)):
        passes += _check(gpu, kind, dtype, nb, n, fused)
    for sweeps in ((2,) if kind == "13pt" else (3, 4)):
        assert (sweeps, BK_PASS_BLOCKS) in passes
