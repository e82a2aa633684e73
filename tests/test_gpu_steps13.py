"""Two sweeps of the 13-point star per pass over a declared box: bit for bit what
single sweeps of the per-brick kernels leave in both fields, by half bricks (up
to 128 bricks), by bricks and by strips (large boxes of FP64 and FP32), ragged
strips and groups, wrapped and ghosted boxes, replays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = {"f64": 0, "f32": 1, "bf16": 2}


def _run(bk, g, st, dt, n, plan, reps=1, **kw):
    a, b = (bk.Brick(g.info, g.field_storage(dt), 0) for _ in range(2))
    for f in (a, b):
        f.storage.buf.zero()
    for _ in range(reps):
        g.fill_uniform(a, 11)
        res = bk.sweeps(st, a, b, g, n, plan=plan, **kw)
        bk.device_sync()
    assert (res is b) == (n % 2 == 1)
    return [np.ascontiguousarray(f.storage.to_host()[g.interior]).view(np.uint8) for f in (a, b)]


def _check(bk, nb, n, dtype, ghosts=(0, 1)):
    st = bk.Stencil.make("13pt", seed=7)
    for ghost in ghosts:
        g = bk.PeriodicGrid(nb, ghost=ghost)
        want = _run(bk, g, st, DT[dtype], n, None)
        for kw in (dict(), dict(use_graph=True, reps=3)):
            for x, y in zip(_run(bk, g, st, DT[dtype], n, "auto", **kw), want):
                assert np.array_equal(x, y), (ghost, kw)


@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("nb,n", [((1, 1, 1), 5), ((1, 2, 1), 9), ((2, 3, 1), 14), ((8, 4, 4), 8),
                                  ((3, 43, 1), 6), ((9, 5, 3), 29), ((8, 1, 17), 31)])
def test_small_boxes(gpu, nb, n, dtype):
    _check(gpu, nb, n, dtype)


@pytest.mark.parametrize("dtype,nb,n", [
    ("f64", (8, 25, 26), 9), ("f64", (15, 19, 18), 5), ("f64", (1, 3, 1700), 5),
    ("f64", (7, 1, 720), 9), ("f64", (20, 23, 31), 13), ("f32", (16, 29, 29), 9),
    ("f32", (6, 47, 47), 5), ("f32", (29, 25, 25), 13), ("bf16", (22, 25, 24), 9)])
def test_strips(gpu, dtype, nb, n):
    _check(gpu, nb, n, dtype, ghosts=(1,))
