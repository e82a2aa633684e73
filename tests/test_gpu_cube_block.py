"""The cube's block form (a workgroup per plan level) and the sizes where it
hands over to one plane a wave, two planes a wave and the marching form: bit
for bit the per-brick kernel's results, for odd boxes, units of several
levels (walked up from their anchors), shuffled and partial brick lists."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = {"f64": 0, "f32": 1, "bf16": 2}


def _pair(bk, g, dt):
    a, b, c = (bk.Brick(g.info, g.field_storage(dt), 0) for _ in range(3))
    g.fill_uniform(a, 21)
    g.ghost_refresh(a)
    for f in (b, c):
        f.storage.buf.zero()
    return a, b, c


@pytest.mark.parametrize("dtype,nb,levels", [
    ("f64", (1, 1, 1), 1), ("f64", (1, 2, 3), 2), ("f64", (5, 3, 4), 3), ("f64", (12, 13, 12), 1),
    ("f64", (13, 13, 12), 2), ("f64", (16, 17, 16), 1), ("f64", (17, 17, 17), 1),
    ("f64", (17, 16, 19), 3), ("f32", (1, 1, 1), 2), ("f32", (3, 5, 2), 1),
    ("f32", (19, 20, 21), 1), ("f32", (21, 21, 21), 2), ("f32", (25, 24, 25), 1),
    ("bf16", (2, 3, 3), 1), ("bf16", (20, 21, 20), 3), ("bf16", (25, 23, 25), 2)])
def test_block_matches_per_brick(gpu, dtype, nb, levels):
    bk = gpu
    st = bk.Stencil.make("125pt", seed=5)
    for ghost in (0, 1):
        g = bk.PeriodicGrid(nb, ghost=ghost)
        a, b, c = _pair(bk, g, DT[dtype])
        bk.sweep(st, b, a, g, plan=g.plan("quad", levels))
        bk.sweep(st, c, a, g, plan=None)
        x, y = b.storage.to_host(), c.storage.to_host()
        assert np.array_equal(x.view(np.uint8), y.view(np.uint8))


@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_partial_lists(gpu, dtype):
    """Plans over some of the bricks, in shuffled order: members that are not
    listed are not written, and their neighbours are not needed."""
    bk = gpu
    st = bk.Stencil.make("125pt", seed=6)
    g = bk.PeriodicGrid((5, 6, 4))
    rng = np.random.default_rng(3)
    for keep in (0.2, 0.6, 1.0):
        lst = rng.permutation(g.interior)[:max(1, int(keep * g.interior.size))]
        a, b, c = _pair(bk, g, DT[dtype])
        plan = bk.Plan(g.info, lst, "quad", 2)
        bk.sweep(st, b, a, g, plan=plan)
        bk.sweep(st, c, a, g, plan=None)
        x, y = b.storage.to_host(), c.storage.to_host()
        assert np.array_equal(x[lst].view(np.uint8), y[lst].view(np.uint8))
        rest = np.setdiff1d(np.arange(g.nbricks), lst)
        assert not x[rest].any()


def test_non_periodic_grid_interior(gpu):
    """A grid whose out-of-range neighbours are brick 0: the plan covers its
    inner bricks only."""
    bk = gpu
    st = bk.Stencil.make("125pt", seed=7)
    g = bk.PeriodicGrid((4, 3, 5))
    a, b, c = _pair(bk, g, 0)
    inner = g.grid[2:-2, 2:-2, 2:-2].reshape(-1)
    bk.sweep(st, b, a, g, plan=bk.Plan(g.info, inner, "quad", 1))
    bk.sweep(st, c, a, g, plan=None)
    x, y = b.storage.to_host(), c.storage.to_host()
    assert np.array_equal(x[inner], y[inner])
