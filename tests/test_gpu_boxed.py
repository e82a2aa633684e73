"""Sequences over a declared periodic box (bk_plan_set_box) whose sweeps read
the periodic images instead of refreshed ghost bricks: every stencil of radius
above 1, boxes down to one brick an axis, odd sizes, both forms of the refresh,
graph replays -- bit for bit the fields of sweeps one by one, each after its
refresh; of the ghost bricks, those of the last sweep's input, and in the fused
form those of both fields, are up to date."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = {"f64": 0, "f32": 1, "bf16": 2}


def _fields(bk, g, dt):
    a, b = (bk.Brick(g.info, g.field_storage(dt), 0) for _ in range(2))
    for f in (a, b):
        f.storage.buf.zero()
    g.fill_uniform(a, 3)
    return a, b


def _bytes(x):
    return np.ascontiguousarray(x).view(np.uint8)


@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("name", ["13pt", "25pt", "125pt"])
@pytest.mark.parametrize("nb,n", [((1, 1, 1), 4), ((1, 2, 3), 5), ((3, 1, 2), 6), ((5, 7, 4), 5),
                                  ((6, 4, 9), 4), ((13, 11, 17), 7), ((33, 20, 21), 4)])
def test_images_for_ghosts(gpu, name, dtype, nb, n):
    bk = gpu
    st = bk.Stencil.make(name, seed=5)
    g = bk.PeriodicGrid(nb)
    wa, wb = _fields(bk, g, DT[dtype])
    src, dst = wa, wb
    for _ in range(n):
        g.ghost_refresh(src)
        bk.sweep(st, dst, src, g)
        src, dst = dst, src
    g.ghost_refresh(src)
    want = [f.storage.to_host() for f in (wa, wb)]
    last = n % 2  # the result's field; the other is the last sweep's input
    for fused in (False, True):
        if fused and name == "125pt":
            continue
        for graph in (False, True):
            f = _fields(bk, g, DT[dtype])
            for rep in range(2 if graph else 1):
                g.fill_uniform(f[0], 3)
                res = bk.sweeps(st, *f, g, n, fused=fused, use_graph=graph)
                assert res is f[last]
            for q in (0, 1):
                x, y = f[q].storage.to_host(), want[q]
                if q == last and not fused:
                    x, y = x[g.interior], y[g.interior]
                assert np.array_equal(_bytes(x), _bytes(y)), (fused, graph, q)
