"""Sequences honour the tables that they are called with, also after the same
sequence has run over the periodic box: ghost pairs, ghost images or an
adjacency replaced or written in place afterwards -- bit for bit what one brick
per wave gives with those tables, and again what the periodic ones give once
they are back."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NB = (6, 5, 4)


def _run(bk, g, st, n, plan, **kw):
    a, b = (bk.Brick(g.info, g.field_storage(0), 0) for _ in range(2))
    for f in (a, b):
        f.storage.buf.zero()
    g.fill_uniform(a, 11)
    g.ghost_refresh(a)
    bk.sweeps(st, a, b, g, n, plan=plan, **kw)
    bk.device_sync()
    return [f.storage.to_host()[g.interior].view(np.uint64) for f in (a, b)]


def _check(bk, g, st, kw):
    got = {}
    for n in (3, 9):
        want = _run(bk, g, st, n, None, **kw)
        got[n] = _run(bk, g, st, n, "auto", **kw)
        for x, y in zip(got[n], want):
            assert np.array_equal(x, y), n
    return got


def _rolled(pairs):
    """Every ghost brick takes another brick's values."""
    p = pairs.reshape(-1, 2).copy()
    p[:, 1] = np.roll(p[:, 1], 7)
    return p


def _images(nbricks, pairs):
    order = np.argsort(pairs[:, 1], kind="stable")
    off = np.zeros(nbricks + 1, np.uint32)
    off[1:] = np.cumsum(np.bincount(pairs[:, 1], minlength=nbricks))
    return off, np.ascontiguousarray(pairs[order, 0], np.uint32)


def _swapped(g):
    """The adjacency with two ghost bricks of the i- face for each other."""
    to = np.arange(g.nbricks, dtype=np.uint32)
    p, q = g.info.adj[g.interior[[0, 2 * NB[0]]], 12]
    to[p], to[q] = q, p
    return to[g.info.adj]


@pytest.mark.parametrize("use_graph", [False, True], ids=["queued", "graph"])
@pytest.mark.parametrize("what,fused", [("pairs", False), ("pairs", True), ("adjacency", False),
                                        ("adjacency", True), ("images", True)])
@pytest.mark.parametrize("name", ["7pt", "25pt"])
def test_changed_tables(gpu, name, what, fused, use_graph):
    bk = gpu
    st = bk.Stencil.make(name, seed=3)
    g = bk.PeriodicGrid(NB)
    kw = dict(fused=fused, use_graph=use_graph)
    first = _check(bk, g, st, kw)

    def put(other, in_place):
        if what == "pairs":
            p = np.ascontiguousarray(_rolled(g.pairs) if other else g.pairs.reshape(-1, 2))
            if in_place:
                g.d_pairs.upload(p)
            else:
                g.d_pairs = bk.DeviceBuffer.from_array(p)
        elif what == "adjacency":
            adj = _swapped(g) if other else g.info.adj
            if in_place:
                g.info.dev.upload(adj)
            else:
                g.info.dev = bk.DeviceBuffer.from_array(adj)
        else:
            off, img = _images(g.nbricks, _rolled(g.pairs) if other else g.pairs.reshape(-1, 2))
            if in_place:
                for t, x in zip(g.ghost_images, (off, img)):
                    t.upload(x)
            else:
                g._images = tuple(bk.DeviceBuffer.from_array(x) for x in (off, img))

    for in_place in (True, False):
        for other in (True, False):
            put(other, in_place)
            got = _check(bk, g, st, kw)
            for n in first:
                same = all(np.array_equal(x, y) for x, y in zip(got[n], first[n]))
                assert same != other, (in_place, n)
            # several sweeps per pass again once the periodic ones are back
            a, b = (bk.Brick(g.info, g.field_storage(0), 0) for _ in range(2))
            passes = bk.sweep_passes(st, a, b, g, 9, fused=fused)
            assert (len(passes) < 9) == (name == "7pt" and not other), (in_place, passes)


def test_unbind(gpu):
    """unbind_box ends the bindings for tables written by other means, and
    bind_box refuses what is not the box."""
    bk = gpu
    g = bk.PeriodicGrid(NB)
    plan = g.plan("quad", 1)
    with pytest.raises(bk.BrickError):
        plan.bind_box(g.info.dptr, g.d_pairs.ptr, g.npairs)  # no box yet
    plan.set_box(g.info, g.nb, g.interior, g.pairs)
    other = bk.DeviceBuffer.from_array(_rolled(g.pairs))
    swapped = bk.DeviceBuffer.from_array(_swapped(g))
    off, img = _images(g.nbricks, _rolled(g.pairs))
    d_off, d_img = (bk.DeviceBuffer.from_array(x) for x in (off, img))
    for args in [(g.info.dptr, other.ptr, g.npairs), (swapped.ptr, g.d_pairs.ptr, g.npairs),
                 (g.info.dptr, g.d_pairs.ptr, g.npairs - 1), (g.info.dptr, 0, 0),
                 (g.info.dptr, g.d_pairs.ptr, g.npairs, d_off.ptr, d_img.ptr)]:
        with pytest.raises(bk.BrickError) as e:
            plan.bind_box(*args)
        assert e.value.code == 4
    st = bk.Stencil.make("7pt", seed=3)
    want = _run(bk, g, st, 9, None)
    plan.bind_box(g.info.dptr, g.d_pairs.ptr, g.npairs, *(t.ptr for t in g.ghost_images))
    for fused in (False, True):
        assert all(np.array_equal(x, y) for x, y in zip(_run(bk, g, st, 9, plan, fused=fused), want))
    plan.unbind_box()
    assert all(np.array_equal(x, y) for x, y in zip(_run(bk, g, st, 9, plan), want))
