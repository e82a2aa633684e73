"""Several sweeps per pass (bk_plan_set_box + bk_sweeps): bit for bit what
single sweeps through the per-brick kernels leave in both fields, at the edges
of the kernels' ranges -- boxes by half bricks (up to 128 bricks), by bricks
and by strips (more than 5000 to 12000 bricks by type), ragged strips and
groups, every form of the refresh, both cond forms, interleaved and unaligned
fields, graph replays -- and the calls that must stay on single sweeps."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = {"f64": 0, "f32": 1, "bf16": 2}


def _stencil(bk, name, theta=None, mode=1):
    st = bk.Stencil.make(name, seed=7, cond_mode=mode)
    if theta is not None:
        st.theta = theta
    return st


def _run(bk, g, st, dt, n, plan, **kw):
    a, b = (bk.Brick(g.info, g.field_storage(dt), 0) for _ in range(2))
    for f in (a, b):
        f.storage.buf.zero()
    g.fill_uniform(a, 11)
    res = bk.sweeps(st, a, b, g, n, plan=plan, **kw)
    bk.device_sync()
    assert (res is b) == (n % 2 == 1)
    return a.storage.to_host(), b.storage.to_host()


def _same(g, got, want, whole=False):
    for x, y in zip(got, want):
        if not whole:
            x, y = x[g.interior], y[g.interior]
        assert np.array_equal(x.view(np.uint8), y.view(np.uint8))


CASES = [  # stencil, theta, cond mode
    ("7pt", None, 0), ("cond", None, 0), ("cond", 0.04, 1), ("cond", -0.07, 1)]


@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}{c[1] or ''}m{c[2]}")
@pytest.mark.parametrize("nb,n", [((1, 1, 1), 4), ((1, 2, 1), 9), ((2, 3, 1), 14), ((8, 4, 4), 8),
                                  ((3, 43, 1), 5), ((9, 5, 3), 25), ((8, 1, 17), 31)])
def test_small_boxes(gpu, nb, n, case, dtype):
    bk = gpu
    st = _stencil(bk, *case)
    for ghost in (0, 1):
        g = bk.PeriodicGrid(nb, ghost=ghost)
        _same(g, _run(bk, g, st, DT[dtype], n, "auto"), _run(bk, g, st, DT[dtype], n, None))


# boxes just above the sizes that go by strips, 1 to 3 strips along i, short
# last groups of strips along j
@pytest.mark.parametrize("case,dtype,nb,n", [
    (CASES[0], "f64", (8, 25, 26), 9), (CASES[0], "f64", (15, 19, 18), 4),
    (CASES[0], "f64", (1, 3, 1700), 5), (CASES[0], "f64", (7, 1, 720), 8),
    (CASES[0], "f32", (16, 29, 26), 9), (CASES[0], "f32", (6, 45, 45), 8),
    (CASES[0], "bf16", (22, 23, 24), 10), (CASES[1], "f64", (8, 33, 31), 9),
    (CASES[2], "f64", (9, 31, 29), 8), (CASES[3], "f64", (13, 25, 25), 8),
    (CASES[1], "f32", (7, 42, 41), 9), (CASES[2], "bf16", (14, 30, 29), 8),
    (CASES[3], "f32", (8, 38, 40), 7), (CASES[3], "bf16", (20, 25, 25), 8)])
def test_strips(gpu, case, dtype, nb, n):
    bk = gpu
    st = _stencil(bk, *case)
    g = bk.PeriodicGrid(nb, ghost=1)
    _same(g, _run(bk, g, st, DT[dtype], n, "auto"), _run(bk, g, st, DT[dtype], n, None))


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("nb", [(4, 4, 4), (5, 6, 9), (16, 28, 28)])
def test_fused_refresh_and_replays(gpu, nb, dtype):
    """Every brick of both fields, ghosts included, over three replays with
    eager work and a synchronisation between them."""
    bk = gpu
    st = _stencil(bk, "7pt")
    g = bk.PeriodicGrid(nb)
    f = [bk.Brick(g.info, g.field_storage(DT[dtype]), 0) for _ in range(4)]
    for q in f:
        q.storage.buf.zero()
    g.fill_uniform(f[0], 5)
    g.fill_uniform(f[2], 5)
    for _ in range(3):
        bk.sweeps(st, f[0], f[1], g, 10, fused=True, use_graph=True)
        bk.sweeps(st, f[2], f[3], g, 10, fused=True, plan=None)
        bk.device_sync()
        for p, q in ((f[0], f[2]), (f[1], f[3])):
            x, y = p.storage.to_host(), q.storage.to_host()
            assert np.array_equal(x.view(np.uint8), y.view(np.uint8))


def test_matches_oracle(gpu, orc):
    bk = gpu
    for name, nb, n in (("7pt", (5, 4, 3), 20), ("cond", (9, 24, 25), 8), ("7pt", (9, 24, 25), 12)):
        st = _stencil(bk, name)
        g = bk.PeriodicGrid(nb)
        a, b = (bk.Brick(g.info, g.field_storage(0), 0) for _ in range(2))
        g.fill_uniform(a, 3)
        got = bk.sweeps(st, a, b, g, n).storage.to_host()
        og = orc.Grid(nb)
        oa, ob = og.storage(), og.storage()
        og.fill_uniform(oa, 3)
        want = og.sweeps(st.kind, st.coeff, oa, ob, n, theta=st.theta, cond_mode=st.cond_mode)
        assert np.array_equal(got[og.interior], want[og.interior])


@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16"])
def test_interleaved_and_unaligned_fields(gpu, dtype):
    """Fields interleaved in one storage, and fields off the 16-byte
    boundaries of the wide stores (which take single sweeps)."""
    bk = gpu
    st = _stencil(bk, "7pt")
    g = bk.PeriodicGrid((6, 5, 4), ghost=0)
    for offs, step in (((0, 512), 1024), ((1, 520), 1040), ((0, 514), 1029)):
        got = []
        for plan in ("auto", None):
            s = bk.BrickStorage.allocate(g.nbricks, step, DT[dtype])
            s.buf.zero()
            a, b = (bk.Brick(g.info, s, o) for o in offs)
            g.fill_uniform(a, 9)
            bk.sweeps(st, a, b, g, 9, plan=plan)
            bk.device_sync()
            got.append(s.to_host())
        assert np.array_equal(got[0].view(np.uint8), got[1].view(np.uint8))


@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}{c[1] or ''}m{c[2]}")
def test_special_values(gpu, case, dtype):
    """Infinities, NaN, zeros of both signs and denormals spread as by single
    sweeps (a NaN's payload may differ)."""
    bk = gpu
    st = _stencil(bk, *case)
    for nb in ((6, 5, 4), (8, 40, 40)):
        g = bk.PeriodicGrid(nb, ghost=0)
        rng = np.random.default_rng(1)
        if dtype == "bf16":
            x = rng.integers(0, 1 << 16, (g.nbricks, 512)).astype(np.uint16)
            x[rng.random(x.shape) < 0.999] = 0x3e80  # most cells 0.25
        else:
            ft = np.float64 if dtype == "f64" else np.float32
            x = np.full((g.nbricks, 512), 0.25, ft)
            odd = np.array([np.inf, -np.inf, np.nan, -0.0, 0.0, np.finfo(ft).tiny / 8, -1.0], ft)
            at = rng.random(x.shape) < 1e-3
            x[at] = rng.choice(odd, int(at.sum()))
        got = []
        for plan in ("auto", None):
            a = bk.Brick(g.info, bk.movBrickStorage(x, DT[dtype]), 0)
            b = bk.Brick(g.info, g.field_storage(DT[dtype]), 0)
            r = bk.sweeps(st, a, b, g, 4, plan=plan).storage.to_host()
            got.append((r.astype(np.uint32) << 16).view(np.float32) if dtype == "bf16" else r)
        u, v = got
        assert np.array_equal(np.isnan(u), np.isnan(v))
        ok = ~np.isnan(u)
        assert np.array_equal(u[ok], v[ok]) and np.array_equal(np.signbit(u[ok]), np.signbit(v[ok]))


def test_single_sweeps_without_the_refresh(gpu):
    """Ghost bricks that nothing refreshes are boundary values: such a
    sequence stays on single sweeps, also after the box was declared."""
    bk = gpu
    st = _stencil(bk, "7pt")
    g = bk.PeriodicGrid((6, 5, 4))
    _run(bk, g, st, 0, 8, "auto")  # declares the box
    _same(g, _run(bk, g, st, 0, 8, "auto", refresh=False),
          _run(bk, g, st, 0, 8, None, refresh=False), whole=True)


def test_box_must_be_periodic(gpu):
    """set_box refuses ids in another order, pairs that leave ghost bricks
    stale or copy the wrong brick, and boxes other than the plan's bricks; the
    plan keeps sweeping."""
    bk = gpu
    g = bk.PeriodicGrid((4, 3, 2))
    plan = bk.Plan(g.info, g.sweep_list, "quad", 1)
    pairs = g.pairs.reshape(-1, 2)
    wrong = pairs.copy()
    wrong[5, 1] = wrong[6, 1]
    swapped = g.interior.copy()
    swapped[[0, 1]] = swapped[[1, 0]]
    for nb, ids, prs in [((4, 3, 2), g.interior, pairs[:-1]), ((4, 3, 2), g.interior, wrong),
                         ((4, 3, 2), swapped, pairs), ((3, 4, 2), g.interior, pairs),
                         ((4, 3, 1), g.interior[:12], pairs),
                         ((4, 3, 2), np.zeros(24, np.uint32), pairs)]:
        with pytest.raises(bk.BrickError) as e:
            plan.set_box(g.info, nb, ids, prs.reshape(-1))
        assert e.value.code == 4
    st = _stencil(bk, "7pt")
    _same(g, _run(bk, g, st, 0, 8, plan), _run(bk, g, st, 0, 8, None))
    plan.set_box(g.info, g.nb, g.interior, g.pairs)
    _same(g, _run(bk, g, st, 0, 8, plan), _run(bk, g, st, 0, 8, None))
    with pytest.raises(bk.BrickError):
        plan.set_box(g.info, g.nb, g.interior, g.pairs)


def test_decomp_grid(gpu):
    from bricklib_amd.decomp import DecompGrid
    bk = gpu
    st = _stencil(bk, "7pt")
    for kw in ({}, {"brick_bytes": 2048}):
        g = DecompGrid((4, 5, 3), **kw)
        _same(g, _run(bk, g, st, 0, 9, "auto"), _run(bk, g, st, 0, 9, None))
