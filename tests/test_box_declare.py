"""The declaration ahead of a sequence of sweeps: what each status of the
library makes of it (host logic, no device)."""
import sys
import threading
from types import SimpleNamespace

import numpy as np
import pytest

from bricklib_amd import _lib
from bricklib_amd.bricks import Plan, PeriodicGrid


class FakePlan:
    """A Plan whose library calls end with the given statuses in turn."""

    def __init__(self, *codes):
        self.shape, self.boxed, self.handle = "quad", False, None
        self.lock, self.tables = threading.Lock(), set()
        self.codes, self.calls = list(codes), 0

    def _end(self):
        self.calls += 1
        code = self.codes.pop(0) if self.codes else 0
        if code:
            raise _lib.BrickError(code, "planted")

    def set_box(self, *args, **kw):
        self._end()
        self.boxed = True

    def bind_box(self, *args, **kw):
        self._end()


def _grid(plan):
    g = PeriodicGrid.__new__(PeriodicGrid)
    g.info, g.d_pairs = SimpleNamespace(dev=SimpleNamespace(ptr=4096)), None
    g.pairs = np.empty(0, np.uint32)
    g.interior, g.nb, g._plans = np.arange(8, dtype=np.uint32), (2, 2, 2), {"p": plan}
    return g


def test_declared_once():
    p = FakePlan()
    g = _grid(p)
    for _ in range(3):
        g._declare_box(p)
    assert p.boxed and p.calls == 2


@pytest.mark.parametrize("at", [0, 1])
def test_not_a_box_is_remembered(at):
    p = FakePlan(*[0] * at, _lib.BK_ERR_UNSUPPORTED)
    g = _grid(p)
    for _ in range(3):
        g._declare_box(p)
    assert p.calls == at + 1


@pytest.mark.parametrize("at", [0, 1])
def test_out_of_memory_is_tried_again(at):
    p = FakePlan(*[0] * at, _lib.BK_ERR_NOMEM)
    g = _grid(p)
    g._declare_box(p)  # the sequence goes on by single sweeps
    assert p.boxed == bool(at)
    g._declare_box(p)
    assert p.boxed and p.calls == 3
    g._declare_box(p)
    assert p.calls == 3


@pytest.mark.parametrize("code", [_lib.BK_ERR_HIP, _lib.BK_ERR_ARG])
def test_other_errors_are_raised(code):
    p = FakePlan(code)
    with pytest.raises(_lib.BrickError) as e:
        _grid(p)._declare_box(p)
    assert e.value.code == code


def test_while_another_thread_adds_plans():
    """grid.plan() of another thread grows the table that is searched."""
    p = FakePlan()
    g = _grid(p)
    g._plans = {("other", q): object() for q in range(500)}
    stop, errors = threading.Event(), []

    def add():
        q = 0
        while not stop.is_set():
            g._plans[("more", q % 4000)] = object()
            q += 1
            if q % 4000 == 0:
                for r in range(4000):
                    del g._plans[("more", r)]

    was = sys.getswitchinterval()
    sys.setswitchinterval(1e-6)
    t = threading.Thread(target=add)
    t.start()
    try:
        for _ in range(300):
            try:
                g._declare_box(p)
            except RuntimeError as e:
                errors.append(e)
    finally:
        stop.set()
        t.join()
        sys.setswitchinterval(was)
    assert not errors and p.calls == 0


def test_plan_has_what_the_declaration_uses():
    assert {"set_box", "bind_box", "unbind_box"} <= set(dir(Plan))


@pytest.mark.parametrize("name", ["7pt", "25pt"])
@pytest.mark.parametrize("ghosts,refresh,n,want", [
    (True, False, 9, False),  # ghost bricks as boundary values: no periodic box
    (True, True, 9, True), (True, True, 3, False), (False, True, 9, None), (False, False, 9, None)])
def test_which_sequences_declare(monkeypatch, name, ghosts, refresh, n, want):
    """Only sequences that may use the box pay for its declaration."""
    from bricklib_amd import bricks
    from bricklib_amd.stencils import Stencil
    p = FakePlan()
    g = _grid(p)
    asked = []
    g._declare_box = lambda *a, **k: asked.append(a)
    if ghosts:
        g.d_pairs, g.pairs = SimpleNamespace(ptr=8192), np.zeros(2, np.uint32)
    monkeypatch.setattr(bricks, "_desc", lambda *a, **k: a[4].append(p) or _lib.bk_sweep_desc())
    monkeypatch.setattr(bricks, "load", lambda: SimpleNamespace(bk_sweeps=lambda *a: 0))
    f = SimpleNamespace(dtype=0)
    bricks.sweeps(Stencil.make(name, seed=1), f, f, g, n, refresh=refresh)
    # a wrapped box has nothing to refresh: only what takes several sweeps per pass
    assert bool(asked) == (name == "7pt" if want is None else want)
