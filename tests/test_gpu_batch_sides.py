"""A captured batched run lets its groups go side by side where their requests
share no field, and keeps the order of ticks where they do: either way each
field holds, bit for bit, what the launches of an eager run leave there."""
import pytest

from bricklib_amd import BK_BF16, BK_F32, BK_F64
from bricklib_amd.batch import Batch, Request, ShapeCache
from bricklib_amd.stencils import Stencil

pytestmark = pytest.mark.gpu

MIX = [((2, 3, 4), "7pt", BK_F64, 25), ((19, 17, 6), "125pt", BK_F64, 37), ((3, 2, 2), "13pt", BK_F32, 36),
       ((12, 2, 5), "25pt", BK_F64, 2), ((5, 3, 1), "cond", BK_F64, 4), ((2, 4, 2), "125pt", BK_F32, 38),
       ((1, 1, 1), "7pt", BK_BF16, 38), ((4, 2, 3), "25pt", BK_F32, 1)]


def requests(mix, ghost):
    shapes, reqs = ShapeCache(), []
    for q, (nb, name, dt, steps) in enumerate(mix):
        reqs.append(Request(rid=q, nb=nb, stencil=Stencil.make(name, seed=q), dtype=dt,
                            steps=steps, seed=q, ghost=ghost))
        reqs[-1].allocate(shapes)
    return reqs


def fields(reqs):
    """The interiors of both fields of every request."""
    out = []
    for r in reqs:
        for parity in (0, 1):
            r.parity = parity
            out.append(r.result_host()[r.interior_index()].tobytes())
    return out


@pytest.mark.parametrize("ghost", [0, 1])
@pytest.mark.parametrize("groups", [1, 4, 5, 6, 8])
def test_graph_leaves_what_eager_does(gpu, ghost, groups):
    got = []
    for use_graph in (False, True):
        reqs = requests(MIX[:groups], ghost)
        batch = Batch(max_reqs=8)
        for ticks in (3, 16, 3, 16):  # in turn and side by side; each replayed
            batch.run(reqs, ticks, use_graph=use_graph)
        got.append(fields(reqs))
    assert got[0] == got[1]


@pytest.mark.parametrize("rep", range(4))
def test_shared_field_keeps_the_order(gpu, rep):
    """A one-sweep request reads the field that a longer one of another group
    overwrites in its second tick."""
    got = []
    for use_graph in (False, True):
        reqs = requests([((32, 32, 16), "125pt", BK_F64, 1), ((32, 32, 16), "7pt", BK_F64, 6)]
                        + MIX[2:], 0)
        reqs[0].f0 = reqs[1].f0
        reqs[0]._rec = bytes(reqs[0].req_struct(0))
        batch = Batch(max_reqs=8)
        batch.run(reqs, 6, use_graph=use_graph)
        got.append(fields(reqs))
    assert got[0] == got[1]
