"""The cube a wave a brick, alone and as the form that plans of 4- and 2-byte
types take from 1201 bricks on: one brick an axis, odd counts, last workgroups
that are not full, both sides of that line -- bit for bit the oracle's sweep."""
import numpy as np
import pytest

import oracle as O
from bricklib_amd import BK_BF16, BK_F32, BK_F64
from bricklib_amd import stencils as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [BK_F64, BK_F32, BK_BF16])
@pytest.mark.parametrize("nb", [(1, 1, 1), (1, 3, 2), (5, 3, 7), (10, 12, 10), (11, 10, 11)])
def test_matches_oracle(gpu, nb, dtype):
    st = S.Stencil.make("125pt", seed=12)
    og = O.Grid(nb)
    oa, ob = og.storage(dtype), og.storage(dtype)
    og.fill_uniform(oa, 5, dtype=dtype)
    want = og.sweeps(st.kind, st.coeff, oa, ob, 1, dtype=dtype)[og.interior]
    for ghost in (1, 0):
        g = gpu.PeriodicGrid(nb, ghost=ghost)
        a, b = (gpu.Brick(g.info, g.field_storage(dtype), 0) for _ in range(2))
        g.fill_uniform(a, 5)
        for plan in (None, "auto", g.plan("quad", 3)):
            b.storage.buf.zero()
            got = gpu.sweeps(st, a, b, g, 1, plan=plan).storage.to_host()[g.interior]
            np.testing.assert_array_equal(got, want)
