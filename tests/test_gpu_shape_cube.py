"""The 125-point cube on 4x8x16 bricks at the edges of its lane and box layout:
one brick an axis (every neighbour the brick itself), odd counts, a last
workgroup that is not full -- bit for bit the oracle's sweep over the same
layout."""
import numpy as np
import pytest

import oracle as O
from bricklib_amd import BK_BF16, BK_F32, BK_F64
from bricklib_amd import stencils as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", [1, 2], ids=["4x8x16", "4x8x16f88"])
@pytest.mark.parametrize("dtype", [BK_F64, BK_F32, BK_BF16])
@pytest.mark.parametrize("nb", [(1, 1, 1), (1, 3, 2), (2, 1, 5), (3, 5, 7)])
def test_matches_oracle(gpu, nb, dtype, layout):
    st = S.Stencil.make("125pt", seed=12)
    for ghost in (1, 0):
        lg = O.LayoutGrid(nb, layout, ghost)
        oa, ob = lg.storage(dtype), lg.storage(dtype)
        lg.fill_uniform(oa, 5, dtype=dtype)
        want = lg.sweeps(st.kind, st.coeff, oa, ob, 2, dtype=dtype, refresh=bool(ghost))
        g = gpu.PeriodicGrid(nb, ghost=ghost, layout=layout)
        a, b = (gpu.Brick(g.info, g.field_storage(dtype), 0) for _ in range(2))
        g.fill_uniform(a, 5)
        for wg in (1, 2, 4):
            g.fill_uniform(a, 5)
            res = gpu.sweeps(st, a, b, g, 2, wg_bricks=wg, plan=None)
            got = res.storage.to_host()
            np.testing.assert_array_equal(got[lg.interior], want[lg.interior])
