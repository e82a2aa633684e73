"""First sequences over one grid from several threads at once: the box is
declared under way by one of them, and every thread gets the same bits."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rep", range(3))
def test_first_sequences_of_four_threads(gpu, rep):
    bk = gpu
    st = bk.Stencil.make("7pt", seed=3)
    g = bk.PeriodicGrid((9, 6, 7))
    fields = [[bk.Brick(g.info, g.field_storage(0), 0) for _ in range(2)] for _ in range(5)]
    streams = [bk.Stream() for _ in range(4)]
    for a, _ in fields:
        g.fill_uniform(a, 4)
    bk.sweep(st, fields[4][1], fields[4][0], g)  # builds the plan
    bk.device_sync()
    start = threading.Barrier(4)

    def work(q):
        start.wait()
        bk.sweeps(st, *fields[q], g, 9, stream=streams[q])

    threads = [threading.Thread(target=work, args=(q,)) for q in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    bk.device_sync()
    bk.sweeps(st, *fields[4], g, 9, plan=None)
    bk.device_sync()
    got = [np.ascontiguousarray(b.storage.to_host()[g.interior]).view(np.uint8)
           for _, b in fields]
    for x in got[:4]:
        assert np.array_equal(x, got[4])
