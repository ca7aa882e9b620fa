"""Grid arrays in and out at the sizes where the staged copies change path
(smaller than a slot, whole and ragged slots, more slots than there are), and
from several threads at once."""
import threading

import numpy as np
import pytest

from instantgr_amd import gpu

pytestmark = pytest.mark.gpu


def _router(X, Y):
    cap = np.full(X * Y, 5.0, np.float32)
    return gpu.Router(1, X, Y, 0, 1.0, 4.0, np.ones(1), np.ones(X - 1, np.int32), np.ones(Y - 1, np.int32), cap)


# X * Y floats: 1 MiB (the smallest staged copy), 2 MiB (a slot), 16 MiB (all
# slots), each with a neighbour on both sides where one exists
@pytest.mark.parametrize("X,Y", [(511, 513), (512, 512), (545, 481), (1024, 512), (1030, 509), (2047, 2049),
                                 (2048, 2048), (1985, 2113), (2300, 3111)])
def test_demand_round_trip(X, Y):
    r = _router(X, Y)
    rng = np.random.default_rng(X)
    for _ in range(2):
        d = rng.integers(0, 1 << 20, X * Y).astype(np.float32)
        r.set_demand(d)
        assert np.array_equal(r.demand(), d)
    r.close()


def test_reads_from_several_threads():
    r = _router(1400, 1500)
    d = np.arange(1400 * 1500, dtype=np.float32)
    r.set_demand(d)
    r.update_cost()
    ts, bad = r.timestamp(), []

    def read():
        for _ in range(5):
            if not np.array_equal(r.demand(), d) or not np.array_equal(r.timestamp(), ts):
                bad.append(1)

    threads = [threading.Thread(target=read) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    r.close()
