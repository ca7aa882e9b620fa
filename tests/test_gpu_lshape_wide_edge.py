"""The row kernel around the batch size where it changes from a net a wave to
four (5120 nets): one batch of every size there, trees of every node count,
against the oracle bit for bit (the larger ones leave the last wave part
empty)."""
import numpy as np
import pytest

import orc
from instantgr_amd import gpu
from instantgr_amd.host import Design
from test_gpu_lshape_rows import _trees

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("metals,n", [(3, 5119), (3, 5121), (7, 5120), (7, 5122), (10, 5120), (10, 5122), (10, 5123), (13, 5121)])
def test_batch_sizes(metals, n):
    X, Y = 60, 50
    d = Design.custom(layers=metals, xsize=X, ysize=Y, nets=10, pin_cap=4, sigma=6.0, seed=metals).build(2)
    rng = np.random.default_rng(1000 * metals + n)
    trees = _trees(rng, X, Y, metals - 1, [1 + int(k) for k in rng.integers(0, 24, n)])
    r, o = gpu.Router.from_design(d), orc.Oracle.from_design(d)
    for t in (r, o):
        t.set_nets(*trees)
    nets = rng.permutation(n).astype(np.int32)
    r.route_batch(nets)
    o.lshape_batch(nets)
    assert np.array_equal(r.demand(), o.demand())
    assert np.array_equal(r.timestamp(), o.timestamp())
    off, data = r.routes_flat()
    for i in range(n):
        assert np.array_equal(data[off[i]:off[i] + data[off[i]]], o.route(i)), i
    r.close()
