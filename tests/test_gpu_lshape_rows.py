"""The batched pattern DP on synthetic trees against the oracle, bit for bit:
every routing-layer count, trees of 1 to 24 nodes (the row kernel's range) and
above (the thread-per-net kernel), chains and stars, straight, L-shaped and
zero-length edges, net counts that leave the last wave part empty."""
import numpy as np
import pytest

import orc
from instantgr_amd import gpu
from instantgr_amd.host import Design

pytestmark = pytest.mark.gpu


def _trees(rng, X, Y, L, sizes):
    node_off, node, parent, pt_off, pt = [0], [], [], [0], []
    for n in sizes:
        shape = int(rng.integers(3))
        xs, ys = [], []
        for k in range(n):
            p = -1 if k == 0 else 0 if shape == 0 else k - 1 if shape == 1 else int(rng.integers(k))
            if k and rng.random() < 0.5:   # straight, or on its parent
                x, y = xs[p], ys[p]
                if rng.random() < 0.5:
                    x = int(np.clip(x + rng.integers(-6, 7), 0, X - 1))
                else:
                    y = int(np.clip(y + rng.integers(-6, 7), 0, Y - 1))
            else:
                x, y = int(rng.integers(X)), int(rng.integers(Y))
            xs.append(x)
            ys.append(y)
            l = L if rng.random() < 0.4 else int(rng.integers(min(2, L)))
            node.append(l * X * Y + x * Y + y)
            parent.append(p)
        node_off.append(len(node))
        pt.extend(np.unique(np.array(xs) * Y + np.array(ys)))
        pt_off.append(len(pt))
    return node_off, node, parent, pt_off, pt


@pytest.mark.parametrize("metals", [3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13])
def test_synthetic_trees_match_the_oracle(metals):
    X, Y = 37, 42
    d = Design.custom(layers=metals, xsize=X, ysize=Y, nets=10, pin_cap=4, sigma=6.0, seed=metals).build(2)
    rng = np.random.default_rng(metals)
    sizes = list(range(1, 25)) + [24, 30, 2, 1, 23, 17, 26, 3, 3][:5 + metals % 5]
    trees = _trees(rng, X, Y, metals - 1, sizes)
    r, o = gpu.Router.from_design(d), orc.Oracle.from_design(d)
    demand = rng.integers(0, 12, r.n).astype(np.float32) / 2
    for t in (r, o):
        t.set_demand(demand)
        t.set_nets(*trees)
    order = rng.permutation(len(sizes)).astype(np.int32)
    st = r.pattern_route(order, form=gpu.FORM_BATCHED)
    assert st["batches"] == o.pattern_route(order)
    assert np.array_equal(r.demand(), o.demand())
    assert np.array_equal(r.timestamp(), o.timestamp())
    for i in range(len(sizes)):
        assert np.array_equal(r.route(i), o.route(i)), (i, sizes[i])
    r.close()
