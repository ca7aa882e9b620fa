"""The plain form's kernels that share a net or a node among lanes, against
the oracle bit for bit: pattern batches of at most and of more than 24 nodes a
net, DAG levels and parent counts around a group of lanes, every direction
split of the layers."""
import numpy as np
import pytest

import orc
from instantgr_amd import gpu
from instantgr_amd.host import Design
from test_gpu_dag_net import _dags
from test_gpu_lshape_rows import _trees

pytestmark = pytest.mark.gpu


def _same(r, o, n):
    assert np.array_equal(r.demand(), o.demand())
    assert np.array_equal(r.timestamp(), o.timestamp())
    for i in range(n):
        assert np.array_equal(r.route(i), o.route(i)), i


@pytest.mark.parametrize("metals,largest", [(3, 24), (3, 25), (6, 1), (9, 24), (10, 30), (13, 24)])
def test_pattern_pass(metals, largest):
    X, Y = 37, 42
    d = Design.custom(layers=metals, xsize=X, ysize=Y, nets=10, pin_cap=4, sigma=6.0, seed=metals).build(2)
    rng = np.random.default_rng(metals + largest)
    sizes = [1 + k % largest for k in range(29)] + [largest]
    trees = _trees(rng, X, Y, metals - 1, sizes)
    r, o = gpu.Router.from_design(d), orc.Oracle.from_design(d)
    for t in (r, o):
        t.set_nets(*trees)
    order = rng.permutation(len(sizes)).astype(np.int32)
    st = r.pattern_route(order, form=gpu.FORM_PLAIN)
    assert st["batches"] == o.pattern_route(order)
    _same(r, o, len(sizes))
    r.close()


@pytest.mark.parametrize("metals,sizes,wide", [
    (3, [1, 2, 17, 64, 65], False), (4, [16, 33, 120], True), (6, [50, 200], False),
    (9, [257, 31, 1], True), (10, [1, 2, 15, 16, 17, 33, 128, 300], True), (13, [100, 400, 9], True)])
def test_dag_pass(metals, sizes, wide):
    d = Design.custom(layers=metals, xsize=75, ysize=70, nets=40, pin_cap=8, sigma=6.0, seed=metals).build(4)
    r, o = gpu.Router.from_design(d), orc.Oracle.from_design(d)
    for t in (r, o):
        t.set_nets_from_design(d)
    r.pattern_route(d.array("order"), form=gpu.FORM_PLAIN)
    o.pattern_route(d.array("order"))
    rng = np.random.default_rng(50 * metals + len(sizes))
    nets = np.arange(len(sizes), dtype=np.int32)
    for _ in range(2):
        dags = _dags(rng, 75, 70, metals - 1, sizes, wide)
        st = r.dag_pass(nets, dags, form=gpu.FORM_PLAIN)
        assert st["batches"] == orc.dag_pass(o, nets, dags)
        _same(r, o, len(sizes))
    r.close()
