"""The device routing order (counting sort by batch and size, the per-net
bases) at the list lengths where its scans change workgroup or leave a
remainder, against the oracle bit for bit; and the checks of the DAG arrays
that moved to the device with it."""
import numpy as np
import pytest

import orc
from instantgr_amd import gpu
from instantgr_amd.host import Design

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def design():
    return Design.custom(layers=6, xsize=90, ysize=80, nets=2500, pin_cap=8, sigma=5.0, seed=31).build(4)


@pytest.mark.parametrize("n", [1, 255, 257, 2047, 2048, 2049])
def test_list_lengths_match_the_oracle(design, n):
    r, o = gpu.Router.from_design(design), orc.Oracle.from_design(design)
    order = design.array("order")
    for t in (r, o):
        t.set_nets_from_design(design)
    r.pattern_route(order[:n], form=gpu.FORM_BATCHED)
    o.pattern_route(order[:n])
    r.pattern_route(order[n:], form=gpu.FORM_BATCHED)
    o.pattern_route(order[n:])
    for _ in range(2):
        xs, ys = r.congestion_view()
        dags = design.build_dags(order[:n], xs, ys, 0, 4)
        st = r.dag_pass(order[:n], dags, form=gpu.FORM_BATCHED)
        assert st["batches"] == orc.dag_pass(o, order[:n], dags)
        assert np.array_equal(r.demand(), o.demand())
    for i in order[:: max(1, n // 50)]:
        assert np.array_equal(r.route(int(i)), o.route(int(i))), i
    r.close()


@pytest.mark.parametrize("key,at,value", [
    ("dag_par_off", 5, lambda a: a[6] + 1), ("dag_par_off", 3, lambda a: -1), ("dag_depth", 4, lambda a: 1 << 20),
    ("dag_depth", 0, lambda a: -1), ("dag_child_num", 7, lambda a: 11), ("dag_child_num", -1, lambda a: -1),
    ("dag_node_off", 1, lambda a: 0)])
def test_bad_dags_are_refused_and_change_nothing(design, key, at, value):
    r = gpu.Router.from_design(design)
    r.set_nets_from_design(design)
    nets = design.array("order")[:60]
    r.pattern_route(design.array("order"), form=gpu.FORM_BATCHED)
    xs, ys = r.congestion_view()
    dags = design.build_dags(nets, xs, ys, 0, 4)
    before = r.demand()
    bad = dict(dags)
    bad[key] = dags[key].copy()
    bad[key][at] = value(bad[key])
    with pytest.raises(RuntimeError, match="malformed DAG|empty DAG"):
        r.dag_pass(nets, bad, form=gpu.FORM_BATCHED)
    assert np.array_equal(r.demand(), before)
    r.dag_pass(nets, dags, form=gpu.FORM_BATCHED)
    r.close()
