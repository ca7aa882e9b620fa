"""The launch order of a DAG batch's nets under dag_order 2: the order of the
net list, the same in every run, at the list lengths where the spans of the list
change; and the routes, which no order changes."""
import numpy as np
import pytest

from instantgr_amd import gpu
from instantgr_amd.host import Design

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def design():
    return Design.custom(layers=6, xsize=90, ysize=80, nets=5000, pin_cap=8, sigma=5.0, seed=31).build(4)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 129, 4095, 4097])
def test_list_order(design, n, tmp_path, monkeypatch):
    nets = design.array("order")[:n]
    routes = {}
    for order in (1, 2):
        path = tmp_path / ("trace%d" % order)
        r = gpu.Router.from_design(design)
        r.set_nets_from_design(design)
        r.pattern_route(design.array("order"), form=gpu.FORM_BATCHED)
        r.set_tuning(dag_order=order)
        dags = design.build_dags(nets, *r.congestion_view(), 0, 4)
        monkeypatch.setenv("IGR_DAG_TRACE", str(path))
        r.dag_pass(nets, dags, form=gpu.FORM_BATCHED)
        monkeypatch.delenv("IGR_DAG_TRACE")
        routes[order] = r.routes_flat()
        r.close()
        lines = path.read_text().splitlines()
        rows = np.array([[int(v) for v in line.split()] for line in lines[2:]])
        assert lines[1].split()[-1] == "unordered" and rows[:, 1].sum() == n
        if order == 2:
            assert not rows[:, -1].any()
    assert gpu.routes_equal(routes[1], routes[2])
