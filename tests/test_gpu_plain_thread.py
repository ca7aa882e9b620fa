"""The pattern pass of the 500k-net configuration with a thread per net (plain
form, lshape_groups 1) against the row kernel that both forms use otherwise:
routes, demand and timestamps bit for bit, at a size the oracle is too slow
for."""
import numpy as np
import pytest

from instantgr_amd import gpu
from instantgr_amd.host import Design

pytestmark = pytest.mark.gpu


def test_thread_per_net_and_row_kernel_agree():
    d = Design.preset(1).build(16)
    assert d.info.nets == 500000
    out = []
    for form, groups in ((gpu.FORM_PLAIN, 1), (gpu.FORM_PLAIN, 0), (gpu.FORM_BATCHED, 1)):
        r = gpu.Router.from_design(d)
        r.set_nets_from_design(d)
        r.set_tuning(lshape_groups=groups)
        r.pattern_route(d.array("order"), form=form)
        out.append((r.routes_flat(), r.demand(), r.timestamp()))
        r.close()
    for routes, demand, stamp in out[1:]:
        assert gpu.routes_equal(routes, out[0][0])
        assert np.array_equal(demand.view(np.uint32), out[0][1].view(np.uint32))
        assert np.array_equal(stamp, out[0][2])

