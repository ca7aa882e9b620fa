"""The built-in choice of scheduler rounds on both sides of its lines (175k nets,
lists of 28): the default gives the batches of either kind, whichever it takes."""
import numpy as np
import pytest

from instantgr_amd import gpu
from instantgr_amd.host import Design

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("x,y,nets,above", [(173, 175, 170000, False), (173, 175, 176000, True), (275, 273, 176000, False)])
def test_default_agrees_with_both_kinds(x, y, nets, above):
    d = Design.custom(layers=5, xsize=x, ysize=y, nets=nets, pin_cap=8, sigma=2.5, seed=nets).build(8)
    r = gpu.Router.from_design(d)
    r.set_nets_from_design(d)
    order = d.array("order")
    lists = d.array("pt_off")[-1] / (x * y)
    assert (len(order) >= 175000 and lists >= 28) == above
    got = []
    for kind in (0, 1, 2):
        r.set_tuning(sched_kind=kind)
        got.append(r.schedule(order, 0, gpu.FORM_BATCHED))
    for nb, batch in got[1:]:
        assert nb == got[0][0]
        assert np.array_equal(batch, got[0][1])
    r.close()
