"""Both kinds of scheduler rounds and the built-in choice between them give the
plain scheduler's batches: dense and sparse lists on both sides of the choice's
thresholds, odd grids, both footprint modes."""
import numpy as np
import pytest

from instantgr_amd import gpu
from instantgr_amd.host import Design

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("x,y,nets,heavy,mode", [(97, 101, 160000, 0.0, 0), (333, 251, 160000, 0.0, 1),
                                                (61, 67, 2500, 0.0, 0), (120, 90, 1500, 0.03, 1), (40, 31, 3, 0.0, 0)])
def test_kinds_agree(x, y, nets, heavy, mode):
    d = Design.custom(layers=5, xsize=x, ysize=y, nets=nets, pin_cap=8, sigma=2.5, heavy_frac=heavy, heavy_max=200,
                      seed=nets + mode).build(8)
    r = gpu.Router.from_design(d)
    r.set_nets_from_design(d)
    order = d.array("order")
    got = []
    for kind in (0, 1, 2):
        r.set_tuning(sched_kind=kind)
        got.append(r.schedule(order, mode, gpu.FORM_BATCHED))
    if nets <= 5000:
        got.append(r.schedule(order, mode, gpu.FORM_PLAIN))
    for nb, batch in got[1:]:
        assert nb == got[0][0]
        assert np.array_equal(batch, got[0][1])
    r.close()
