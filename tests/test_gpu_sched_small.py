"""The one-workgroup scheduler rounds, at the list lengths and point counts
where they start, stop and do not fit, against the plain form and the other
kinds of rounds: the same batches for the same order, in all three modes."""
import numpy as np
import pytest

from instantgr_amd import gpu
from instantgr_amd.host import Design

pytestmark = pytest.mark.gpu


def _check(d, lengths, modes=(0, 1, 2)):
    r = gpu.Router.from_design(d)
    r.set_nets_from_design(d)
    order = d.array("order")
    for n in lengths:
        sub = order[-n:].copy()
        for mode in modes:
            r.set_tuning()
            want = r.schedule(sub, mode, gpu.FORM_PLAIN)
            got = r.schedule(sub, mode, gpu.FORM_BATCHED)
            assert got[0] == want[0] and np.array_equal(got[1], want[1]), (n, mode)
            for kind in (1, 2):
                r.set_tuning(sched_kind=kind)
                got = r.schedule(sub, mode, gpu.FORM_BATCHED)
                assert got[0] == want[0] and np.array_equal(got[1], want[1]), (n, mode, kind)
    r.close()


def test_list_lengths():
    d = Design.custom(layers=6, xsize=60, ysize=50, nets=2600, pin_cap=6, sigma=4.0, seed=5).build(4)
    _check(d, [1, 2, 15, 16, 17, 63, 65, 256, 257, 1023, 1025, 2047, 2048, 2049, len(d.array("order"))])


def test_dense_conflicts():
    # every net meets most others: as many batches as the order allows
    d = Design.custom(layers=4, xsize=12, ysize=11, nets=900, pin_cap=5, sigma=6.0, seed=8).build(4)
    _check(d, [33, 700], modes=(0, 1))


def test_nets_that_do_not_fit():
    # large nets: the points of the list exceed the limits although the nets
    # do not, so the rounds stop early and go on; and a tail that fits later
    d = Design.custom(layers=9, xsize=300, ysize=290, nets=1800, pin_cap=64, heavy_frac=0.9, hotspots=6,
                      hotspot_scale=0.7, seed=9).build(4)
    _check(d, [100, 1500, min(2048, len(d.array("order"))), len(d.array("order"))], modes=(0, 2))
