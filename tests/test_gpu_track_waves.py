"""The fused track update on tracks of one to sixteen waves, with commits,
rip-ups, vias at wave boundaries and every cells-per-thread setting, against
the oracle: demand, timestamps, costs and prefix sums bit for bit."""
import numpy as np
import pytest

import orc
from instantgr_amd import gpu
from instantgr_amd.host import Design

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("x,y,track_k", [(20, 257, 0), (300, 23, 4), (513, 18, 4), (1030, 17, 0), (2100, 24, 4),
                                         (16, 4096, 4), (1100, 20, 8), (2050, 19, 16), (24, 5000, 0)])
def test_long_tracks_match_the_oracle(x, y, track_k):
    d = Design.custom(layers=6, xsize=x, ysize=y, nets=x * y // 30, pin_cap=8, sigma=9.0, seed=x + y).build(4)
    r, o = gpu.Router.from_design(d), orc.Oracle.from_design(d)
    if track_k:
        r.set_tuning(track_k=track_k)
    for t in (r, o):
        t.set_nets_from_design(d)
    r.pattern_route(d.array("order"), form=gpu.FORM_BATCHED)
    o.pattern_route(d.array("order"))

    def same():
        assert np.array_equal(r.demand(), o.demand())
        assert np.array_equal(r.timestamp(), o.timestamp())
        for a, b in zip(r.costs(), o.costs()):
            assert np.array_equal(a, b)

    same()
    nets = np.arange(0, r.num_nets, 2, dtype=np.int32)
    for _ in range(2):
        xs, ys = r.congestion_view()
        dags = d.build_dags(nets, xs, ys, 0, 4)
        r.dag_pass(nets, dags, form=gpu.FORM_BATCHED)
        orc.dag_pass(o, nets, dags)
        same()
    r.close()
