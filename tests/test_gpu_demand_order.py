"""Demand that is not on the half grid (igr_set_demand takes any float): the
fused track update rounds its FP32 sums in the order of the passes, each batch's
commit (wires, then vias) before the next batch's rip-up (wires, then vias).
Against a float32 model of that order, bit for bit."""
import numpy as np
import pytest

from instantgr_amd import gpu
from instantgr_amd.host import Design

pytestmark = pytest.mark.gpu


def _footprint(r, route):
    """Wire edges and ungated via cuts of a route, counts by (layer, x, y)."""
    edges, vias = np.zeros((r.L, r.X, r.Y), int), np.zeros((r.L, r.X, r.Y), int)
    covered = np.zeros((r.L, r.X, r.Y), bool)
    pos = [(int(v) // (r.X * r.Y), int(v) // r.Y % r.X, int(v) % r.Y) for v in route[1:]]
    for (la, xa, ya), (lb, xb, yb) in zip(pos[::2], pos[1::2]):
        if la == lb:
            x0, x1, y0, y1 = min(xa, xb), max(xa, xb), min(ya, yb), max(ya, yb)
            covered[la, x0:x1 + 1, y0:y1 + 1] = True
            if x0 < x1:
                edges[la, x0:x1, y0] += 1
            if y0 < y1:
                edges[la, x0, y0:y1] += 1
        else:
            vias[min(la, lb):max(la, lb), xa, ya] += 1
    vias[covered] = 0
    return edges, vias


def _add_vias(r, dem, vias, sign):
    for l in range(r.L):
        d, v = (dem[l], vias[l]) if (l & 1) ^ r.DIR else (dem[l].T, vias[l].T)   # tracks as rows
        n = v.shape[1]
        share = np.full((2, n), 0.5, np.float32)     # a cut's share of the edge after it, before it
        share[0, 0] = share[1, n - 1] = 1.0
        for e in range(n - 1):
            d[:, e] += np.float32(sign) * (share[0, e] * v[:, e].astype(np.float32))
            d[:, e] += np.float32(sign) * (share[1, e + 1] * v[:, e + 1].astype(np.float32))


def _model(r, dem, old, new, in_order):
    """Two nets, a batch each: rip up a; commit a, rip up b; commit b."""
    (oa, ob), (na, nb) = old, new
    dem = dem.copy()
    for (ce, cv), (re, rv) in (((None, None), oa), (na, ob), (nb, (None, None))):
        steps = [(ce, 1, False), (cv, 1, True), (re, -1, False), (rv, -1, True)]
        if not in_order:
            steps = [steps[k] for k in (0, 2, 1, 3)]
        for what, sign, is_via in steps:
            if what is None:
                continue
            if is_via:
                _add_vias(r, dem, what, sign)
            else:
                dem += np.float32(sign) * what.astype(np.float32)
    return dem


def _chains(r, nets, shared):
    """DAGs that are chains of (layer, x, y) pins, each net's points 'shared'."""
    k = [len(n) for n in nets]
    off = np.concatenate(([0], np.cumsum(k)))
    cat = lambda f: np.concatenate([f(m) for m in k]).astype(np.int32)  # noqa: E731
    return {"dag_node": np.array([l * r.X * r.Y + x * r.Y + y for n in nets for l, x, y in n], np.int32),
            "dag_node_off": off, "dag_par": cat(lambda m: np.arange(m - 1)), "dag_slot": cat(lambda m: np.zeros(m - 1)),
            "dag_par_off": np.concatenate(([0], np.cumsum(cat(lambda m: np.arange(m) > 0)))),
            "dag_child_num": cat(lambda m: np.arange(m) < m - 1), "dag_depth": cat(np.arange),
            "dag_pt_off": np.arange(len(nets) + 1), "dag_pt": np.full(len(nets), shared, np.int32)}


def test_any_float_demand_is_summed_in_pass_order():
    d = Design.custom(layers=6, xsize=40, ysize=37, nets=40, pin_cap=8, sigma=6.0, seed=5).build(4)
    r = gpu.Router.from_design(d)
    assert r.DIR == 1   # layers 0, 2 and 4 run along y
    r.set_nets_from_design(d)
    r.pattern_route(d.array("order"), form=gpu.FORM_BATCHED)
    rng = np.random.default_rng(1)
    # Net 0 runs along x between pins on layers 0 and 4, so one of its via
    # stacks crosses layer 2 where net 1's wires ran along y in the pass before.
    nets, order = np.array([0, 1], np.int32), np.array([1, 0], np.int32)
    told_apart = 0
    for k in range(10):
        # half a track more from here loses a bit of the sum, a track less does not
        start = rng.uniform(1.5, 2.0, (r.L, r.X, r.Y)).astype(np.float32)
        start[[0, 4]] = 30.0   # keeps net 1 on layer 2
        r.set_demand(start.ravel())
        before = [_footprint(r, r.route(int(i))) for i in nets]
        was, now = 8 + (k + 1) % 2, 8 + k % 2
        pins = [[(2, now, 2), (2, now, 14), (2, now + 4, 14), (2, now + 4, 2)], [(0, was, 3 + k), (4, was + 4, 3 + k)]]
        # a batch each; the list's last net has the lowest priority, so the
        # last batch, which is routed first
        dags = _chains(r, pins, 8 * r.Y + 8)
        assert r.dag_pass(order, dags, form=gpu.FORM_BATCHED)["batches"] == 2
        after = [_footprint(r, r.route(int(i))) for i in nets]
        want = _model(r, start, before, after, True)
        assert np.array_equal(r.demand().reshape(want.shape), want), k
        told_apart += not np.array_equal(want, _model(r, start, before, after, False))
    assert told_apart >= 3
    r.close()
