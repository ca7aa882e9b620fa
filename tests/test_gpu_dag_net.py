"""The batched DAG kernels at the sizes where they change path, against the
oracle bit for bit: every layer count's direction split, nets whose tables
exceed LDS, levels wider and narrower than a workgroup's step, nodes with many
parents, slots with many candidates, edges of length 0, 1, 4, 5, 39, 40 and
above (the sampling step changes at 40)."""
import numpy as np
import pytest

import orc
from instantgr_amd import gpu
from instantgr_amd.host import Design

pytestmark = pytest.mark.gpu


def _dag(rng, XY, X, Y, L, n, wide):
    """A random DAG of n nodes: each node steps along x or y from a parent, and
    takes further parents that share its row or column."""
    px, py, depth = [int(rng.integers(X))], [int(rng.integers(Y))], [0]
    layer = [int(rng.integers(L))]
    par, slot, nslots, par_off = [], [], [0], [0, 0]
    steps = [0, 1, 2, 4, 5, 9, 39, 40, 47, 60]
    for k in range(1, n):
        while True:
            p = int(rng.integers(max(0, k - (40 if wide else 3)), k))
            if nslots[p] < 10 or wide:
                break
        x, y, s = px[p], py[p], int(rng.choice(steps)) * int(rng.choice([-1, 1]))
        if rng.random() < 0.5:
            x = min(X - 1, max(0, x + s))
        else:
            y = min(Y - 1, max(0, y + s))
        px.append(x)
        py.append(y)
        layer.append(L if rng.random() < 0.75 else int(rng.integers(L)))
        nslots.append(0)
        parents = [p] + [q for q in range(k) if q != p and (px[q] == x or py[q] == y) and rng.random() < 0.08]
        for q in parents[:20]:
            # an alternative of a slot the parent has, or a slot of its own
            reuse = nslots[q] > 0 and (nslots[q] >= 10 or rng.random() < 0.6)
            sl = int(rng.integers(nslots[q])) if reuse else nslots[q]
            nslots[q] = max(nslots[q], sl + 1)
            par.append(q)
            slot.append(sl)
        depth.append(1 + max(depth[q] for q in parents[:20]))
        par_off.append(len(par))
    node = np.array(layer) * XY + np.array(px) * Y + np.array(py)
    pts = np.unique(np.array(px) * Y + np.array(py))
    return node, np.array(par_off[1:]) - 0, par, slot, nslots, depth, pts


def _dags(rng, X, Y, L, sizes, wide):
    out = {k: [] for k in ("dag_node", "dag_par", "dag_slot", "dag_child_num", "dag_depth", "dag_pt")}
    node_off, par_off, pt_off = [0], [0], [0]
    for n in sizes:
        node, ends, par, slot, cn, depth, pts = _dag(rng, X * Y, X, Y, L, n, wide)
        base = par_off[-1]
        par_off += [base + int(e) for e in ends]
        for k, v in zip(out, (node, par, slot, cn, depth, pts)):
            out[k].extend(int(t) for t in v)
        node_off.append(node_off[-1] + n)
        pt_off.append(pt_off[-1] + len(pts))
    d = {k: np.array(v, np.int32) for k, v in out.items()}
    d.update(dag_node_off=np.array(node_off, np.int64), dag_par_off=np.array(par_off, np.int64),
             dag_pt_off=np.array(pt_off, np.int64))
    return d


@pytest.mark.parametrize("metals,sizes,wide", [
    (3, [1, 2, 17, 64, 65], False), (4, [16, 33, 120], True), (5, [80, 3, 40], True), (6, [50, 200], False),
    (9, [257, 31, 1], True), (10, [1, 2, 15, 16, 17, 33, 128, 300], True), (10, [900, 20, 700], False),
    (13, [100, 600, 9], True)])
def test_synthetic_dags_match_the_oracle(metals, sizes, wide):
    d = Design.custom(layers=metals, xsize=75, ysize=70, nets=40, pin_cap=8, sigma=6.0, seed=metals).build(4)
    r, o = gpu.Router.from_design(d), orc.Oracle.from_design(d)
    for t in (r, o):
        t.set_nets_from_design(d)
    r.pattern_route(d.array("order"), form=gpu.FORM_BATCHED)
    o.pattern_route(d.array("order"))
    rng = np.random.default_rng(100 * metals + len(sizes))
    nets = np.arange(len(sizes), dtype=np.int32)
    for _ in range(2):
        dags = _dags(rng, 75, 70, metals - 1, sizes, wide)
        st = r.dag_pass(nets, dags, form=gpu.FORM_BATCHED)
        assert st["batches"] == orc.dag_pass(o, nets, dags)
        assert np.array_equal(r.demand(), o.demand())
        assert np.array_equal(r.timestamp(), o.timestamp())
        for a, b in zip(r.costs(), o.costs()):
            assert np.array_equal(a, b)
        for i in range(len(sizes)):
            assert np.array_equal(r.route(i), o.route(i)), i
    r.close()
