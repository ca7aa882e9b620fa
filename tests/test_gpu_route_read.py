"""Single route reads at the lengths where they change path (a workgroup's
width, the mailbox's size), against the bulk read of all routes and from
several threads at once."""
import threading

import numpy as np
import pytest

from instantgr_amd import gpu
from instantgr_amd.host import Design
from test_gpu_dag_net import _dags

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[1, 2, 16, 31, 32, 33, 64, 400], [2046, 2047, 2048, 2100]])
def test_single_reads_match_the_bulk_read(sizes):
    d = Design.custom(layers=6, xsize=75, ysize=70, nets=40, pin_cap=8, sigma=6.0, seed=3).build(4)
    r = gpu.Router.from_design(d)
    r.set_nets_from_design(d)
    r.pattern_route(d.array("order"), form=gpu.FORM_BATCHED)
    nets = np.arange(len(sizes), dtype=np.int32)
    r.dag_pass(nets, _dags(np.random.default_rng(7), 75, 70, 5, sizes, False), form=gpu.FORM_BATCHED)
    off, data = r.routes_flat()
    want = [data[off[i]:off[i] + data[off[i]]] for i in range(r.num_nets)]
    bad = []

    def read():
        for i in range(r.num_nets):
            if not np.array_equal(r.route(i), want[i]):
                bad.append(i)

    threads = [threading.Thread(target=read) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    # a buffer shorter than the route: its head, and the whole length
    buf, ln = np.full(8, -7, np.int32), gpu.C.c_int()
    i = len(sizes) - 1
    assert gpu.lib().igr_get_route(r.h, i, buf.ctypes.data, 3, gpu.C.byref(ln)) == 0
    assert ln.value == len(want[i]) and np.array_equal(buf[:3], want[i][:3]) and (buf[3:] == -7).all()
    r.close()
