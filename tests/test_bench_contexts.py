"""bench.py holds one routing context at a time: a context of the headline
design takes over half of the device memory."""
import argparse
import os
import sys
import time

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


@pytest.mark.parametrize("warmup,steps", [(0, 1), (0, 3), (2, 2)])
def test_one_context_is_open_at_a_time(monkeypatch, warmup, steps):
    state = {"open": 0, "most": 0, "made": 0}

    class StubRouter:
        def __init__(self):
            state["open"] += 1
            state["made"] += 1
            state["most"] = max(state["most"], state["open"])
            self.closed = False

        def close(self):
            state["open"] -= not self.closed
            self.closed = True

        def device_memory(self):
            return 100, 200

        def routes_flat(self):
            assert not self.closed
            return np.array([0, 1]), np.array([1])

        def evaluate(self, design):
            assert not self.closed
            return {"total": 1.0}

        def kernel_times(self):
            return {}

        def kernel_bytes(self):
            return {}

    stats = {"step_s": 0.01, "pattern_batches": 1, "ripped": [], "rrr_batches": [], "tree_s": 0.0, "pattern_s": 0.0,
             "pattern_schedule_s": 0.0, "rrr_dag_build_s": [], "rrr_route_s": [], "rrr_schedule_s": []}
    monkeypatch.setattr(bench, "one_step", lambda *a, **k: (StubRouter(), dict(stats)))
    args = argparse.Namespace(warmup=warmup, steps=steps, no_profile=False, rrr=1, threads=1)
    out = bench.run_form(None, 1, "batched", args, None, 60.0, time.perf_counter())
    assert len(out["step_s"]) == steps and out["warmup"] == warmup
    assert state["made"] == warmup + steps + (warmup == 0) and state["open"] == 0
    assert state["most"] == 1
