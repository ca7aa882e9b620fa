"""The kernel symbols bench.py's roofline names: every one is a kernel of the
HIP sources, and the pattern DP's is the one the committed traffic summary
measured."""
import glob
import os
import re
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


def test_symbols_are_kernels():
    text = "".join(open(p).read() for p in glob.glob(os.path.join(ROOT, "instantgr_amd", "csrc", "hip", "*.hip")))
    kernels = set(re.findall(r"__global__[^;{]*?\b(k_\w+)\s*\(", text))
    assert set(bench.KERNEL_SYMBOL.values()) <= kernels


def test_the_pattern_dp_is_priced_with_its_measured_traffic():
    want = bench._traffic("k_lshape_wave", 1)[0]
    assert want and want > 0
    r = bench.roofline({"lshape_dp": (4.0, 56)}, {"lshape_dp": 4.0e8}, 1)
    assert r["symbol"] == "k_lshape_wave" and r["traffic"] == pytest.approx(want)
