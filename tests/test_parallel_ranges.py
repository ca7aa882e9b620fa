"""The host parallel loop with threads and where none can be created
(tests/host/parallel_ranges.cpp): every element once, no abort."""
import os
import subprocess

from instantgr_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


def test_with_and_without_threads(tmp_path):
    exe = str(tmp_path / "parallel_ranges")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I" + os.path.join(build.CSRC, "host"),
                    os.path.join(HERE, "host", "parallel_ranges.cpp"), "-o", exe, "-lpthread"], check=True)
    for args in ([], ["limited"]):
        p = subprocess.run([exe] + args, capture_output=True, text=True, timeout=60)
        assert p.returncode == 0, (args, p.stdout, p.stderr)
