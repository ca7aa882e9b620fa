"""Large host copies and the route mailbox on the CPU (tests/host/pinned.cpp, the
HIP calls stubbed): what arrives, with pinned memory and without."""
import os
import subprocess

from instantgr_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


def test_with_and_without_pinned_memory(tmp_path):
    objs = []
    for src in (os.path.join(HERE, "host", "pinned.cpp"), os.path.join(build.CSRC, "hip", "staging.hip")):
        objs.append(str(tmp_path / (os.path.basename(src) + ".o")))
        subprocess.run([build.HIPCC, "--offload-arch=" + build.ARCH, "--offload-host-only", "-O1", "-std=c++17", "-fPIE",
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I" + build.INCLUDE,
                        "-I" + os.path.join(build.CSRC, "host"), "-I" + os.path.join(build.CSRC, "hip"),
                        "-c", src, "-o", objs[-1]], check=True, capture_output=True, text=True)
    exe = str(tmp_path / "pinned")
    subprocess.run(["g++"] + objs + ["-o", exe, "-lpthread"], check=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout
