"""Route buffers of rip-up-and-reroute passes on the CPU (tests/host/pass_routes.cpp,
the HIP calls stubbed): a pass that fails after its kernels ran leaves no device
pointer into memory that later passes free or reuse."""
import os
import subprocess

from instantgr_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


def test_pass_routes_buffers(tmp_path):
    exe = str(tmp_path / "pass_routes")
    obj = exe + ".o"
    subprocess.run([build.HIPCC, "--offload-arch=" + build.ARCH, "--offload-host-only", "-O1", "-std=c++17", "-fPIE",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "-I" + build.INCLUDE, "-I" + os.path.join(build.CSRC, "host"), "-I" + os.path.join(build.CSRC, "hip"),
                    "-c", os.path.join(HERE, "host", "pass_routes.cpp"), "-o", obj], check=True,
                   capture_output=True, text=True)
    subprocess.run(["g++", obj, "-o", exe, "-lpthread"], check=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout
