"""What orders the library's launches on several streams and threads, on the CPU:
the host library linked to a HIP runtime that records calls instead of running
them (tests/native/hip_recorder.h, stream_order_check.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
CHECKS = ["fft_per_thread"]

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not os.path.exists(os.path.join(ROCM, "include", "hip")),
                                reason="needs g++ and the HIP headers")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = tmp_path_factory.mktemp("order") / "stream_order_check"
    csrc = os.path.join(ROOT, "convfpga_amd", "csrc")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-fopenmp", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I" + os.path.join(ROCM, "include"), "-I" + os.path.join(ROOT, "include"), "-I" + csrc,
                    os.path.join(ROOT, "tests", "native", "stream_order_check.cpp"),
                    os.path.join(csrc, "engine.cpp"), os.path.join(csrc, "capi.cpp"), "-o", str(exe)], check=True)
    return str(exe)


@pytest.mark.parametrize("name", CHECKS)
def test_stream_order(check, name):
    r = subprocess.run([check, name], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.endswith("ok %s\n" % name), r.stdout
