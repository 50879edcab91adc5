"""The host side of the server and of the host-memory calls, compiled with g++ against a fake HIP runtime
(tests/native): what they do when work is slow, shared or repeated, without a GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "ckfft_amd", "csrc")
HIP = os.environ.get("ROCM_PATH", "/opt/rocm")

pytestmark = pytest.mark.skipif(not os.path.exists(os.path.join(HIP, "include", "hip", "hip_runtime.h")),
                                reason="needs the HIP headers")


def run(tmp_path, test, source):
    exe = str(tmp_path / test)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(HIP, "include"),
                    "-I", os.path.join(ROOT, "include"), "-I", CSRC, "-o", exe,
                    os.path.join(ROOT, "tests", "native", test + ".cpp"), os.path.join(CSRC, source), "-pthread"],
                   check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stderr


def test_server_orders_batches_that_share_an_output(tmp_path):
    run(tmp_path, "serve_outputs", "fft_serve.cpp")


def test_host_memory_calls(tmp_path):
    run(tmp_path, "staging_calls", "fft_staging.cpp")
