"""The library's host code against a stand-in for the HIP runtime's host
calls (tests/hip_host.cpp; no GPU): what its entry points do on a second
device and where a launch is refused."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def host_runtime(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("hip_host") / "libhip_host.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", so, os.path.join(ROOT, "tests", "hip_host.cpp")],
                   check=True)
    return so


def _run(host_runtime, body):
    """body in a process of its own, where `host` is the stand-in and `lib` the library."""
    head = ("import ctypes, sys\n"
            "host = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)\n"
            "from diablo_amd import channel, configs\n"
            "lib = channel.load_library()\n")
    r = subprocess.run([sys.executable, "-c", head + body, host_runtime], cwd=ROOT, capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("fp32", [0, 1])
def test_fft512_on_a_second_device(host_runtime, fp32):
    # 96 planes: the FP32 column pass's larger tile too
    _run(host_runtime, f"""
buf = ctypes.create_string_buffer(64)
for dev in (0, 1, 0):
    host.host_set_device(dev)
    for call in (lib.dh_fft512_xz_to_fourier_dev, lib.dh_fft512_xz_to_physical_dev):
        rc = call(ctypes.addressof(buf), ctypes.addressof(buf) + (1 << 40), 96, {fp32}, None)
        assert rc == 0, (dev, lib.dh_batched_last_error())
""")
