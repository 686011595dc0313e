"""The library's host code against a stand-in for the HIP runtime's host
calls (tests/hip_host.cpp; no GPU): what its entry points do on a second
device, with buffers that share memory and where a launch is refused."""
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


@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("n,ahead", [(1, 0), (16, 0), (40, 0), (40, 4096)])
def test_fft512_inverse_into_its_own_input(host_runtime, n, ahead, fp32):
    """phys = four, or `ahead` bytes before it: the column pass (four, -, its
    output) must not write to the input, nor the row pass (its input, phys) to
    planes that a later column pass reads."""
    _run(host_runtime, f"""
n, ahead, real = {n}, {ahead}, {4 if fp32 else 8}
four = 1 << 40
host.host_record(3)
rc = lib.dh_fft512_xz_to_physical_dev(four, four - ahead, n, {fp32}, None)
assert rc == 0, lib.dh_batched_last_error()
log = (ctypes.c_uint64 * 4096)()
k = host.host_recorded(log, 4096)
assert k % 6 == 0 and k > 0
plane_in, plane_out, end = 512 * 257 * 2 * real, 512 * 512 * real, four + n * 512 * 257 * 2 * real
calls = [tuple(log[i:i + 3]) for i in range(0, k, 3)]
cols, rows = calls[0::2], calls[1::2]
for i, ((src, _, mid), (rin, out, _)) in enumerate(zip(cols, rows)):
    p0 = (src - four) // plane_in
    p1 = (cols[i + 1][0] - four) // plane_in if i + 1 < len(cols) else n
    assert rin == mid and out == four - ahead + p0 * plane_out
    assert mid + (p1 - p0) * plane_out <= four - ahead or mid >= end
    assert out + (p1 - p0) * plane_out <= four + p1 * plane_in
assert p1 == n
""")


def test_refused_tables_leave_the_form(host_runtime):
    """dh_set_mixed_precision where the other form's solve tables cannot be made."""
    _run(host_runtime, """
p, gy, ic = configs.CONFIGS["small_case"]()
ch = channel.Channel(p, gy)
for form in (1, 0):
    host.host_refuse_launches(1)
    assert lib.dh_set_mixed_precision(ch.h, form) != 0
    assert lib.dh_mixed_precision(ch.h) == 1 - form, "switched without its tables"
    host.host_refuse_launches(0)
    assert lib.dh_set_mixed_precision(ch.h, form) == 0
    assert lib.dh_mixed_precision(ch.h) == form
""")
