"""Registers of the nonlinear pass's large-block kernels in the built library
(no GPU): each fits its 256 registers per lane without spills or scratch.
They lie at the edge, so a transform routine that the compiler no longer
inlines into them shows here first."""
import os
import re
import struct
import subprocess

import pytest

from diablo_amd import build, channel

LLVM = os.path.join(os.path.dirname(os.path.dirname(build.HIPCC)), "llvm", "bin")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


@pytest.fixture(scope="module")
def resources(tmp_path_factory):
    """Kernel (mangled) -> (spilled registers, scratch bytes) of the library's gfx950 code."""
    tmp = tmp_path_factory.mktemp("fatbin")
    fat = str(tmp / "fatbin")
    subprocess.run([os.path.join(LLVM, "llvm-objcopy"), f"--dump-section=.hip_fatbin={fat}", channel.LIB_PATH,
                    os.devnull], check=True)
    data = open(fat, "rb").read()
    out = {}
    for base in (m.start() for m in re.finditer(MAGIC, data)):
        n, = struct.unpack_from("<Q", data, base + len(MAGIC))
        at = base + len(MAGIC) + 8
        for _ in range(n):
            off, size, ln = struct.unpack_from("<QQQ", data, at)
            triple = data[at + 24: at + 24 + ln]
            at += 24 + ln
            if b"gfx950" not in triple or size == 0:
                continue
            co = str(tmp / "co")
            open(co, "wb").write(data[base + off: base + off + size])
            notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", co], check=True,
                                   capture_output=True, text=True).stdout
            for k in re.split(r"\n  - (?=\.)", notes)[1:]:
                f = dict(re.findall(r"^\s*(\.\w+):\s+(\S+)$", k, re.M))
                if ".vgpr_spill_count" in f:
                    out[f[".symbol"]] = (int(f[".vgpr_spill_count"]), int(f[".private_segment_fixed_size"]))
    return out


# k_nonlinear<REG, modes per thread, LES, block bound>: the x rows of NX = 128 in
# registers, and blocks of at most 512 threads
@pytest.mark.parametrize("kernel", ["k_nonlinearILb1ELi8ELb0ELi512E", "k_nonlinearILb0ELi4ELb0ELi512E",
                                    "k_nonlinearILb0ELi4ELb1ELi512E"])
def test_no_spills(resources, kernel):
    hits = {k: v for k, v in resources.items() if kernel in k}
    assert len(hits) == 1, sorted(resources)
    assert set(hits.values()) == {(0, 0)}, hits
