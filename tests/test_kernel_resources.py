"""What the compiler gave the step kernels, from the code object in the built library: the plan that the four-lane FP64
kernels keep in registers must not end up in memory per lane, nor a step's state of the gridded FP32 kernels."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from spectrum_amd import engine as E

READELF = "/opt/rocm/llvm/bin/llvm-readelf" if os.path.exists("/opt/rocm/llvm/bin/llvm-readelf") else shutil.which("llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def device_code(lib):
    """The gfx950 code objects of every bundle in the library."""
    at = lib.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", lib, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", lib, pos)
            name = lib[pos + 24:pos + 24 + idlen]
            pos += 24 + idlen
            if b"gfx950" in name and size:
                yield lib[at + off:at + off + size]
        at = lib.find(MAGIC, at + 1)


def scratch(tmp_path):
    """{kernel: bytes of memory per lane}"""
    with open(E.LIB_PATH, "rb") as f:
        lib = f.read()
    out = {}
    for i, code in enumerate(device_code(lib)):
        p = tmp_path / f"code{i}"
        p.write_bytes(code)
        notes = subprocess.run([READELF, "--notes", str(p)], check=True, capture_output=True, text=True).stdout
        for k in notes.split("- .agpr_count:")[1:]:
            out[re.search(r"\.name:\s+(\S+)", k).group(1)] = int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", k).group(1))
    return out


def test_four_lane_kernels_keep_the_plan_in_registers(tmp_path):
    if not READELF or not os.path.exists(E.LIB_PATH):
        pytest.skip("llvm-readelf or the built library missing")
    of = scratch(tmp_path)
    quad = {k: v for k, v in of.items() if re.search(r"(parker_step|parker_grid_step|gc_step)_kernelId\w*Li1EEEv", k)}
    assert len(quad) > 40, sorted(of)[:5]
    # the arguments and results of a called function at most; the plan would take more than a kilobyte
    assert max(quad.values()) <= 64, {k: v for k, v in quad.items() if v > 64}


def test_gridded_fp32_kernels_hold_a_step_in_registers(tmp_path):
    if not READELF or not os.path.exists(E.LIB_PATH):
        pytest.skip("llvm-readelf or the built library missing")
    of = scratch(tmp_path)
    one_lane = {k: v for k, v in of.items() if re.search(r"parker_grid_step_kernelIf\w*Li0EEEv", k)}
    assert len(one_lane) == 6
    for k, v in one_lane.items():
        # what is spilled once around the step loop; the kernels with a source keep four more values per trajectory
        assert v <= (92 if re.search(r"IfLi[01]ELi1E", k) else 16), (k, v)
