"""Registers of the step kernels, from the metadata of the built library: a
kernel whose particles stay in the lanes' registers that spills them to
scratch memory loses what it was made for (8 spilled VGPRs cost the FP64
one-step launch of one particle per lane 5 %)."""
import os
import re
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "viennaemc_amd",
                   "libemcgpu.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _kernels(tmp_path):
    """(name, bytes of scratch per lane) of the kernels of every code object"""
    with open(LIB, "rb") as f:
        data = f.read()
    out, at = [], data.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            target = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in target and size:
                elf = tmp_path / "code.o"
                elf.write_bytes(data[at + off:at + off + size])
                notes = subprocess.run([READELF, "--notes", str(elf)], capture_output=True,
                                       text=True, check=True).stdout
                for k in re.split(r"\n\s*- \.", notes):
                    name = re.search(r"\.name:\s+(\S+)", k)
                    scratch = re.search(r"\.private_segment_fixed_size:\s+(\d+)", k)
                    if name and scratch:
                        out.append((name.group(1), int(scratch.group(1))))
        at = data.find(MAGIC, at + 1)
    return out


@pytest.mark.skipif(not (os.path.exists(LIB) and os.path.exists(READELF)),
                    reason="needs the built library and the LLVM tools")
def test_one_particle_per_lane_does_not_spill(tmp_path):
    # k_bulk_*<float | double, 1, ...> and everything that runs k_bulk_lanes
    mine = [k for k in _kernels(tmp_path)
            if re.search(r"k_bulk_(fused|once)I[fd]Li1E|k_bulk_lanesI", k[0])]
    assert len(mine) >= 16
    assert not [k for k in mine if k[1]]
