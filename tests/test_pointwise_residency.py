"""Registers and LDS of the pointwise kernels agree on the workgroups of a CU.

`walkersFor` sizes the grid by LDS: kernels of four k-slices (64 input channels
of fp16, 128 of fp8) and up to three channel tiles have room for two workgroups
of ten waves, which takes at most 96 registers a lane.  Two more, and half the
grid waits for the other half.
"""
import os
import re
import struct
import subprocess

import pytest

import poplibs_amd as pa

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
LIBRARY = os.path.join(os.path.dirname(pa.__file__), "libmxconv.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
VGPRS = 512     # of a SIMD's lane
GRANULE = 8


def code_objects(data):
    """The gfx950 code objects of the library's offload bundles."""
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, name = struct.unpack_from("<QQQ", data, entry)
            triple = data[entry + 24:entry + 24 + name]
            entry += 24 + name
            if triple.endswith(b"gfx950") and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + 1)


def pointwise_kernels(tmp_path):
    """Template arguments and registers of every pointwise kernel."""
    found = {}
    with open(LIBRARY, "rb") as f:
        data = f.read()
    for i, elf in enumerate(code_objects(data)):
        if b"pointwiseKernel" not in elf:
            continue
        path = tmp_path / ("%d.elf" % i)
        path.write_bytes(elf)
        notes = subprocess.run([READELF, "--notes", str(path)], check=True,
                               capture_output=True, text=True).stdout
        for kernel in notes.split("- .agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel).group(1)
            if "pointwiseKernel" not in name:
                continue
            ints = re.findall(r"L[ib](\d+)E", name)
            # (KS, TM, NB, LW, NT, operands, stores), half or float outputs
            key = tuple(map(int, ints)) + ("6__half" in name,)
            vgprs = int(re.search(r"\.vgpr_count:\s+(\d+)", kernel).group(1))
            spills = int(re.search(r"\.vgpr_spill_count:\s+(\d+)",
                                   kernel).group(1))
            found[key] = vgprs, spills
    return found


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_two_workgroups_to_a_cu(tmp_path):
    kernels = {k: v for k, v in pointwise_kernels(tmp_path).items()
               if k[0] == 4 and k[4] <= 3}
    # one to three channel tiles; fp16 with half and float outputs, four kinds
    # of fp8; two ways to store
    assert len(kernels) == 3 * 6 * 2
    for (ks, tm, nb, lw, nt, *rest), (vgprs, spills) in kernels.items():
        waves = 2 * (tm // 16 + lw)
        most = VGPRS // -(-waves // 4) // GRANULE * GRANULE
        assert vgprs <= most and not spills, (ks, nt, rest, vgprs, most)
