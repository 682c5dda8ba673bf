"""Registers and scratch of built kernels (CPU only): the code objects in the
library state them in their metadata notes."""
import os
import re
import struct
import subprocess

import pytest

from conftest import PKG

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def _kernels(tmp_path):
    """Kernel name -> (VGPRs, scratch bytes, threads a block may have) of every
    device code object."""
    with open(os.path.join(PKG, "libsplatt.so"), "rb") as f:
        data = f.read()
    found = {}
    at = data.find(b"\x7fELF", 4)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == 224:      # EM_AMDGPU
            obj = tmp_path / ("%d.o" % at)
            obj.write_bytes(data[at:])
            notes = subprocess.run([READELF, "--notes", str(obj)], capture_output=True,
                                   text=True).stdout
            for k in re.split(r"\n\s+- \.a", notes)[1:]:
                def field(name):
                    m = re.search(r"\.%s:\s*(\S+)" % name, k)
                    return m.group(1) if m else None
                if field("name") and field("vgpr_count"):
                    found[field("name")] = (int(field("vgpr_count")),
                                            int(field("private_segment_fixed_size")),
                                            int(field("max_flat_workgroup_size")))
        at = data.find(b"\x7fELF", at + 4)
    return found


pytestmark = pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")


def test_norm_kernels_take_the_blocks_they_are_launched_with(tmp_path):
    # the norm of the model is summed by 256 threads, alone and batched
    seen = 0
    for name, (_, _, threads) in _kernels(tmp_path).items():
        if re.match(r"_Z\d+kb?_cpd_norm", name):
            seen += 1
            assert threads >= 256, name
    assert seen == 2


def test_fp32_walks_keep_their_registers(tmp_path):
    # root (0) and row-copy (4) walks of FP32 with 16-byte lanes over chunks
    # of 64 and 256 nonzeros: four waves per SIMD (512 / 4 VGPRs) without
    # scratch in four modes, five in three
    seen = 0
    for name, (vgprs, scratch, _) in _kernels(tmp_path).items():
        m = re.match(r"_Z7k_walksIfLi([34])ELi[04]ELi4E", name)
        if m:
            seen += 1
            assert scratch == 0, name
            assert vgprs <= (96 if m.group(1) == "3" else 128), name
    assert seen == 2 * 2 * 4 * 2
