"""Registers of the transform kernels in the built library (CPU).

A workgroup of the longest transforms takes 67,584 bytes of LDS, so that two share a
compute unit if their registers allow it: with 32-bit words both radices leave four
waves per SIMD (128 registers), with 64-bit ones radix 16 does and radix 32 two (256).
Past 128 registers the radix-32 kernels of 32-bit words run one workgroup at a time (8
products of 32 x 32 x 32, length 6000: 1.77 ms against 1.61)."""
import os
import re
import struct
import subprocess

import pytest

from pml_amd import build

LLVM = "/opt/rocm/llvm/bin"


def code_objects(path):
    """the gfx950 code objects of the library's offload bundles"""
    data = path.read_bytes()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(magic))
        pos = at + len(magic) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + length].decode()
            pos += 24 + length
            if name.endswith("gfx950") and size:
                yield data[at + offset:at + offset + size]
        at = data.find(magic, pos)


@pytest.mark.skipif(not os.path.exists(LLVM + "/llvm-readelf"), reason="no llvm-readelf")
def test_registers_leave_the_waves(tmp_path):
    if not os.path.exists(build.LIB):
        pytest.fail("libpmlgpu.so is not built (python -m pml_amd.build)")
    fat, elf = tmp_path / "fatbin", tmp_path / "code.elf"
    subprocess.run([LLVM + "/llvm-objcopy", "--dump-section", ".hip_fatbin=%s" % fat, build.LIB,
                    str(tmp_path / "copy.so")], check=True)
    seen = 0
    for code in code_objects(fat):
        elf.write_bytes(code)
        notes = subprocess.run([LLVM + "/llvm-readelf", "--notes", str(elf)], stdout=subprocess.PIPE, text=True,
                               check=True).stdout
        for kernel in notes.split("- .agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel.split(".private_segment")[0]) or \
                re.search(r"\.symbol:\s+(\S+)\.kd", kernel)
            k = re.search(r"ntt_(fwd|inv)_regI([jm])([jm])Lb[01]ELi(\d+)ELi(\d+)E", name.group(1))
            if not k:
                continue
            word = k.group(3) if k.group(1) == "fwd" else k.group(2)
            limit = 256 if word == "m" and k.group(5) == "5" else 128
            seen += 1
            assert int(re.search(r"\.vgpr_count:\s+(\d+)", kernel).group(1)) <= limit, name.group(1)
    assert seen > 100
