"""Registers of the single-step kernels as built: a masked pull step waits for
two rounds of loads per cell, and its bandwidth is the number of wavefronts
that wait side by side, so code for rare cells (outlets, obstacles) must not
take registers that cost the others a wavefront."""
import os
import re
import struct
import subprocess

import pytest

from lettuce_amd import _build, _native as N

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(path):
    """the gfx950 ELF files bundled in a library"""
    data = open(path, "rb").read()
    for m in re.finditer(re.escape(MAGIC), data):
        at, out = m.start() + len(MAGIC), []
        count, = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(min(count, 8)):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            name = data[at + 24:at + 24 + length]
            at += 24 + length
            if name.endswith(_build.ARCH.encode()) and size:
                out.append(data[m.start() + offset:m.start() + offset + size])
        yield from out


@pytest.fixture(scope="module")
def registers(tmp_path_factory):
    """VGPRs by mangled kernel name"""
    if not os.path.exists(READELF):
        pytest.skip("llvm-readelf is not installed")
    N.lib()  # builds the library if there is none
    found = {}
    for i, elf in enumerate(_code_objects(_build.LIB)):
        path = tmp_path_factory.mktemp("co") / f"{i}.elf"
        path.write_bytes(elf)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True,
                               check=True).stdout
        for name, vgprs in re.findall(r"\.name: +(\S+)\n(?:(?!\.name:).)*?\.vgpr_count: +(\d+)", notes, re.S):
            found[name] = int(vgprs)
    return found


# 512 VGPRs per SIMD lane, handed out in eights
@pytest.mark.parametrize("stencil,kbc,waves", [("D2Q9", True, 8), ("D2Q9", False, 8),
                                               ("D3Q19", False, 6), ("D3Q27", False, 6),
                                               ("D3Q27", True, 5)])
def test_masked_pull_steps_keep_their_wavefronts(registers, stencil, kbc, waves):
    seen = 0
    for name, vgprs in registers.items():
        m = re.match(r"_ZN3lbm11step_kernelINS_\d" + stencil + r"ENS_\d+(St\w+?)ELi(\d)ELb1ELi2E", name)
        if m and m.group(1) != "StF64" and (m.group(2) == "3") == kbc:
            seen += 1
            assert 512 // (-(-vgprs // 8) * 8) >= waves, (name, vgprs)
    assert seen == (8 if kbc else 32), seen  # 4 formats, 2 kinds of blocks, 4 other collisions
