"""Registers of the compiled kernels: as few as leave room for the wavefronts per
SIMD that a kernel's speed rests on (512 vector registers per lane, in steps of
eight).  Read from the code objects' notes in the built library."""
import os
import re
import struct
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(REPO, "qcdgpu_amd", "libqcdhip.so")
LLVM = "/opt/rocm/llvm/bin"

pytestmark = [
    pytest.mark.skipif(not os.path.exists(LIB), reason="libqcdhip.so not built"),
    pytest.mark.skipif(not os.path.exists(os.path.join(LLVM, "llvm-readelf")), reason="llvm-readelf missing"),
]


@pytest.fixture(scope="module")
def registers(tmp_path_factory):
    """{mangled kernel name: vector registers}."""
    d = tmp_path_factory.mktemp("notes")
    fat = str(d / "fat")
    subprocess.run([os.path.join(LLVM, "llvm-objcopy"), "--dump-section", ".hip_fatbin=" + fat, LIB, str(d / "rest")],
                   check=True, capture_output=True)
    data = open(fat, "rb").read()
    magic, out, pos = b"__CLANG_OFFLOAD_BUNDLE__", {}, 0
    while True:   # one bundle per source file
        pos = data.find(magic, pos)
        if pos < 0:
            return out
        at = pos + len(magic)
        (count,) = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, at)
            name = data[at + 24:at + 24 + n].decode()
            at += 24 + n
            if "gfx950" not in name:
                continue
            obj = str(d / "object")
            open(obj, "wb").write(data[pos + off:pos + off + size])
            notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", obj], check=True, capture_output=True,
                                   text=True).stdout
            for block in notes.split("  - .agpr_count")[1:]:
                out[re.search(r"\.name:\s+(\S+)", block).group(1)] = int(re.search(r"\.vgpr_count:\s+(\d+)", block).group(1))
        pos += len(magic)


def _waves(vgprs):
    return min(8, 512 // (-(-vgprs // 8) * 8))


@pytest.mark.parametrize("kernel,waves", [
    ("k_wilsonIfLi2ELi4ELb0ELj1E", 8),     # Wilson loop, a thread per site
    ("k_wilsonIfLi3ELi12ELb0ELj1E", 4),
    ("k_wilsonIfLi3ELi12ELb1ELj1E", 4),
    ("k_wilsonIfLi3ELi18ELb0ELj1E", 4),
    ("k_update1IfLi3ELi18ELb0ELi2ELb1E", 4),        # one wavefront per 64 links, heatbath with the plaquette
    ("k_update1IfLi3ELi18ELb0ELi3ELb1E", 4),
    ("k_update_batch1IfLi3ELi18ELb0ELi2ELb1E", 4),
    ("k_update_batch3IdLi3ELi12ELb1ELi0ELb0ELb1E", 3),   # overrelaxation of large FP64 batches
    ("k_update_batch3IdLi3ELi18ELb1ELi0ELb0ELb1E", 3),
    ("k_update_batch3IdLi3ELi18ELb1ELi0ELb1ELb1E", 3),
])
def test_wavefronts_per_simd(registers, kernel, waves):
    found = [v for n, v in registers.items() if kernel in n]
    assert found, "no kernel " + kernel
    assert all(_waves(v) >= waves for v in found), found
