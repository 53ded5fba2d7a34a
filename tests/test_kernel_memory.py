"""No kernel of the built library keeps anything in scratch memory: an array
that the compiler could not resolve into registers, or a spill, costs the
kernel trips to memory in its inner loop and fails no other test."""
import re
import shutil
import struct
import subprocess

import pytest

from gcge_amd import abi

READELF = shutil.which("llvm-readelf", path="/opt/rocm/llvm/bin") or shutil.which("llvm-readelf")


def scratch_bytes(path, tmp):
    """Scratch bytes per lane of each gfx950 kernel, from the notes of the
    library's offload bundles."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    with open(path, "rb") as f:
        lib = f.read()
    out = {}
    for at in (m.start() for m in re.finditer(magic, lib)):
        count, = struct.unpack_from("<Q", lib, at + len(magic))
        p = at + len(magic) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", lib, p)
            target = lib[p + 24:p + 24 + length].decode()
            p += 24 + length
            if "gfx950" not in target or size == 0:
                continue
            tmp.write_bytes(lib[at + offset:at + offset + size])
            notes = subprocess.run([READELF, "--notes", str(tmp)], check=True,
                                   capture_output=True, text=True).stdout
            for k in re.finditer(r"\.name:\s+(\S+)\n.*?\.private_segment_fixed_size:\s+(\d+)",
                                 notes, re.S):
                out[k[1]] = int(k[2])
    return out


@pytest.mark.skipif(READELF is None, reason="llvm-readelf is not here")
def test_no_scratch(tmp_path):
    got = scratch_bytes(abi.LIB_PATH, tmp_path / "code")
    assert len(got) > 100
    assert {k: v for k, v in got.items() if v} == {}
