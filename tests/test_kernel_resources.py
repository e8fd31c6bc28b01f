"""What the compiler gave the kernels, from the metadata of the library as built: no kernel keeps registers in memory.  (Spills cost
the shrink of 64-token tiles up to 13 % before its bounds were set by them.)"""
import os
import re
import shutil
import struct
import subprocess

import pytest

from valora_amd import _lib

LLVM = "/opt/rocm/llvm/bin"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(fatbin: bytes):
    """The device images of every translation unit's bundle."""
    at = fatbin.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", fatbin, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", fatbin, p)
            name = fatbin[p + 24:p + 24 + length].decode()
            p += 24 + length
            if "gfx950" in name and size:
                yield fatbin[at + off:at + off + size]
        at = fatbin.find(MAGIC, at + 1)


def test_no_kernel_spills(tmp_path):
    tools = [os.path.join(LLVM, t) for t in ("llvm-objcopy", "llvm-readelf")]
    if not all(shutil.which(t) for t in tools):
        pytest.skip("needs the toolchain's llvm-objcopy and llvm-readelf")
    fat = tmp_path / "fatbin"
    subprocess.run([tools[0], f"--dump-section=.hip_fatbin={fat}", _lib.LIB_PATH, str(tmp_path / "copy.so")], check=True)
    spills, kernels = [], 0
    for i, image in enumerate(code_objects(fat.read_bytes())):
        f = tmp_path / f"{i}.co"
        f.write_bytes(image)
        notes = subprocess.run([tools[1], "--notes", str(f)], check=True, capture_output=True, text=True).stdout
        for entry in re.split(r"\n\s*- \.agpr_count", notes)[1:]:
            kernels += 1
            count = re.search(r"\.vgpr_spill_count:\s*(\d+)", entry)
            if int(count.group(1)):
                spills.append((re.search(r"\.symbol:\s*(\S+)", entry).group(1), count.group(1)))
    assert kernels > 100, "the library's metadata was not read"
    assert not spills
