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


def kernel_metadata(tmp_path):
    """(symbol, function of a metadata field's name -> its number) of every kernel of the library."""
    tools = [os.path.join(LLVM, t) for t in ("llvm-objcopy", "llvm-readelf")]
    if not all(shutil.which(t) for t in tools):
        pytest.skip("needs the toolchain's llvm-objcopy and llvm-readelf")
    fat = tmp_path / "fatbin"
    subprocess.run([tools[0], f"--dump-section=.hip_fatbin={fat}", _lib.LIB_PATH, str(tmp_path / "copy.so")], check=True)
    for i, image in enumerate(code_objects(fat.read_bytes())):
        f = tmp_path / f"{i}.co"
        f.write_bytes(image)
        notes = subprocess.run([tools[1], "--notes", str(f)], check=True, capture_output=True, text=True).stdout
        for entry in re.split(r"\n\s*- \.agpr_count", notes)[1:]:
            yield (re.search(r"\.symbol:\s*(\S+)", entry).group(1),
                   lambda field, entry=entry: int(re.search(r"\." + field + r":\s*(\d+)", entry).group(1)))


def test_no_kernel_spills(tmp_path):
    spills, kernels = [], 0
    for symbol, number in kernel_metadata(tmp_path):
        kernels += 1
        if number("vgpr_spill_count"):
            spills.append((symbol, number("vgpr_spill_count")))
    assert kernels > 100, "the library's metadata was not read"
    assert not spills


def test_scalar_spills_are_the_known_ones(tmp_path):
    """A scalar that does not fit goes to a lane of a vector register, not to memory, at two instructions.  The kernels
    that have some, and how many at most: those of rank above 64 with a look-up or a step of its own per unit, the one-launch
    kernel, whose two halves share one argument block, the plan of more than 2048 adapters, and the contiguous allocator."""
    known = {r"plan_kernelILb0ELi1024ELb1E": 2, r"shrink_kernelI\w+Li[12]ELi8E": 47, r"expand_small_kernelI\w+Li4ELb0ELb0ELb1E": 44,
             r"expand_small_kernelI\w+Li4ELb0ELb1ELb0E": 14, r"\d+expand_kernelI\w+Li4ELb0ELb0ELb1E": 58,
             r"\d+expand_kernelI\w+Li4ELb0ELb1ELb0E": 27, r"decode_kernelI": 9, r"pool_alloc_contiguous_kernel": 12}
    for symbol, number in kernel_metadata(tmp_path):
        assert number("private_segment_fixed_size") == 0, symbol
        allowed = max((n for pattern, n in known.items() if re.search(pattern, symbol)), default=0)
        assert number("sgpr_spill_count") <= allowed, (symbol, number("sgpr_spill_count"))


def kernel_code(tmp_path, pattern):
    """(symbol, its instructions) of the library's kernels whose symbol matches."""
    objdump = os.path.join(LLVM, "llvm-objdump")
    if not shutil.which(objdump):
        pytest.skip("needs the toolchain's llvm-objdump")
    for _ in kernel_metadata(tmp_path):   # (leaves the device images behind)
        pass
    for f in sorted(tmp_path.glob("*.co")):
        if re.search(pattern.encode(), f.read_bytes()):
            text = subprocess.run([objdump, "-d", "--no-show-raw-insn", str(f)], check=True, capture_output=True, text=True).stdout
            for part in re.split(r"\n(?=[0-9a-f]+ <)", text):
                name = re.match(r"[0-9a-f]+ <(\S+)>:", part)
                if name and re.search(pattern, name.group(1)):
                    yield name.group(1), part


def test_small_expand_stores_y_one_way(tmp_path):
    """A launch that writes y through and one that does not are different kernels: with both kinds in one, every launch of a few tokens
    pays for the exchange of halves that only the former need (0.15 of 3.6 us)."""
    kinds = {}
    for symbol, code in kernel_code(tmp_path, "expand_small_kernel"):
        stores = re.findall(r"global_store_dwordx4 [^\n]*", code)
        kinds.setdefault(frozenset("sc1" in s for s in stores), []).append(symbol)
    assert set(kinds) == {frozenset([True]), frozenset([False])}, {k: len(v) for k, v in kinds.items()}


def test_tall_compensation_has_no_form_that_writes_y_through(tmp_path):
    """How much of y a compensation writes is not known at the launch; in 16-token tiles it pays however little that is."""
    symbols = [s for s, _ in kernel_metadata(tmp_path)]
    forms = {re.search(r"Lb(\d)ELb(\d)ELb\dEEE", s).groups() for s in symbols if re.search(r"\d+expand_kernelI", s)}   # ..., COMP, THROUGH, ONCE
    assert forms == {("0", "0"), ("0", "1"), ("1", "0")}


def test_partials_are_read_once_in_a_form_of_their_own(tmp_path):
    """Rows of the partials that are no whole lines, and a compensation's, are read the plain way: some launch has no non-temporal load."""
    kinds = {bool(re.search(r"global_load_dwordx4 [^\n]*\bnt\b", code)) for _, code in kernel_code(tmp_path, "shrink_reduce_kernel")}
    assert kinds == {True, False}
