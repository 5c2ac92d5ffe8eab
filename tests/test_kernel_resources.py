"""Registers of the compiled kernels (CPU only: the code object metadata in the
library that was built here): none spills its operands to scratch, and the
kernels whose speed rests on a number of waves per SIMD keep it."""

from __future__ import annotations

import struct
import subprocess
from pathlib import Path

import pytest

LIB = Path(__file__).resolve().parent.parent / "maxsim_amd" / "libmaxsim_amd.so"
msgpack = pytest.importorskip("msgpack")


def _code_objects(data: bytes):
    """The gfx950 ELF images of the library's offload bundles."""
    at = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + 24)
        pos = at + 32
        for _ in range(count):
            offset, size, name_len = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + name_len]
            pos += 24 + name_len
            if b"gfx950" in name and size:
                yield data[at + offset:at + offset + size]
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)


def _kernels(elf: bytes):
    """Kernel entries of an image's metadata note (ELF64, note type 32)."""
    phoff, = struct.unpack_from("<Q", elf, 32)
    phentsize, phnum = struct.unpack_from("<HH", elf, 54)
    for i in range(phnum):
        kind, _, offset, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + i * phentsize)
        if kind != 4:  # PT_NOTE
            continue
        pos, end = offset, offset + size
        while pos < end:
            name_len, desc_len, note = struct.unpack_from("<III", elf, pos)
            desc = pos + 12 + (name_len + 3) // 4 * 4
            if note == 32:
                yield from msgpack.unpackb(elf[desc:desc + desc_len])["amdhsa.kernels"]
            pos = desc + (desc_len + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    if not LIB.exists():
        pytest.fail(f"{LIB} is not built; run python maxsim_amd/_build.py")
    found = {k[".name"]: k for elf in _code_objects(LIB.read_bytes()) for k in _kernels(elf)}
    assert found
    out = subprocess.run(["c++filt"], input="\n".join(found), text=True, capture_output=True,
                         check=True).stdout.split("\n")
    return {n.replace("maxsim::", "").removeprefix("void ").split("(")[0]: k
            for n, k in zip(out, found.values())}


def test_no_kernel_spills_its_operands(kernels):
    # up to 50 spilled registers were measured and pay (mixed row loads)
    spilled = {n: k[".vgpr_spill_count"] for n, k in kernels.items()
               if k[".vgpr_spill_count"] > 50}
    assert not spilled, spilled


def test_contrastive_dd_two_workgroups_per_cu(kernels):
    # 512 threads are two waves per SIMD: four waves in 512 registers
    of = {n: k[".vgpr_count"] for n, k in kernels.items()
          if n.startswith("dd_contrastive_kernel<") and ", true, 1, " in n}
    assert len(of) == 5 and max(of.values()) <= 128, of
