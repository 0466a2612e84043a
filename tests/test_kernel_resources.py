"""What the compiler gave the kernels of the built library, read from their code objects' metadata."""
import os
import struct

import pytest

msgpack = pytest.importorskip("msgpack")


def _library() -> bytes:
    from flute_extended import _lib
    with open(_lib.lib._name, "rb") as f:
        return f.read()


def _code_objects(data: bytes):
    """The gfx950 ELF images of the offload bundles in the library (one bundle per source file)."""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := data.find(magic, at)) >= 0:
        pos = at + len(magic) + 8
        for _ in range(struct.unpack_from("<Q", data, pos - 8)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            triple = data[pos + 24:pos + 24 + length]
            pos += 24 + length
            if triple.endswith(b"gfx950") and size:
                yield data[at + offset:at + offset + size]
        at += len(magic)


def _kernels():
    """{mangled name: metadata} of every kernel (the notes of type 32 hold them as msgpack)."""
    found = {}
    for elf in _code_objects(_library()):
        assert elf[:4] == b"\x7fELF"
        table, = struct.unpack_from("<Q", elf, 40)
        entry, count = struct.unpack_from("<HH", elf, 58)
        for i in range(count):
            kind, offset, size = struct.unpack_from("<4xI16xQQ", elf, table + i * entry)
            if kind != 7:
                continue
            end = offset + size
            while offset < end:
                name, desc, note = struct.unpack_from("<III", elf, offset)
                start = offset + 12 + (name + 3 & ~3)
                if note == 32:
                    for k in msgpack.unpackb(elf[start:start + desc])["amdhsa.kernels"]:
                        found[k[".name"]] = k
                offset = start + (desc + 3 & ~3)
    return found


@pytest.mark.parametrize("kernel", ["gemm_few_kernel", "gemv4_kernel"])
def test_lookup_kernels_use_no_scratch_memory(kernel):
    """Tables, codes and sums live in registers and LDS: a kernel with a private segment fetches some of
    them from memory (a local array with a runtime index, or registers spilled)."""
    kernels = {n: k for n, k in _kernels().items() if kernel in n}
    assert kernels
    assert not {n: k[".private_segment_fixed_size"] for n, k in kernels.items() if k[".private_segment_fixed_size"]}


def test_few_row_kernel_takes_width_pairs_in_one_launch():
    """Every pair of widths, the wider first, in 16- and 32-row workgroups, both LUT types, one weight and
    several; not (4, 4), whose tables and codes exceed a CU's LDS."""
    kernels = _kernels()
    for rows in (1, 2):
        for bf16 in (0, 1):
            for segs in (0, 1):
                for b1 in (1, 2, 3, 4):
                    for b2 in range(b1 + 1):
                        name = f"_ZN5flute15gemm_few_kernelILi{rows}ELb{bf16}ELi{b1}ELi{b2}ELb{segs}EEEvNS_10GemmParamsE"
                        assert (name in kernels) == ((b1, b2) != (4, 4)), name
