"""Registers kept in scratch memory, read from the code objects of the built
library: a spilled value costs a memory round trip wherever it is used, and a
function that was not compiled into its kernel brings scratch of its own."""
import os
import struct

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flash_attn_v100_amd",
                   "libflash_attn_mi355x.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(blob):
    """The GPU code objects of a host library's offload bundles."""
    at = blob.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", blob, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, name_len = struct.unpack_from("<QQQ", blob, entry)
            name = blob[entry + 24:entry + 24 + name_len]
            entry += 24 + name_len
            if name.startswith(b"hip") and size:
                yield blob[at + offset:at + offset + size]
        at = blob.find(MAGIC, at + len(MAGIC))


def kernels(elf):
    """The kernels' records in a code object's AMDGPU metadata note (ELF64, little endian)."""
    msgpack = pytest.importorskip("msgpack")
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        kind, = struct.unpack_from("<I", elf, shoff + i * shentsize + 4)
        offset, size = struct.unpack_from("<QQ", elf, shoff + i * shentsize + 24)
        end = offset + size
        while kind == 7 and offset < end:  # SHT_NOTE
            namesz, descsz, note = struct.unpack_from("<III", elf, offset)
            desc = offset + 12 + (namesz + 3) // 4 * 4
            if note == 32:  # NT_AMDGPU_METADATA
                yield from msgpack.unpackb(elf[desc:desc + descsz], strict_map_key=False)["amdhsa.kernels"]
            offset = desc + (descsz + 3) // 4 * 4


@pytest.fixture(scope="module")
def scratch():
    if not os.path.exists(LIB):
        pytest.skip("library not built")
    with open(LIB, "rb") as f:
        blob = f.read()
    return {k[".name"]: k[".private_segment_fixed_size"] for elf in code_objects(blob) for k in kernels(elf)}


@pytest.mark.parametrize("kernel", ["verify_kernel", "evict_kernel", "decode_splitkv_kernel", "query_major_kernel",
                                    "dkdv_kernel"])
def test_no_scratch(scratch, kernel):
    found = {n: s for n, s in scratch.items() if kernel in n}
    assert found
    assert not {n: s for n, s in found.items() if s}
