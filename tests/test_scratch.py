"""Kernels whose operands are meant to stay in registers use no scratch memory: read from the metadata of the code objects in the built
library, so that a compiler's spill shows up without a GPU."""

import os
import struct

import pytest

import scaffold_amd

msgpack = pytest.importorskip("msgpack")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    at = blob.find(MAGIC)
    while at >= 0:
        pos = at + len(MAGIC) + 8
        for _ in range(struct.unpack_from("<Q", blob, at + len(MAGIC))[0]):
            offset, size, length = struct.unpack_from("<QQQ", blob, pos)
            name = blob[pos + 24:pos + 24 + length]
            pos += 24 + length
            if b"gfx950" in name and size:
                yield blob[at + offset:at + offset + size]
        at = blob.find(MAGIC, at + 1)


def _kernels():
    """(mangled name, metadata) of every kernel in the library: the notes of its ELF code objects hold one msgpack map each."""
    with open(os.path.join(os.path.dirname(scaffold_amd.__file__), "libscaffold_hip.so"), "rb") as f:
        blob = f.read()
    for elf in _code_objects(blob):
        shoff, = struct.unpack_from("<Q", elf, 40)
        shentsize, shnum = struct.unpack_from("<HH", elf, 58)
        for i in range(shnum):
            kind, = struct.unpack_from("<I", elf, shoff + i * shentsize + 4)
            if kind != 7:  # SHT_NOTE
                continue
            offset, = struct.unpack_from("<Q", elf, shoff + i * shentsize + 24)
            namesz, descsz, note = struct.unpack_from("<III", elf, offset)
            if note == 32:  # NT_AMDGPU_METADATA
                start = offset + 12 + (namesz + 3) // 4 * 4
                for k in msgpack.unpackb(elf[start:start + descsz], raw=False)["amdhsa.kernels"]:
                    yield k[".name"], k


@pytest.mark.parametrize("kernel", ["patch_reduce_kernel", "patch_gather_kept_kernel"])
def test_no_scratch(kernel):
    found = [(n, k) for n, k in _kernels() if kernel in n]
    assert found
    assert [(n, k[".private_segment_fixed_size"], k.get(".vgpr_spill_count", 0)) for n, k in found
            if k[".private_segment_fixed_size"] or k.get(".vgpr_spill_count", 0)] == []
