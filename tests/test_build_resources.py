"""Register spills of the built kernels, read from the metadata that the
compiler writes into libvx_attn.so (no GPU needed)."""
import re
import struct

import msgpack

from vidax_amd import _lib

NT_AMDGPU_METADATA = 32


def _code_objects(blob):
    """The gfx950 ELF images of every offload bundle in the library."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    for m in re.finditer(re.escape(magic), blob):
        at = m.start()
        (count,) = struct.unpack_from("<Q", blob, at + len(magic))
        pos = at + len(magic) + 8
        for _ in range(count):
            offset, size, name_len = struct.unpack_from("<QQQ", blob, pos)
            name = blob[pos + 24:pos + 24 + name_len].decode()
            pos += 24 + name_len
            if "gfx950" in name and size:
                yield blob[at + offset:at + offset + size]


def _kernels(elf):
    """Metadata maps of the kernels of one code object (ELF64, little endian)."""
    assert elf[:6] == b"\x7fELF\x02\x01"
    (shoff,) = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        sh = shoff + i * shentsize
        (kind,) = struct.unpack_from("<I", elf, sh + 4)
        pos, size = struct.unpack_from("<QQ", elf, sh + 24)
        end = pos + size
        while kind == 7 and pos < end:  # SHT_NOTE
            name_size, desc_size, note = struct.unpack_from("<III", elf, pos)
            desc = pos + 12 + (name_size + 3) // 4 * 4
            if note == NT_AMDGPU_METADATA:
                yield from msgpack.unpackb(elf[desc:desc + desc_size], strict_map_key=False)["amdhsa.kernels"]
            pos = desc + (desc_size + 3) // 4 * 4


def test_kernels_do_not_spill():
    """Only the pairs over key halves at head dim 128, which hold the second
    group's copies and the partials' addresses, spill a few registers."""
    with open(_lib.LIB_PATH, "rb") as f:
        blob = f.read()
    kernels = {k[".name"]: k for elf in _code_objects(blob) for k in _kernels(elf)}
    assert sum("na3d" in n for n in kernels) >= 13 and sum("flash" in n for n in kernels) >= 40, sorted(kernels)
    for name, k in kernels.items():
        allowed = 12 if re.search(r"flash_pair_split_kernelILi[01]ELi128E", name) else 0
        assert k[".vgpr_spill_count"] <= allowed, (name, k[".vgpr_spill_count"])
        assert k[".private_segment_fixed_size"] <= 4 * allowed, (name, k[".private_segment_fixed_size"])
