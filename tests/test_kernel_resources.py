"""What the built library's own metadata says of its kernels' registers: the small-tile kernel (csrc/decode.hip), whose instances are
held to a number of registers by their launch bounds, keeps none of them in memory."""

import re
import struct

import msgpack

from nanovllm_voxcpm_amd import _hip


def _kernels():
    """Metadata of every kernel for the GPU in the library's device images."""
    data = open(_hip.library_path(), "rb").read()
    magic, at, found = b"__CLANG_OFFLOAD_BUNDLE__", 0, []
    while (at := data.find(magic, at)) >= 0:
        place = at + len(magic)
        (images,) = struct.unpack_from("<Q", data, place)
        place += 8
        for _ in range(images):
            offset, size, length = struct.unpack_from("<QQQ", data, place)
            name = data[place + 24 : place + 24 + length]
            place += 24 + length
            if b"gfx950" in name and size:
                found += _notes(data[at + offset : at + offset + size])
        at += len(magic)
    return found


def _notes(elf):
    phoff, phentsize, phnum = struct.unpack_from("<Q", elf, 32)[0], *struct.unpack_from("<HH", elf, 54)
    kernels = []
    for i in range(phnum):
        kind, _, offset, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + i * phentsize)
        end = offset + size
        while kind == 4 and offset < end:  # PT_NOTE
            namesz, descsz, note = struct.unpack_from("<III", elf, offset)
            desc = offset + 12 + (namesz + 3 & ~3)
            if note == 32 and elf[offset + 12 : offset + 18] == b"AMDGPU":
                kernels += msgpack.unpackb(elf[desc : desc + descsz])["amdhsa.kernels"]
            offset = desc + (descsz + 3 & ~3)
    return kernels


def test_small_tile_kernel_keeps_its_registers():
    decode = {k[".name"]: k for k in _kernels() if "decode_kernel" in k[".name"]}
    assert len(decode) > 100
    assert [n for n, k in decode.items() if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]] == []


def test_two_small_tile_workgroups_fit_a_compute_unit():
    """Up to rank 16 and K = 2048 (four, eight steps of K a wavefront) eight wavefronts hold at most 128 registers each, whatever the instance."""
    staged = re.compile(r"decode_kernelI\w+?Li(8|16)ELi(4|8)ELb1E")
    some = {k[".name"]: k[".vgpr_count"] for k in _kernels() if staged.search(k[".name"])}
    assert len(some) >= 48 and [n for n, v in some.items() if v > 128] == []


def test_kernels_over_64_token_tiles_keep_their_registers():
    some = {k[".name"]: k for k in _kernels() if re.search("wide_kernel|sgmv_shrink_kernel", k[".name"])}
    assert len(some) == 10
    assert [n for n, k in some.items() if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"] or k[".vgpr_count"] > 128] == []
