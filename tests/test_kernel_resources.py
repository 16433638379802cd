"""Resources of the built kernels, from the metadata that the compiler writes beside them."""

import re
import struct

import pytest

msgpack = pytest.importorskip("msgpack")


def _code_objects(data):
    """The gfx950 ELF images of the library's offload bundles."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        n = struct.unpack_from("<Q", data, at + len(magic))[0]
        p = at + len(magic) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in name and size:
                yield data[at + off:at + off + size]
        at = data.find(magic, at + len(magic))


def _kernels(elf):
    shoff, = struct.unpack_from("<Q", elf, 40)
    entsize, count = struct.unpack_from("<HH", elf, 58)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, shoff + i * entsize + 4)
        off, size = struct.unpack_from("<QQ", elf, shoff + i * entsize + 24)
        if kind != 7:  # SHT_NOTE
            continue
        while size >= 12:
            namesz, descsz, ntype = struct.unpack_from("<III", elf, off)
            desc = off + 12 + (namesz + 3) // 4 * 4
            if ntype == 32 and elf[off + 12:off + 18] == b"AMDGPU":
                yield from msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]
            step = desc + (descsz + 3) // 4 * 4 - off
            off, size = off + step, size - step


@pytest.fixture(scope="module")
def kernels():
    from nexusquant_amd import _lib
    with open(_lib.LIB_PATH, "rb") as f:
        data = f.read()
    found = {k[".name"]: k for elf in _code_objects(data) for k in _kernels(elf)}
    assert any("paged_attn_kernel" in n for n in found) and any("quant_rows_kernel" in n for n in found)
    return found


def test_no_kernel_spills(kernels):
    for name, k in kernels.items():
        assert k[".private_segment_fixed_size"] == 0, name


def test_attention_kernels_keep_their_waves(kernels):
    """4 waves per SIMD at head_dim 64 and 128 (128 registers), 2 at 256."""
    for name, k in kernels.items():
        if "paged_attn_kernel" in name:
            assert k[".vgpr_count"] <= (256 if "ILi256E" in name else 128), name


def test_quantizer_kernels_leave_room_for_their_waves(kernels):
    """LDS of a block: four to a CU's 160 KB, three of padded keys.  Registers at head_dim 256: 4 waves
    per SIMD for values up to 8 levels and 3 past that, 2 for keys (gathered keys of 16 levels have 1)."""
    seen = 0
    for name, k in kernels.items():
        m = re.search(r"quant_rows_kernelILi(\d+)ELi(\d+)ELb([01])ELi(\d)ELi(\d+)ELb([01])ELi(\d)E", name)
        if not m:
            continue
        seen += 1
        head_dim, levels, is_key, sel = int(m[5]), int(m[2]), m[3] == "1", int(m[7])
        assert k[".group_segment_fixed_size"] <= (49152 if head_dim == 96 and is_key else 40960), name
        if head_dim == 256 and not (is_key and levels == 16 and sel == 2):
            registers = 256 if is_key else 168 if levels == 16 else 128
            assert k[".vgpr_count"] + k[".agpr_count"] <= registers, name
    assert seen > 100
