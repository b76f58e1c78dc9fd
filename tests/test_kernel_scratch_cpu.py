"""The attention backward's kernels and the fp32 forward's use no scratch memory (per-lane private memory), which the runtime
would have to allocate, at the latest on a kernel's first launch: dt_flash_attn_bwd_noalloc and captured calls depend on
that. Read from the metadata of the built library's own code objects."""

import struct

import pytest

msgpack = pytest.importorskip("msgpack")

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
NT_AMDGPU_METADATA = 32


def _code_objects(data):
    """The device ELF images bundled into the library, one per source file."""
    at = data.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, id_len = struct.unpack_from("<QQQ", data, pos)
            ident = data[pos + 24:pos + 24 + id_len].decode()
            pos += 24 + id_len
            if "gfx950" in ident and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, pos)


def _kernels(elf):
    """The metadata of an ELF image's kernels, from its note sections."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    entsize, count = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, shoff + i * entsize + 4)
        if kind != 7:  # SHT_NOTE
            continue
        off, size = struct.unpack_from("<QQ", elf, shoff + i * entsize + 24)
        pos, end = off, off + size
        while pos < end:
            namesz, descsz, note = struct.unpack_from("<III", elf, pos)
            desc = pos + 12 + (namesz + 3) // 4 * 4
            if note == NT_AMDGPU_METADATA:
                yield from msgpack.unpackb(elf[desc:desc + descsz], strict_map_key=False)["amdhsa.kernels"]
            pos = desc + (descsz + 3) // 4 * 4


def test_attention_kernels_use_no_scratch_memory():
    import dirktensor_amd as dt

    if not dt.LIB_PATH.exists():
        pytest.skip("the library is not built")
    data = dt.LIB_PATH.read_bytes()
    sizes = {k[".name"]: (k[".private_segment_fixed_size"], bool(k.get(".uses_dynamic_stack")))
             for elf in _code_objects(data) for k in _kernels(elf)}
    mine = {n: s for n, s in sizes.items() if "flash_bwd" in n or "flash_fwd_f32" in n}
    assert len(mine) >= 13, sorted(sizes)  # prep and dQ in both modes, dK/dV and combined with one and two groups
    assert {n: s for n, s in mine.items() if s != (0, False)} == {}
