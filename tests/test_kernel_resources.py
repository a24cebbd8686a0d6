"""What the compiler made of kernels whose speed or whose shared memory depends on it, read from the built library's own
metadata (no GPU)."""
import struct

import pytest


def kernels_metadata():
    """{kernel name: its metadata} of the device code in the built library."""
    msgpack = pytest.importorskip("msgpack")
    from picolm_amd.csrc import build
    build.load()
    with open(build._built_library(), "rb") as f:
        data = f.read()
    found, at = {}, data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        entries = struct.unpack_from("<Q", data, at + 24)[0]
        p = at + 32
        for _ in range(entries):
            offset, size, id_len = struct.unpack_from("<QQQ", data, p)
            target = data[p + 24:p + 24 + id_len]
            p += 24 + id_len
            if b"gfx950" in target and size:
                found.update(code_object_metadata(data[at + offset:at + offset + size], msgpack))
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)
    return found


def code_object_metadata(elf, msgpack):
    assert elf[:4] == b"\x7fELF"
    headers, (entry, count) = struct.unpack_from("<Q", elf, 32)[0], struct.unpack_from("<HH", elf, 54)
    for i in range(count):
        kind, _, offset, _, _, size = struct.unpack_from("<IIQQQQ", elf, headers + i * entry)
        end = offset + size
        while kind == 4 and offset + 12 <= end:              # notes
            name, length, what = struct.unpack_from("<III", elf, offset)
            start = offset + 12 + (name + 3) // 4 * 4
            if what == 32:                                   # the kernels' metadata
                return {k[".name"]: k for k in msgpack.unpackb(elf[start:start + length])["amdhsa.kernels"]}
            offset = start + (length + 3) // 4 * 4
    return {}


def test_plain_page_attention_stays_in_registers():
    """No private memory: a page looked up there is a wait for everything that is on its way."""
    kernels = {n: k for n, k in kernels_metadata().items() if "attn_plain_mfma_kernel" in n}
    assert len(kernels) == 18
    for name, k in kernels.items():
        assert k[".private_segment_fixed_size"] == 0 and k[".vgpr_spill_count"] == 0, name


def test_shared_rows_begin_at_16_bytes():
    """Rows in dynamic LDS lie behind a kernel's fixed part, and are read and written 16 bytes at a time."""
    for name, k in kernels_metadata().items():
        if "attn_plain_mfma_kernel" in name or "state_chunk_prepare_kernel" in name:
            assert k[".group_segment_fixed_size"] % 16 == 0, name
