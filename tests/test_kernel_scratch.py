"""The kernels that the allocation-free SVD entry point launches use no scratch
memory, which the runtime would allocate at a launch: their frame size in the
metadata of the built library is zero."""

import os
import struct

import pytest

from oqupy_amd.build import TARGET

msgpack = pytest.importorskip("msgpack")

KERNELS = ["transpose_kernel", "small_svd_kernel", "gram_svd_kernel", "gram_replay_kernel",
           "qrcp_kernel", "build_rh_kernel", "jacobi_kernel", "jacobi_tile_kernel",
           "column_norm_kernel", "rank_sort_kernel", "truncate_kernel", "apply_q_kernel",
           "apply_q_wave_kernel", "emit_kernel"]

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    """ELF images for the GPU in the library's offload bundles."""
    at = data.find(MAGIC)
    while at >= 0:
        pos = at + len(MAGIC)
        count, = struct.unpack_from("<Q", data, pos)
        pos += 8
        for _ in range(count):
            off, size, length = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + length]
            pos += 24 + length
            if b"gfx950" in name and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + 1)


def _notes(elf):
    """Descriptors of the AMDGPU metadata notes."""
    phoff, = struct.unpack_from("<Q", elf, 32)
    phentsize, phnum = struct.unpack_from("<HH", elf, 54)
    for k in range(phnum):
        kind, _, off, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + k * phentsize)
        if kind != 4:
            continue
        pos, end = off, off + size
        while pos < end:
            n, d, typ = struct.unpack_from("<III", elf, pos)
            pos += 12
            name = elf[pos:pos + n].rstrip(b"\0")
            pos += (n + 3) // 4 * 4
            if name == b"AMDGPU" and typ == 32:
                yield elf[pos:pos + d]
            pos += (d + 3) // 4 * 4


def _frames():
    with open(TARGET, "rb") as f:
        data = f.read()
    out = {}
    for elf in _code_objects(data):
        for note in _notes(elf):
            for k in msgpack.unpackb(note, strict_map_key=False)["amdhsa.kernels"]:
                out[k[".name"]] = k[".private_segment_fixed_size"]
    return out


@pytest.mark.skipif(not os.path.exists(TARGET), reason="library not built")
def test_allocation_free_kernels_use_no_scratch():
    frames = _frames()
    for kernel in KERNELS:
        mangled = f"{len(kernel)}{kernel}"
        found = {k: v for k, v in frames.items() if mangled in k}
        assert found, kernel
        assert not any(found.values()), found
