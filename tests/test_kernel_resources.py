"""What the compiler gave the kernels of the built libraries, from the metadata of their code objects: no private memory where a
kernel's chain of loads is its time."""
import os
import struct

import pytest

msgpack = pytest.importorskip("msgpack")
PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "eventgpt_amd")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(data):
    """Device ELF images of the offload bundles of a library."""
    at = data.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + len(MAGIC))
        o = at + len(MAGIC) + 8
        for _ in range(n):
            start, size, length = struct.unpack_from("<3Q", data, o)
            if b"gfx950" in data[o + 24:o + 24 + length]:
                yield data[at + start:at + start + size]
            o += 24 + length
        at = data.find(MAGIC, at + 1)


def kernels(elf):
    """The kernels' entries in the AMDGPU metadata note (type 32) of an ELF64 image."""
    off, = struct.unpack_from("<Q", elf, 32)
    entry, count = struct.unpack_from("<HH", elf, 54)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, off + i * entry)
        at, = struct.unpack_from("<Q", elf, off + i * entry + 8)
        size, = struct.unpack_from("<Q", elf, off + i * entry + 32)
        end = at + size
        while kind == 4 and at < end:
            name, desc, note = struct.unpack_from("<3I", elf, at)
            body = at + 12 + (name + 3) // 4 * 4
            if note == 32:
                yield from msgpack.unpackb(elf[body:body + desc])["amdhsa.kernels"]
            at = body + (desc + 3) // 4 * 4


def private_bytes(library):
    path = os.path.join(PKG, library)
    if not os.path.exists(path):
        pytest.skip(f"{library} is not built")
    with open(path, "rb") as f:
        data = f.read()
    return {k[".name"]: k[".private_segment_fixed_size"] for elf in code_objects(data) for k in kernels(elf)}


@pytest.mark.parametrize("kernel", ["parallel_step_kernel", "attend_step_kernel", "ssd_step_kernel", "scan_chunk_state_kernel",
                                    "scan_chunk_pass_kernel", "scan_chunk_out_kernel"])
def test_no_private_memory(kernel):
    """(The scans' instances for row strides of 2^24 elements and more, offsets of 64 bits, keep a few registers there.)"""
    found = {name: size for name, size in private_bytes("_D.so").items() if kernel in name and "128ExEEv" not in name}
    assert found and not any(found.values()), found
