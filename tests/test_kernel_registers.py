"""Registers of the built kernels, read from the code objects inside libntship.so (no GPU): a SIMD has 512 of them a lane, so
64 leave eight wavefronts and 65 seven; some kernels are bound by memory latency and were measured slower with fewer."""
import re
import struct

import msgpack
import pytest

from neutronbench_amd import abi


def code_objects(blob):
    """The gfx950 code objects of every offload bundle in the library."""
    for start in (m.start() for m in re.finditer(rb"__CLANG_OFFLOAD_BUNDLE__", blob)):
        (count,) = struct.unpack_from("<Q", blob, start + 24)
        at = start + 32
        for _ in range(count):
            offset, size, name = struct.unpack_from("<QQQ", blob, at)
            triple = blob[at + 24:at + 24 + name]
            at += 24 + name
            if triple.endswith(b"gfx950"):
                yield blob[start + offset:start + offset + size]


def metadata(elf):
    """The AMDGPU metadata note (type 32) of a code object."""
    (table,) = struct.unpack_from("<Q", elf, 32)
    entry, number = struct.unpack_from("<HH", elf, 54)
    for i in range(number):
        kind, = struct.unpack_from("<I", elf, table + i * entry)
        if kind != 4:  # PT_NOTE
            continue
        at, = struct.unpack_from("<Q", elf, table + i * entry + 8)
        name, size, note = struct.unpack_from("<III", elf, at)
        if note == 32:
            at += 12 + (name + 3) // 4 * 4
            return msgpack.unpackb(elf[at:at + size], raw=False)
    raise AssertionError("a code object without metadata")


@pytest.fixture(scope="module")
def kernels():
    with open(abi.LIB_PATH, "rb") as f:
        blob = f.read()
    return {k[".symbol"]: k for elf in code_objects(blob) for k in metadata(elf)["amdhsa.kernels"]}


FLOAT4 = "15HIP_vector_typeIfLj4EE"


@pytest.mark.parametrize("kernel,most", [
    (f"edge_copy_kernelI{FLOAT4}Li4E", 64),  # rows of up to 16 floats copied to edges
    (f"gather_edge_to_row_balanced_kernelI{FLOAT4}Li64ELi1ELb0E", 64),  # permuted sums of rows of 132 to 256 floats
])
def test_registers(kernels, kernel, most):
    found = [k for name, k in kernels.items() if kernel in name]
    assert len(found) == 1
    assert found[0][".vgpr_count"] <= most and found[0][".vgpr_spill_count"] == 0
