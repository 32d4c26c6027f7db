"""What the compiler made of the joint forward, whose operands (up to 328 registers a lane) have to stay in registers, and of the
lattices on probabilities, whose helper waves count their loads and stores in flight.  An instantiation whose arrays went to scratch gives
the right results, only slower, so no other test sees it.  Read from the resource records of the library that was built here;
nothing is launched."""

import os
import re
import struct

import msgpack
import pytest

from speech_amd import _native


def _code_objects(library):
    """The gfx950 ELF images of the offload bundle in `library`."""
    at = library.index(b"__CLANG_OFFLOAD_BUNDLE__")
    (count,) = struct.unpack_from("<Q", library, at + 24)
    entry = at + 32
    for _ in range(count):
        offset, size, name_size = struct.unpack_from("<QQQ", library, entry)
        name = library[entry + 24 : entry + 24 + name_size].decode()
        entry += 24 + name_size
        if name.endswith("gfx950"):
            yield library[at + offset : at + offset + size]


def _kernels(elf):
    """The kernel records (msgpack) of the code object's AMDGPU metadata note."""
    (sections_at,) = struct.unpack_from("<Q", elf, 0x28)
    size, number = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(number):
        kind, _, _, offset = struct.unpack_from("<IQQQ", elf, sections_at + i * size + 4)
        if kind != 7:  # SHT_NOTE
            continue
        name_size, text_size, _ = struct.unpack_from("<III", elf, offset)
        text_at = offset + 12 + (name_size + 3) // 4 * 4
        return msgpack.unpackb(elf[text_at : text_at + text_size])["amdhsa.kernels"]
    raise AssertionError("no metadata note")


@pytest.fixture(scope="module")
def kernels():
    if not os.path.exists(_native.LIB_PATH):
        _native.build()
    with open(_native.LIB_PATH, "rb") as file:
        library = file.read()
    return {k[".name"]: k for elf in _code_objects(library) for k in _kernels(elf)}


@pytest.mark.parametrize("H", [256, 320, 384, 512, 640])
def test_joint_forward_uses_no_scratch(kernels, H):
    found = {}
    for name, kernel in kernels.items():
        m = re.search(r"joint_lse_kernelILi(\d+)ELi(\d)ELb([01])ELb([01])ELi(\d)EE", name)
        if m and int(m[1]) == H:
            found[m.groups()[1:]] = kernel[".private_segment_fixed_size"]
    assert len(found) == 3 * 2 * 2 * 2  # losses, ReLU or smooth, with and without the backward's operands, groups of cells
    assert not any(found.values()), {k: v for k, v in found.items() if v}


# MAXD, diagonals a batch, helper waves, and the largest workgroup launched: up to two groups of 64 columns, three or four, ...
LATTICES = [(4, 8, 4, 640), (4, 4, 2, 768), (8, 8, 4, 320), (8, 4, 4, 640), (8, 4, 2, 576)]


@pytest.mark.parametrize("kernel", ["tdt_lattice_pair_kernel", "multiblank_lattice_kernel"])
def test_lattices_on_probabilities_use_no_scratch(kernels, kernel):
    found = {}
    for name, record in kernels.items():
        m = re.search(rf"{kernel}ILi(\d)ELi(\d)ELi(\d)EE", name)
        if m:
            found[tuple(map(int, m.groups())) + (record[".max_flat_workgroup_size"],)] = record[".private_segment_fixed_size"]
    assert sorted(found) == sorted(LATTICES)
    assert not any(found.values()), {k: v for k, v in found.items() if v}
