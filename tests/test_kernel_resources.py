"""What the compiler gave the kernels, from the metadata of the gfx950 code objects in liblbtree.so (built here from source):
registers that were moved to memory, and bytes of scratch memory per lane."""
import os
import re
import struct

import pytest

msgpack = pytest.importorskip("msgpack")

_BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"
_NOTES, _AMDGPU_METADATA = 7, 32  # section type, note type


def _code_objects(data):
    at = data.find(_BUNDLE)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + 24)
        entry = at + 32
        for _ in range(n):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            if b"gfx950" in data[entry + 24:entry + 24 + length]:
                yield data[at + offset:at + offset + size]
            entry += 24 + length
        at = data.find(_BUNDLE, at + 24)


def _kernels_of(elf):
    section, = struct.unpack_from("<Q", elf, 40)
    size, count = struct.unpack_from("<HH", elf, 58)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, section + i * size + 4)
        if kind != _NOTES:
            continue
        at, length = struct.unpack_from("<QQ", elf, section + i * size + 24)
        end = at + length
        while at < end:
            name, desc, note = struct.unpack_from("<III", elf, at)
            at += 12 + (name + 3) // 4 * 4
            if note == _AMDGPU_METADATA:
                yield from msgpack.unpackb(elf[at:at + desc])["amdhsa.kernels"]
            at += (desc + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    import lbtree

    path = os.path.join(os.path.dirname(os.path.dirname(lbtree.__file__)), "csrc", "liblbtree.so")
    with open(path, "rb") as f:
        found = {k[".name"]: k for elf in _code_objects(f.read()) for k in _kernels_of(elf)}
    assert len(found) > 50
    return found


# template arguments as the symbol has them: bins of one byte (h) or two (t), bins of a load, gradients in the record, root,
# striped, bins of a row that a lane takes where four lanes share them evenly (0: they do not)
@pytest.mark.parametrize("arguments,spilled", [
    ("hLi16ELb0ELb0ELb1ELi0", 3), ("hLi16ELb1ELb0ELb1ELi0", 3), ("hLi16ELb0ELb1ELb1ELi0", 8), ("hLi16ELb1ELb1ELb1ELi0", 8),
    ("hLi16ELb0ELb0ELb0ELi0", 0), ("hLi16ELb1ELb0ELb0ELi0", 0), ("hLi16ELb0ELb1ELb0ELi0", 0), ("hLi16ELb1ELb1ELb0ELi0", 0),
    ("tLi4ELb0ELb0ELb0ELi0", 0), ("tLi4ELb1ELb0ELb0ELi0", 0), ("tLi4ELb0ELb1ELb0ELi0", 0), ("tLi4ELb1ELb1ELb0ELi0", 0),
    ("hLi16ELb0ELb0ELb1ELi14", 2), ("hLi16ELb0ELb0ELb1ELi16", 2), ("hLi16ELb1ELb0ELb1ELi14", 0),
])
def test_histogram_kernels_keep_their_registers(kernels, arguments, spilled):
    """The layout's variants are one source: what one of them needs must not cost the others registers."""
    match = [k for name, k in kernels.items() if "binned_histogram_kernelI" + arguments + "E" in name]
    assert len(match) == 1
    assert match[0].get(".vgpr_spill_count", 0) <= spilled


def test_scans_that_decide_use_no_scratch_memory(kernels):
    """They ask for all that they read before the first answer is waited for; what is kept in scratch memory is waited for."""
    match = [k for name, k in kernels.items() if "small_scan_kernelI" in name and "ELb1ELb1EE" in name]
    assert len(match) == 3
    assert [k[".private_segment_fixed_size"] for k in match] == [0, 0, 0]


def test_histogram_kernels_that_address_the_lds_from_0_have_no_static_lds(kernels):
    """Their launch refuses to run otherwise: this is where a __shared__ variable too many shows."""
    match = [k for name, k in kernels.items() if "binned_histogram_kernelIhLi16E" in name and re.search("ELb1ELi1[2346]EE", name)]
    assert len(match) == 14
    assert {k[".group_segment_fixed_size"] for k in match} == {0}
