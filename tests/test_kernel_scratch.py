"""Kernels that many workgroups run must not use scratch memory: it slows down the start of every workgroup, those without
work included (20 bytes of it: 3 us for a launch of 8 704 workgroups without work)."""
import os
import re
import struct

import msgpack
import pytest

from mako_amd import api

# (the instances for logits loaded one at a time, for histories of more than 8 192 entries and for large batches hold more
# than fits)
NONE = re.compile(r"(scan_kernelI|index_weights_kernelI|index_groups_kernelI|sort_kernelE|sort_kernel_unsortedE|sort_beside_kernelI"
                  r"|finish_kernelILb1ELi2|finish_beside_kernelILb1ELi2)")


def _code_objects(data):
    """The AMD GPU ELF files inside a shared library's bytes."""
    at = data.find(b"\x7fELF", 4)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == 224:  # EM_AMDGPU
            size = struct.unpack_from("<Q", data, at + 40)[0] + struct.unpack_from("<H", data, at + 60)[0] * struct.unpack_from("<H", data, at + 58)[0]
            yield data[at:at + size]
        at = data.find(b"\x7fELF", at + 4)


def _kernels(elf):
    """{mangled name: bytes of scratch memory} from the metadata note."""
    off, size, count = struct.unpack_from("<Q", elf, 40)[0], *struct.unpack_from("<HH", elf, 58)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, off + i * size + 4)
        start, length = struct.unpack_from("<QQ", elf, off + i * size + 24)
        if kind != 7:  # SHT_NOTE
            continue
        n, d, t = struct.unpack_from("<III", elf, start)
        desc = elf[start + 12 + (n + 3) // 4 * 4:][:d]
        if t == 32:  # NT_AMDGPU_METADATA
            return {k[".name"]: k[".private_segment_fixed_size"] for k in msgpack.unpackb(desc)["amdhsa.kernels"]}
    return {}


def test_kernels_of_many_workgroups_use_no_scratch_memory():
    if not os.path.exists(api.LIB_PATH):
        pytest.skip("the library is not built")
    with open(api.LIB_PATH, "rb") as f:
        data = f.read()
    found = {}
    for elf in _code_objects(data):
        found.update(_kernels(elf))
    many = {k: v for k, v in found.items() if NONE.search(k)}
    assert len(many) > 20, sorted(found)
    assert not {k: v for k, v in many.items() if v}, {k: v for k, v in many.items() if v}


def test_the_tail_of_the_whole_row_path_is_a_call():
    # (in line, the path to it is a call longer, and a third slower for rows with few survivors)
    if not os.path.exists(api.LIB_PATH):
        pytest.skip("the library is not built")
    with open(api.LIB_PATH, "rb") as f:
        elves = [e for e in _code_objects(f.read()) if any("index_tail_kernel" in k for k in _kernels(e))]
    assert elves
    for elf in elves:
        assert b"\0_ZN4mako11sorted_tailILb0ELb0ELb0ELb0ELb0EEE" in elf
        assert b"\0_ZN4mako18sort_truncate_drawILb1EEE" not in elf
