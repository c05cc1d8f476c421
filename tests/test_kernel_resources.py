"""CPU: no kernel of the built library uses scratch memory.

A register spilled to scratch costs a memory access on the path between a
kernel's loads, which is where these kernels spend their time, and nothing in
their results shows it.  Read from the code objects' own metadata."""

import re

from akas_amd import _lib


def _uint(blob):
    """First MessagePack unsigned integer of ``blob``."""
    width = {0xCC: 1, 0xCD: 2, 0xCE: 4, 0xCF: 8}.get(blob[0])
    return blob[0] if width is None else int.from_bytes(blob[1:1 + width], "big")


def kernels(path=_lib.LIBRARY):
    """(name, scratch bytes per lane) of every kernel: the metadata's keys are
    sorted, so the size follows the name."""
    data = open(path, "rb").read()
    pattern = rb"\xa5\.name(?:[\xa0-\xbf]|\xd9.|\xda..)(_Z\w+)\xbb\.private_segment_fixed_size"
    found = []
    for m in re.finditer(pattern, data, re.S):
        found.append((m.group(1).decode(), _uint(data[m.end():m.end() + 9])))
    return found


def test_no_kernel_uses_scratch():
    found = kernels()
    assert len(found) > 100  # the pattern still matches the metadata
    assert [k for k in found if k[1]] == []
