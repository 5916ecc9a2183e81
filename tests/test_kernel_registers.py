"""Register use of the built kernels, from the metadata of this build's own code
objects (CPU)."""

from __future__ import annotations

import re
import struct

import pytest

msgpack = pytest.importorskip("msgpack")


def _kernels():
    """{kernel name: metadata} of the gfx950 code objects in the built library."""
    import os
    from sophia_amd import _native
    if not os.path.exists(_native.LIB_PATH):
        pytest.skip("HIP library not built (run `python -m sophia_amd.build`)")
    data = open(_native.LIB_PATH, "rb").read()
    found = {}
    for bundle in (m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)):
        entries, at = struct.unpack_from("<Q", data, bundle + 24)[0], bundle + 32
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            target, at = data[at + 24:at + 24 + length].decode(), at + 24 + length
            if "gfx950" not in target:
                continue
            elf = data[bundle + offset:bundle + offset + size]
            table, (entry, count) = struct.unpack_from("<Q", elf, 0x28)[0], struct.unpack_from("<HH", elf, 0x3A)
            for s in range(count):
                _, kind, _, _, where, *_ = struct.unpack_from("<IIQQQQ", elf, table + s * entry)
                if kind == 7:   # notes: name size, descriptor size, type, name, descriptor
                    name, desc, _ = struct.unpack_from("<III", elf, where)
                    body = where + 12 + (name + 3 & ~3)
                    for k in msgpack.unpackb(elf[body:body + desc])["amdhsa.kernels"]:
                        found[k[".name"]] = k
    assert found
    return found


def test_projection_kernels_hold_their_batches_in_registers():
    """Every form of the few-row and per-head projections keeps the loads that it
    issues together in registers (a spilled load is waited for, written and read
    back)."""
    rows = {n: k for n, k in _kernels().items() if "row_linear_kernel" in n or "head_linear_kernel" in n}
    assert len(rows) > 50
    assert {n: k[".private_segment_fixed_size"] for n, k in rows.items() if k[".private_segment_fixed_size"]} == {}
