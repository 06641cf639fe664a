"""The device code in the built library, from its own metadata (no GPU needed):
no kernel keeps arrays in scratch memory, and none spills registers."""
import struct

import pytest

from mfrbf import _lib as L

EM_AMDGPU, SHT_NOTE, NT_AMDGPU_METADATA = 224, 7, 32


def code_objects(blob):
    """The AMDGPU ELF files embedded in the library."""
    at = blob.find(b"\x7fELF", 4)
    while at >= 0:
        if len(blob) > at + 64 and struct.unpack_from("<H", blob, at + 18)[0] == EM_AMDGPU:
            yield at
        at = blob.find(b"\x7fELF", at + 4)


def kernels(blob, base, msgpack):
    shoff, = struct.unpack_from("<Q", blob, base + 40)
    size, count = struct.unpack_from("<HH", blob, base + 58)
    for q in range(count):
        kind, _, _, off, length = struct.unpack_from("<IQQQQ", blob, base + shoff + q * size + 4)
        if kind != SHT_NOTE:
            continue
        at, end = base + off, base + off + length
        while at + 12 <= end:
            nname, ndesc, ntype = struct.unpack_from("<III", blob, at)
            desc = at + 12 + (nname + 3) // 4 * 4
            if ntype == NT_AMDGPU_METADATA:
                yield from msgpack.unpackb(blob[desc:desc + ndesc])["amdhsa.kernels"]
            at = desc + (ndesc + 3) // 4 * 4


def test_kernels_use_no_scratch_memory():
    msgpack = pytest.importorskip("msgpack")
    with open(L.LIB_PATH, "rb") as f:
        blob = f.read()
    found = [k for base in code_objects(blob) for k in kernels(blob, base, msgpack)]
    assert len(found) > 300  # the stencil kernels alone
    bad = [(k[".name"], k[".private_segment_fixed_size"]) for k in found
           if k[".name"].startswith("_ZN2mf") and (k[".private_segment_fixed_size"] or k[".vgpr_spill_count"])]
    assert not bad
