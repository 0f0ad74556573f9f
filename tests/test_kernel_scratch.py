"""Scratch memory of the kernels that hold their state in registers, from the built library's own code
objects: a few spilled registers at most, never the state itself."""
import struct

import pytest

from convstencil_amd import _lib

msgpack = pytest.importorskip("msgpack")


def _kernels():
    """name -> metadata of every gfx950 kernel in the library."""
    data = open(_lib.LIB_PATH, "rb").read()
    out, at = {}, data.find(b"\x7fELF", 4)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == 224:  # EM_AMDGPU
            shoff, = struct.unpack_from("<Q", data, at + 40)
            size, count = struct.unpack_from("<HH", data, at + 58)
            for i in range(count):
                head = at + shoff + i * size
                kind, = struct.unpack_from("<I", data, head + 4)
                off, length = struct.unpack_from("<QQ", data, head + 24)
                if kind == 7:  # SHT_NOTE
                    name, desc, _ = struct.unpack_from("<III", data, at + off)
                    start = at + off + 12 + (name + 3) // 4 * 4
                    meta = msgpack.unpackb(data[start:start + desc])
                    out.update({k[".name"]: k for k in meta["amdhsa.kernels"]})
        at = data.find(b"\x7fELF", at + 4)
    return out


KERNELS = _kernels()


@pytest.mark.parametrize("family", ["k2d_pipe", "k2d_block", "k3d_tile"])
def test_state_is_not_in_scratch(family):
    found = {n: k for n, k in KERNELS.items() if family in n}
    assert len(found) >= 10
    # the smallest state, one level of the radius-1 pipeline, is 24 partial sums a lane: 192 bytes
    bad = {n: k[".private_segment_fixed_size"] for n, k in found.items() if k[".private_segment_fixed_size"] >= 192}
    assert not bad
