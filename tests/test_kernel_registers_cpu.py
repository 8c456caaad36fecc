"""What the built kernels' own descriptions say about scratch memory (no GPU): the notes of the gfx950 code objects inside the two libraries."""
import os
import struct

import msgpack
import pytest

from tests.conftest import load_pkg

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dash-infer_amd", "lib")


def kernels(path):
    """name -> (bytes of scratch memory a lane, spilled vector registers) of every kernel in the library's device code"""
    d, out, at = open(path, "rb").read(), {}, 0
    while (i := d.find(b"\x7fELF\x02\x01\x01\x40", at)) >= 0:          # (64 bits, little endian, the OS ABI of AMD's device code)
        at = i + 4
        headers, (size, count) = struct.unpack_from("<Q", d, i + 0x28)[0], struct.unpack_from("<HH", d, i + 0x3A)
        for k in range(count):
            b = i + headers + k * size
            if struct.unpack_from("<I", d, b + 4)[0] != 7:               # a section of notes
                continue
            p = i + struct.unpack_from("<Q", d, b + 0x18)[0]
            name, length, kind = struct.unpack_from("<III", d, p)
            if kind == 32:                                               # the metadata of code objects, in MessagePack
                p += 12 + (name + 3 & ~3)
                for x in msgpack.unpackb(d[p:p + length], strict_map_key=False)["amdhsa.kernels"]:
                    out[x[".name"]] = (x[".private_segment_fixed_size"], x.get(".vgpr_spill_count", 0))
    return out


@pytest.mark.parametrize("name,least", [("libdashinfer_hip_seq.so", 400), ("libdashinfer_hip.so", 600)])
def test_no_kernel_keeps_an_array_in_scratch_memory(name, least):
    """Scratch memory without spilled registers is an array with an index that the compiler does not know -- a loop over sums that it did not unroll; such a kernel took 3.6 times as long."""
    load_pkg()
    found = kernels(os.path.join(LIB, name))
    assert len(found) >= least
    assert not {k: v for k, v in found.items() if v[0] and not v[1]}
