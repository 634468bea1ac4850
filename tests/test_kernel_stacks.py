"""What the compiler says of the built kernels (the notes of the code objects inside the libraries): an array of a thread lies in registers, not in memory."""
import os
import struct

import msgpack
import pytest

from poptransformer_amd import _hybrid_lib, _lib, build

AMDGPU, NOTE, METADATA = 224, 7, 32                   # ELF machine, section type, note type


def kernels(path):
    """The metadata of every gfx950 kernel of a library."""
    with open(path, "rb") as f:
        data = f.read()
    at = data.find(b"\x7fELF", 1)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == AMDGPU:
            sections, = struct.unpack_from("<Q", data, at + 40)
            size, count = struct.unpack_from("<HH", data, at + 58)
            for section in range(at + sections, at + sections + count * size, size):
                if struct.unpack_from("<I", data, section + 4)[0] != NOTE:
                    continue
                offset, length = struct.unpack_from("<QQ", data, section + 24)
                p = at + offset
                while p < at + offset + length:
                    name, bytes_, kind = struct.unpack_from("<III", data, p)
                    p += 12 + (name + 3) // 4 * 4
                    if kind == METADATA:
                        yield from msgpack.unpackb(data[p:p + bytes_])["amdhsa.kernels"]
                    p += (bytes_ + 3) // 4 * 4
        at = data.find(b"\x7fELF", at + 1)


@pytest.mark.parametrize("lib", [_lib, _hybrid_lib], ids=["operators", "hybrid"])
def test_no_array_of_a_thread_is_kept_in_memory(lib):
    """Memory of a thread's own that is no register spilled is an array that the compiler could not take apart, as behind a lambda that it did not inline: 2.4 times the
    time of a prompt's attention.  (beam_update_kernel sorts in one.)"""
    if not os.path.exists(lib.LIB_PATH):
        build.build(force=False)
    found = list(kernels(lib.LIB_PATH))
    assert len(found) > 100
    stacks = {k[".name"] for k in found if k[".private_segment_fixed_size"] and not k[".vgpr_spill_count"]}
    assert not [name for name in stacks if "beam_update_kernel" not in name]
