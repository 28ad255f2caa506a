"""CPU: what the compiler's metadata in the built library says of kernels' registers."""
import os
import re
import struct

import pytest

from leviathan_amd import capi


def kernels():
    """{mangled name: its metadata} of every code object in the library (the note of an AMD GPU ELF is msgpack)."""
    msgpack = pytest.importorskip("msgpack")
    if not os.path.exists(capi.LIB_PATH):
        pytest.skip("library not built")
    with open(capi.LIB_PATH, "rb") as f:
        data = f.read()
    found = {}
    for m in re.finditer(b"\x7fELF", data):
        at = m.start()
        if struct.unpack_from("<H", data, at + 18)[0] != 224:       # EM_AMDGPU
            continue
        shoff, = struct.unpack_from("<Q", data, at + 40)
        shentsize, shnum = struct.unpack_from("<HH", data, at + 58)
        for k in range(shnum):
            head = at + shoff + k * shentsize
            kind, = struct.unpack_from("<I", data, head + 4)
            offset, size = struct.unpack_from("<QQ", data, head + 24)
            if kind != 7:                                            # SHT_NOTE
                continue
            note = at + offset
            while note < at + offset + size:
                namesz, descsz, _ = struct.unpack_from("<III", data, note)
                desc = note + 12 + (namesz + 3 & ~3)
                meta = msgpack.unpackb(data[desc:desc + descsz], strict_map_key=False)
                found.update({kernel[".name"]: kernel for kernel in meta.get("amdhsa.kernels", [])})
                note = desc + (descsz + 3 & ~3)
    assert found
    return found


@pytest.mark.parametrize("pattern", ["moe_gate_up_mfma", "moe_pf_kernel"])
def test_kernels_keep_their_registers(pattern):
    """The time of these kernels is what a wave issues and waits for: nothing of them goes through scratch memory."""
    mine = {name: k for name, k in kernels().items() if pattern in name}
    assert mine
    assert {name: k[".vgpr_spill_count"] for name, k in mine.items() if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]} == {}
