"""CPU: which kernels of the built library use scratch memory (the metadata the
compiler writes beside this repository's kernels). A choice between two vectors,
or an indexed register array, quietly becomes a trip through memory; only the
kernels named here are allowed one."""
import re

from pyroclastmpm_amd import capi

# stand-alone return maps (every material in one kernel); the 3D adjoint G2P's return-map adjoint
ALLOWED = ("stress_update_kernel", "18g2p_adjoint_kernelILi3E")


def _scratch():
    data = open(capi.LIB_PATH, "rb").read()
    # msgpack: ".name" <string> ".private_segment_fixed_size" <unsigned>
    found = {}
    for m in re.finditer(rb"\xa5\.name(?:[\xa0-\xbf]|\xd9.|\xda..)([\x20-\x7e]+)\xbb\.private_segment_fixed_size(.)(..?)", data,
                         re.S):
        kind, rest = m.group(2)[0], m.group(3)
        size = kind if kind < 0x80 else {0xcc: rest[0], 0xcd: int.from_bytes(rest[:2], "big")}[kind]
        found[m.group(1).decode()] = size
    return found


def test_no_kernel_but_the_named_uses_scratch():
    sizes = _scratch()
    assert len(sizes) > 100 and any("p2g_adjoint3_kernel" in k for k in sizes)
    assert any(v for v in sizes.values())  # (the metadata is read at all)
    users = {k: v for k, v in sizes.items() if v and not any(a in k for a in ALLOWED)}
    assert not users, users
