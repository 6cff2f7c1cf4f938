"""What the compiler made of the resident kernels, from the library's own code objects.  The
rules that place LSRK registers in LDS and that choose between resident and stage launches
(resident_lds_k, resident_range) rest on which kernels spill: another compiler that spills
more makes them wrong, and this fails."""
import os
import re
import struct

import msgpack
import pytest

from nekwave_amd import _lib

EM_AMDGPU, SHT_NOTE, NT_AMDGPU_METADATA = 224, 7, 32


def _kernels():
    data = open(_lib.LIB_PATH, "rb").read()
    out = {}
    at = data.find(b"\x7fELF", 1)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == EM_AMDGPU:
            shoff = struct.unpack_from("<Q", data, at + 40)[0]
            size, count = struct.unpack_from("<HH", data, at + 58)
            for s in range(count):
                kind = struct.unpack_from("<I", data, at + shoff + s * size + 4)[0]
                off, length = struct.unpack_from("<QQ", data, at + shoff + s * size + 24)
                p, end = at + off, at + off + length
                while kind == SHT_NOTE and p < end:
                    namesz, descsz, typ = struct.unpack_from("<III", data, p)
                    desc = p + 12 + (namesz + 3) // 4 * 4
                    if typ == NT_AMDGPU_METADATA:
                        for k in msgpack.unpackb(data[desc:desc + descsz], raw=False)["amdhsa.kernels"]:
                            out[k[".name"]] = k
                    p = desc + (descsz + 3) // 4 * 4
        at = data.find(b"\x7fELF", at + 4)
    return out


@pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="library not built")
def test_resident_kernels_spill_no_more_than_the_rules_assume():
    seen = 0
    for name, k in _kernels().items():
        m = re.search(r"k_residentILi(\d+)ELi(\d+)E(\w)(\w)Lb(\d)", name)
        if not m:
            continue
        seen += 1
        em, scratch = int(m.group(2)), k[".private_segment_fixed_size"]
        # bytes per thread: with four and eight elements per workgroup kernels of 72 win and of
        # 88 lose against stage launches; with one and two those of 124 win (n1 = 9, FP64)
        assert scratch <= (80 if em >= 4 else 128), (name, scratch)
        assert k[".group_segment_fixed_size"] <= 160 * 1024
    assert seen >= 100
