"""What the compiler made of the library's own kernels, read from the built library: the waits of a ring of LDS-DMA requests name the number of requests that may stay
in flight, and a wait for all of them, which gives the same results, would be seen by no other test."""
import os
import re
import struct
import subprocess

import pytest

import trackiellm_amd as tk

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
LIB = os.path.join(os.path.dirname(tk.__file__), "libtrackie_mi355x.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(data):
    """the gfx950 parts of the bundles: per bundle a count of entries, each {offset, size, length of the target's name, name}"""
    at = data.find(MAGIC)
    while at >= 0:
        n, p = struct.unpack_from("<Q", data, at + len(MAGIC))[0], at + len(MAGIC) + 8
        for _ in range(n if n < 16 else 0):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + length]
            p += 24 + length
            if b"gfx950" in name:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + 1)


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
def test_the_value_ring_of_a_long_context_waits_for_one_chunk(tmp_path):
    with open(LIB, "rb") as f:
        data = f.read()
    found = {}
    for i, code in enumerate(code_objects(data)):
        if b"k_att_pv_chain" not in code:
            continue
        path = tmp_path / ("%d.co" % i)
        path.write_bytes(code)
        names = ["_Z14k_att_pv_chainILi%dELi%dEEvPKfPKtPKiS5_iiiiiPfS6_" % f for f in ((128, 3), (128, 2), (64, 3), (64, 2))]
        text = subprocess.run([OBJDUMP, "-d", "--disassemble-symbols=" + ",".join(names), str(path)], capture_output=True, text=True, check=True).stdout
        for m in re.finditer(r"<_Z14k_att_pv_chainILi(\d+)ELi(\d)E\w*>:\n(.*?)(?=\n\n|\Z)", text, re.S):
            found[int(m[1]), int(m[2])] = {int(v) for v in re.findall(r"s_waitcnt vmcnt\((\d+)\)", m[3])}
    assert set(found) == {(128, 3), (128, 2), (64, 3), (64, 2)}
    for (dim, slots), waits in found.items():
        requests = dim // 8  # of a chunk: 64 rows of `dim` halves, 1 KiB each
        assert waits == {k * requests for k in range(slots)}, (dim, slots, waits)
