"""No kernel of the built library spills vector registers.

The compiler places a vector register's spill at the start of the block where
diverged lanes join again, before it turns them on: lanes lose the value, and
the kernel's results depend on what the scratch memory held.  The counts stand
in the metadata of the library's code objects (a msgpack map per kernel)."""
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "2degas_amd", "lib2degas_hip.so")


def _spills(blob):
    out = []
    key = b".vgpr_spill_count"
    at = blob.find(key)
    while at >= 0:
        sym = re.findall(rb"\.symbol[\xa0-\xbf\xd9\xda][\x00-\xff]{0,2}?(_?[A-Za-z0-9_]+)\.kd", blob[max(0, at - 4096):at])
        b = blob[at + len(key)]
        n = b if b < 0x80 else int.from_bytes(blob[at + len(key) + 1:at + len(key) + 1 + (1 << (b - 0xcc))], "big")
        out.append((sym[-1].decode() if sym else "?", n))
        at = blob.find(key, at + 1)
    return out


def test_no_kernel_spills_vector_registers():
    if not os.path.exists(LIB):
        pytest.skip("library not built")
    found = _spills(open(LIB, "rb").read())
    assert len(found) > 20
    bad = [(k, n) for k, n in found if n]
    assert not bad, bad
