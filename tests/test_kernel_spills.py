"""No kernel of the library spills vector registers, read from the built code objects' own metadata.

The compiler has put such a spill at the head of a join block, before the lanes of the other branch were back:
only some lanes' values were kept (thread indices, which the candidate search then took from garbage).
"""
import re
import subprocess
from pathlib import Path

import pytest

LIB = Path(__file__).resolve().parents[1] / "lsdem2.0_amd" / "liblsdem.so"
READELF = Path("/opt/rocm/llvm/bin/llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    """The gfx950 code objects of every offload bundle in the library."""
    at = data.find(MAGIC)
    while at >= 0:
        pos = at + len(MAGIC)
        n = int.from_bytes(data[pos:pos + 8], "little")
        pos += 8
        for _ in range(n):
            off, size, length = (int.from_bytes(data[pos + 8 * k:pos + 8 * k + 8], "little") for k in range(3))
            if b"gfx950" in data[pos + 24:pos + 24 + length]:
                yield data[at + off:at + off + size]
            pos += 24 + length
        at = data.find(MAGIC, at + 1)


@pytest.mark.skipif(not READELF.exists(), reason="llvm-readelf is not installed")
def test_no_vector_register_spills(tmp_path):
    spills = {}
    for k, obj in enumerate(_code_objects(LIB.read_bytes())):
        path = tmp_path / f"{k}.o"
        path.write_bytes(obj)
        notes = subprocess.run([str(READELF), "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for kernel in re.split(r"\n  - ", notes)[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel)
            count = re.search(r"\.vgpr_spill_count:\s+(\d+)", kernel)
            if name and count:
                spills[name.group(1)] = int(count.group(1))
    assert any("k_broad_phase" in k for k in spills) and any("k_candidates" in k for k in spills)
    assert {k: v for k, v in spills.items() if v} == {}
