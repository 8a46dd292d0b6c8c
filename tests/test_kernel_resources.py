"""What the compiler made of the kernels: none keeps registers in memory (a lane's scratch is a trip to memory in the
loops these kernels are about)."""
import os
import re
import struct
import subprocess

import pytest

from vtl_amd import capi

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(library):
    """The gfx950 code objects of a library: each bundle has a table of (offset, size, target)."""
    for bundle in re.finditer(MAGIC, library):
        at = bundle.start() + len(MAGIC)
        count, = struct.unpack_from("<Q", library, at)
        at += 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", library, at)
            target = library[at + 24:at + 24 + length]
            at += 24 + length
            if b"gfx950" in target:
                yield library[bundle.start() + offset:bundle.start() + offset + size]


@pytest.mark.skipif(not os.path.exists(READELF), reason="needs llvm-readelf")
def test_no_kernel_spills(tmp_path):
    found, spilled = 0, []
    for i, code in enumerate(_code_objects(open(capi.LIB_PATH, "rb").read())):
        path = tmp_path / f"{i}.o"
        path.write_bytes(code)
        notes = subprocess.run([READELF, "--notes", str(path)], stdout=subprocess.PIPE, text=True, check=True).stdout
        for kernel in notes.split("- .agpr_count")[1:]:
            value = {k: v for k, v in re.findall(r"\.(\w+): +(\S+)", kernel)}
            found += 1
            if int(value["private_segment_fixed_size"]) or int(value["vgpr_spill_count"]):
                spilled.append((value["name"], value["vgpr_spill_count"], value["private_segment_fixed_size"]))
    assert found > 100 and not spilled, spilled
