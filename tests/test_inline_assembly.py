"""No inline assembly in the kernels accesses memory or multiplies matrices: the compiler does not see what it is, and puts no
wait states around it (gfx950 wants two before a vector instruction may write the registers of a 16-byte store).  Nor does it behind a
16-byte buffer store, made by a builtin, whose scalar offset is a register: such a store has the wait states written behind it."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vtl_amd", "csrc")


@pytest.mark.parametrize("path", sorted(glob.glob(CSRC + "/*.h*")), ids=os.path.basename)
def test_inline_assembly_needs_no_wait_states(path):
    for text in re.findall(r'\basm\s*(?:volatile)?\s*\(\s*((?:"[^"]*"\s*)+)', open(path).read()):
        text = "".join(re.findall(r'"([^"]*)"', text))
        assert not re.search(r"store|load|atomic|mfma", text), text


def wide_stores(text):
    """Of each buffer store of 12 or 16 bytes: its scalar offset, and what comes behind it up to the end of its function."""
    for call in re.finditer(r"raw_buffer_store_b(?:96|128)\s*\(", text):
        depth, at, args = 1, call.end(), [""]
        while depth:
            c = text[at]
            depth += (c in "({[") - (c in ")}]")
            if c == "," and depth == 1:
                args.append("")
            elif depth:
                args[-1] += c
            at += 1
        assert len(args) == 5, args      # value, buffer, a lane's offset, the scalar offset, cache policy
        yield args[3].strip(), re.sub(r"//[^\n]*\n", "", text[at:text.index("\n}", at)])


GUARD = r"\s*;\s*__builtin_amdgcn_sched_barrier\(0\);\s*asm volatile\(\"s_nop [1-9]\"\);\s*__builtin_amdgcn_sched_barrier\(0\);"


@pytest.mark.parametrize("path", sorted(glob.glob(CSRC + "/*.h*")), ids=os.path.basename)
def test_wide_stores_with_a_scalar_offset_wait(path):
    for offset, behind in wide_stores(open(path).read()):
        assert offset == "0" or re.match(GUARD, behind), (offset, behind[:200])


def test_wide_stores_are_found():
    assert [o for o, _ in wide_stores(open(CSRC + "/common.hpp").read())] == ["0"]
    assert [o for o, _ in wide_stores(open(CSRC + "/matmul_f64acc.hip").read())] == ["along"]
    planted = "{\n    __builtin_amdgcn_raw_buffer_store_b128(v, b, off, along, 0);\n    v[0] = 1;\n}\n"
    (offset, behind), = wide_stores(planted)
    assert offset == "along" and not re.match(GUARD, behind)
