"""No inline assembly in the kernels accesses memory or multiplies matrices: the compiler does not see what it is, and puts no
wait states around it (gfx950 wants two before a vector instruction may write the registers of a 16-byte store)."""
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
