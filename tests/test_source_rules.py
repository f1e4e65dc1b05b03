"""Rules of the kernel sources that no compiler checks (CPU only)."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qppocr_amd", "csrc")
SOURCES = sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h")))


@pytest.mark.parametrize("path", SOURCES, ids=os.path.basename)
def test_m0_write_is_followed_by_a_wait_state(path):
    """A scalar write of m0 needs one wait state before a load to LDS that
    reads it; the compiler inserts it for its own code, not inside an asm."""
    text = open(path).read()
    for m in re.finditer(r"s_mov_b32 m0,[^\\\"]*((?:\\n\\t[^\\\"]*)?)", text):
        line = text.count("\n", 0, m.start()) + 1
        assert m.group(1).startswith("\\n\\ts_nop"), f"{os.path.basename(path)}:{line}"
