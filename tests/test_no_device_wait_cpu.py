"""No kernel waits for another workgroup: workgroups that share an item store
their partial results and count themselves, and the one that counts last sums
them.  A wait for a word in memory would hang the device where that word is
uncleared or belongs to an overlapping call (the allocation-free entry's scratch
is one array per device)."""

import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flash-attention-turing_amd", "csrc")


def test_no_kernel_polls_memory():
    sources = sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h")))
    assert len(sources) >= 5
    for path in sources:
        code = re.sub(r"//[^\n]*|/\*.*?\*/", "", open(path).read(), flags=re.S)
        assert "s_sleep" not in code, path
        for loop in re.finditer(r"\bwhile\s*\(", code):
            depth, end = 1, loop.end()
            while depth:
                depth += {"(": 1, ")": -1}.get(code[end], 0)
                end += 1
            assert not re.search(r"atomic|volatile", code[loop.end():end]), f"{path}: {code[loop.start():end]}"
