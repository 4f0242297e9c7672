"""Inline assembly names the registers it writes: m0 and vcc wherever an instruction sets them."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "backprojector_amd", "csrc")


def asm_statements():
    for path in glob.glob(os.path.join(CSRC, "*.h*")):
        text = open(path).read()
        for m in re.finditer(r"\basm(?: volatile)?\(", text):
            depth, i = 1, m.end()
            while depth:
                depth += {"(": 1, ")": -1}.get(text[i], 0)
                i += 1
            yield os.path.basename(path), text[m.end():i - 1]


def test_written_registers_are_clobbered():
    found = {"m0": 0, "vcc": 0}
    for where, stmt in asm_statements():
        code, clobbers = stmt.rpartition(":")[::2]
        for reg, writes in (("m0", r"\bs_\w+ m0,"), ("vcc", r"\bv_cmp_\w+ vcc,")):
            if re.search(writes, code):
                found[reg] += 1
                assert f'"{reg}"' in clobbers, (where, stmt)
    assert all(found.values()), found
