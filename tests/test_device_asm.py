"""Inline assembly of the device code that writes M0, read from the sources (no GPU): the compiler inserts no wait states into
inline assembly, and a load into LDS that follows a write of M0 needs one between them; the statement declares that it writes M0."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cubework_amd", "csrc")


def test_loads_into_lds_wait_for_m0():
    found = 0
    for path in glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip")):
        with open(path) as f:
            source = f.read()
        for statement in re.findall(r"\basm\b[^;]*?\(.*?\)\s*;", source, re.S):
            code = "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', statement.split(":")[0]))
            lines = [line.strip() for line in re.split(r"\\n\\t|\\n|;", code) if line.strip()]
            for i, line in enumerate(lines):
                if re.match(r"s_mov_b32\s+m0\b", line):
                    found += 1
                    assert lines[i + 1].startswith("s_nop"), "%s: no wait state behind %s" % (path, line)
                    assert '"m0"' in statement, "%s: M0 is not declared as written: %s" % (path, statement)
    assert found >= 2
