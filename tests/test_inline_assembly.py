"""Inline assembly says which registers it writes: m0, the LDS base of the
direct copies, can hold a value of the compiler's."""
import glob
import os
import re

from gprat_amd import build


def test_statements_that_write_m0_name_it():
    statements = []
    for path in glob.glob(os.path.join(build.CSRC, "*.h*")):
        with open(path) as f:
            for s in re.findall(r"\basm\b(?: volatile)?\((.*?)\);\n", f.read(), re.S):
                text = s.split("\n")[0]
                if re.search(r"s_\w+ m0\b", text):
                    statements.append((os.path.basename(path), s))
    assert len(statements) >= 2
    for path, s in statements:
        assert '"m0"' in s.split(":")[-1], (path, s)
