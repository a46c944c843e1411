"""Inline assembly that needs m0 (global loads into LDS take their LDS address from it)
says so, as an operand or as overwritten: the compiler keeps values of its own there and
does not look into the text."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "quantumbilliards.jl_amd", "csrc")


def _statements(src):
    for m in re.finditer(r"\basm\s*(?:volatile\s*)?\(", src):
        depth, i = 1, m.end()
        while depth:
            depth += {"(": 1, ")": -1}.get(src[i], 0)
            i += 1
        yield src[m.end():i - 1]


def test_m0_is_declared():
    seen = 0
    for f in sorted(glob.glob(os.path.join(CSRC, "*.h*"))):
        for s in _statements(open(f).read()):
            if not re.search(r"\bm0\s*,|_load_lds_", s):
                continue
            seen += 1
            written = re.search(r"\bs_\w+\s+m0\s*,", s)
            ok = '"m0"' in s.rsplit(":", 1)[-1] if written else '"{m0}"(' in s
            assert ok, (os.path.basename(f), s)
    assert seen
