"""Inline assembly of the kernels, read as text: a statement that writes m0
names it as clobbered (the compiler may keep a value of its own there), and
clobbers memory, since what such statements start reads or writes it."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mimir-model_amd", "csrc")


def asm_statements(text):
    """The parenthesised text of every asm statement."""
    for m in re.finditer(r"\basm\s+volatile\s*\(", text):
        depth, i, quoted = 1, m.end(), False
        while depth:
            c = text[i]
            if c == '"' and text[i - 1] != "\\":
                quoted = not quoted
            elif not quoted:
                depth += (c == "(") - (c == ")")
            i += 1
        yield text[m.end():i - 1]


def test_m0_is_clobbered():
    seen = 0
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h*")) + glob.glob(os.path.join(CSRC, "*.cpp"))):
        for stmt in asm_statements(open(path).read()):
            if re.search(r"\bs_mov_b32 m0\b", stmt):
                seen += 1
                clobbers = re.findall(r'"(\w+)"', stmt.rsplit(":", 1)[1])
                assert {"m0", "memory"} <= set(clobbers), f"{os.path.basename(path)}: {stmt}"
    assert seen > 0
