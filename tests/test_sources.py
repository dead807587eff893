"""What the kernels' inline assembly has to tell the compiler, read from the
sources (CPU)."""
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = sorted(glob.glob(os.path.join(ROOT, "midge_amd", "csrc", "*")))


def asm_statements():
    for path in CSRC:
        with open(path) as f:
            text = f.read()
        for m in re.finditer(r"\basm\s+(?:volatile\s*)?\(", text):
            depth, i, quoted = 1, m.end(), False
            while depth:
                c = text[i]
                if c == '"' and text[i - 1] != "\\":
                    quoted = not quoted
                elif not quoted:
                    depth += (c == "(") - (c == ")")
                i += 1
            yield os.path.basename(path), text[m.end():i - 1]


def test_m0_is_set_by_the_compiler():
    """m0 holds the LDS address of a memory-to-LDS load. The compiler may keep
    a value of its own there, so no statement writes it, and every statement
    that reads it says so with an operand."""
    loads = [(f, s) for f, s in asm_statements() if re.search(r"_load_lds_", s)]
    assert len(loads) >= 4
    for f, s in loads:
        assert '"{m0}"(' in s, (f, s)
    for f, s in asm_statements():
        assert not re.search(r"\bm0\s*,", s), (f, s)
