"""Inline assembly states what it overwrites: a statement that writes m0 lists it as clobbered, else the
compiler may keep a value of its own there across it."""
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def statements(text):
    """The asm statements of a source, macros they take included (one level, by textual use)."""
    macros = dict(re.findall(r"#define (\w+)((?:[^\n]*\\\n)*[^\n]*)", text))
    for m in re.finditer(r"\basm volatile\(", text):
        s = text[m.start():text.index(";", m.end())]
        yield s + "".join(body for name, body in macros.items() if re.search(rf"\b{name}\b", s))


def test_m0_is_listed():
    seen = 0
    for path in glob.glob(os.path.join(ROOT, "kestrel-llm_amd", "csrc", "*")):
        for s in statements(open(path).read()):
            if re.search(r"\bm0,", s):
                seen += 1
                assert '"m0"' in s, (path, s[:120])
    assert seen >= 2
