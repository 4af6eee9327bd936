"""Inline assembly in the kernels: a load that the compiler does not wait for must not have a register of the compiler's
for its result, which it may copy or spill before the data is there.  (Into LDS it may go: reads of that are ordered by
the asm's memory clobber.)"""
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "sparseconvnet-archived_amd", "csrc")


def statements(text):
    """(instructions, rest) of every asm statement: its string literals up to the first colon, what follows"""
    for m in re.finditer(r"\basm\s*(?:volatile\s*)?\(", text):
        depth, at = 1, m.end()
        while depth:
            if text[at] == '"':
                at = re.compile(r'"(?:[^"\\]|\\.)*"').match(text, at).end()
                continue
            depth += {"(": 1, ")": -1}.get(text[at], 0)
            at += 1
        body = text[m.end():at - 1]
        head = re.match(r'\s*(?:"(?:[^"\\]|\\.)*"\s*)*', body).group(0)
        yield head, body[len(head):]


def test_no_load_into_a_register():
    found = 0
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h"))):
        for code, rest in statements(open(path).read()):
            found += 1
            if "load" in code or "ds_read" in code:
                assert not re.search(r'"=[^"]*"', rest), "%s: %s%s" % (os.path.basename(path), code, rest)
                assert '"memory"' in rest, "%s: %s%s" % (os.path.basename(path), code, rest)
    assert found >= 5
