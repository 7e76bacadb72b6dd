"""Inline assembly of the device sources: a register that a statement's text names itself is one the compiler does not see, so each
such register has to be among the statement's operands or clobbers."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "n2d2_amd", "csrc")
FIXED = r"\b(?:m0|vcc(?:_lo|_hi)?|exec(?:_lo|_hi)?|[sv]\d+|[sv]\[\d+:\d+\])\b"


def _statements(text):
    """(template, operands and clobbers) of each asm statement."""
    for m in re.finditer(r"\basm\s*(?:volatile)?\s*\(", text):
        depth, i = 1, m.end()
        while depth:
            depth += {"(": 1, ")": -1}.get(text[i], 0)
            i += 1
        body = text[m.end():i - 1]
        template = re.match(r'(?:\s*"(?:[^"\\]|\\.)*")+', body)
        yield template.group(0), body[template.end():]


def test_registers_named_in_the_text_are_declared():
    count = 0
    for path in sorted(sum((glob.glob(os.path.join(CSRC, "**", e), recursive=True) for e in ("*.hip", "*.hpp", "*.h")), [])):
        for template, rest in _statements(open(path).read()):
            count += 1
            for reg in re.findall(FIXED, template.replace("\\n", " ").replace("\\t", " ")):
                assert re.search(r'"[=+&]*\{?%s\}?"' % re.escape(reg), rest), "%s: %s names %s" % (os.path.basename(path), template, reg)
    assert count > 50          # (the sources were found and read)
