"""Inline assembly of the kernels names the registers it writes besides its outputs."""
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SPECIAL = ("m0", "vcc", "exec", "scc")


def asm_statements():
    for path in sorted(glob.glob(os.path.join(ROOT, "libbi_amd", "csrc", "*.h*"))):
        text = re.sub(r"//[^\n]*", "", open(path).read())
        for m in re.finditer(r"\basm\s*(?:volatile)?\s*\((.*?)\)\s*;", text, re.S):
            yield os.path.basename(path), m.group(1)


def written(template):
    """Special registers that are an instruction's first operand."""
    out = set()
    for line in template.replace("\\t", " ").split("\\n"):
        op = re.match(r"\s*[\w.]+\s+(\w+)", line)
        if op and op.group(1) in SPECIAL:
            out.add(op.group(1))
    return out


def test_special_registers_written_are_clobbers():
    found = 0
    for name, body in asm_statements():
        strings = re.findall(r'"((?:[^"\\]|\\.)*)"', body)
        need = written(strings[0])
        found += len(need)
        clobbers = re.findall(r'"(\w+)"', body.rsplit(":", 1)[1]) if ":" in body else []
        assert need <= set(clobbers), (name, body)
    assert found > 0  # the copies to LDS set m0
