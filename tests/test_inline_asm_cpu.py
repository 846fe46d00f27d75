"""What inline assembly has to tell the compiler: the special registers it writes, and no result that is still under way."""
import glob
import os
import re

ROOT = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "fandhe_ai_amd", "csrc")
SPECIAL = ("m0", "vcc", "exec", "scc")


def statements(text):
    """Every asm statement of a source: what stands between its parentheses."""
    for m in re.finditer(r"\basm\s+(?:volatile\s*)?\(", text):
        depth, at, quoted = 1, m.end(), False
        while depth:
            c = text[at]
            if c == '"' and text[at - 1] != "\\":
                quoted = not quoted
            elif not quoted:
                depth += (c == "(") - (c == ")")
            at += 1
        yield text[m.end():at - 1]


def parts(statement):
    """Template, outputs, inputs, clobbers."""
    out, depth, quoted = [""], 0, False
    for i, c in enumerate(statement):
        if c == '"' and statement[i - 1] != "\\":
            quoted = not quoted
        elif not quoted:
            depth += (c in "([{") - (c in ")]}")
            if c == ":" and depth == 0:
                out.append("")
                continue
        out[-1] += c
    return out + [""] * (4 - len(out))


def test_special_registers_are_named_as_clobbers():
    seen = 0
    for path in sorted(glob.glob(os.path.join(ROOT, "*.h*"))):
        for s in statements(open(path).read()):
            seen += 1
            p = parts(s)
            for line in re.split(r"\\n|\\t|;", "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', p[0]))):
                w = re.match(r"\s*[sv]_\w+\s+(\w+)", line)
                if w and w.group(1) in SPECIAL:
                    assert '"%s"' % w.group(1) in p[3], "%s: %s" % (os.path.basename(path), s.strip())
    assert seen > 10


def test_loads_into_registers_are_waited_for_in_their_statement():
    """The compiler takes an output as written when the statement ends and may move or reuse its register from there on.  (LDS
    reads ahead of their waits are followed through the machine code of the one kernel that has them.)"""
    for path in sorted(glob.glob(os.path.join(ROOT, "*.h*"))):
        for s in statements(open(path).read()):
            p = parts(s)
            if p[1].strip() and re.search(r"\b(global|buffer|flat|scratch|s)_load", p[0]):
                assert "s_waitcnt" in p[0][p[0].rindex("_load"):], "%s: %s" % (os.path.basename(path), s.strip())
