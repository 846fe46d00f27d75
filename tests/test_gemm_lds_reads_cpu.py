"""Build-time check of the large-tile GEMM kernels' fragment reads.

The kernels read fragments from LDS with inline assembly and wait for them in later statements, which the compiler cannot
tell from registers that are ready.  In the machine code of the built library no instruction may therefore touch a register
that an LDS read is still on its way to; the body of the main loop is walked twice, so that what its tail requests is
followed into the next pass.
"""
import os
import re
import shutil
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin"


def registers(operands):
    """Vector registers that an instruction names."""
    out = set()
    for m in re.finditer(r"\bv(?:(\d+)\b|\[(\d+):(\d+)\])", operands):
        lo, hi = (m.group(1), m.group(1)) if m.group(1) else (m.group(2), m.group(3))
        out.update(range(int(lo), int(hi) + 1))
    return out


def early_touches(lines):
    """Instructions that touch the destination of an LDS read before a wait that covers it; LDS operations finish in order."""
    pending, bad, reads = [], [], 0
    for line in lines:
        op, _, operands = line.partition(" ")
        wait = re.search(r"lgkmcnt\((\d+)\)", operands) if op == "s_waitcnt" else None
        if wait:
            pending = pending[len(pending) - int(wait.group(1)):] if int(wait.group(1)) < len(pending) else pending
            if wait.group(1) == "0":
                pending = []
            continue
        used = registers(operands)
        if op.startswith("ds_read"):
            dst, _, addr = operands.partition(",")
            if any(registers(operands) & p for p in pending):
                bad.append(line)
            pending.append(registers(dst))
            reads += 1
        else:
            if any(used & p for p in pending):
                bad.append(line)
            if op.startswith("ds_"):
                pending.append(set())
    return bad, reads


def test_a_touch_before_the_wait_is_found():
    ok = ["ds_read_b128 v[0:3], v9", "ds_read_b128 v[4:7], v9 offset:16", "s_waitcnt lgkmcnt(1)", "v_mov_b32_e32 v8, v3", "s_waitcnt lgkmcnt(0)"]
    assert early_touches(ok + ["v_mov_b32_e32 v8, v4"]) == ([], 2)
    assert early_touches(ok[:4] + ["v_mov_b32_e32 v8, v4"])[0] == ["v_mov_b32_e32 v8, v4"]
    assert early_touches(ok[:1] + ["v_add_u32_e32 v2, v8, v8"])[0]
    assert early_touches(ok[:1] + ["ds_read_b128 v[4:7], v3"])[0]


@pytest.mark.skipif(not os.path.exists(os.path.join(LLVM, "llvm-objdump")), reason="no LLVM tools")
def test_no_fragment_is_touched_while_it_is_read(tmp_path):
    from fandhe_ai_amd import capi
    objdump = os.path.join(LLVM, "llvm-objdump")
    lib = shutil.copy(capi.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([objdump, "--offloading", lib], check=True, capture_output=True, cwd=tmp_path)
    kernels = 0
    for f in sorted(tmp_path.iterdir()):
        if "gfx950" not in f.name:
            continue
        names = subprocess.run([objdump, "-t", str(f)], check=True, capture_output=True, text=True).stdout
        names = sorted(set(re.findall(r" F .*?(\S*gemm_mfma_big_kernel\S*)$", names, flags=re.M)))
        if not names:
            continue
        text = subprocess.run([objdump, "-d", "--disassemble-symbols=" + ",".join(names), str(f)], check=True, capture_output=True, text=True).stdout
        for body in re.split(r"^[0-9a-f]+ <(?=\S*gemm_mfma_big_kernel)", text, flags=re.M)[1:]:
            base, lines, at, jumps = None, [], {}, []
            for l in body.split("\n")[1:]:
                m = re.match(r"\s*(\S.*?)\s*//\s*([0-9A-F]+):", l)
                if not m:
                    continue
                addr = int(m.group(2), 16)
                base = addr if base is None else base
                at[addr] = len(lines)
                lines.append(m.group(1))
                j = re.search(r"<\S+\+0x([0-9a-f]+)>\s*$", l)
                if j and m.group(1).startswith("s_cbranch"):
                    jumps.append((len(lines) - 1, base + int(j.group(1), 16)))
            loops = [(at[to], i) for i, to in jumps if to in at and at[to] < i and any("v_mfma" in x for x in lines[at[to]:i])]
            assert loops, body[:100]
            begin, end = min(loops, key=lambda x: x[0])
            bad, reads = early_touches(lines[:end + 1] + lines[begin:])
            assert reads > 24 and not bad, "%s: %s" % (body[:100], bad[:3])
            kernels += 1
    assert kernels >= 12
