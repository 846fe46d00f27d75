"""Build-time check of the waits in the bf16 linears of up to 64 rows.

Their rows are loaded straight into LDS and read back with inline assembly behind a wait that counts the loads issued since.
The count is right only as long as the compiler leaves the loads where the source has them, so the machine code of every
instance is walked: no row tile is read with one of its own loads under way, none is loaded again with a read of it under way,
and no wait inside the loop asks for the pair that was requested last.
"""
import re

import pytest

from machine_code import HAVE_TOOLS, disassemble

LDS_LOAD = re.compile(r"(buffer|global)_load_dwordx4 .* lds$|global_load_lds")
VMEM = re.compile(r"(buffer|global|flat|scratch)_(load|store|atomic)")


def faults(lines, row_tiles, jumps=(), start=0, wait_at_least=0):
    """What the paths from `start` to the next barrier do wrong; loads into LDS come 2 row_tiles to a slot, first slot 0, then slot 1."""
    target = dict(jumps)
    bad, seen, todo = [], set(), [(start, (), (), 0)]
    while todo:
        at, loads, reads, issued = state = todo.pop()
        if state in seen or at >= len(lines) or lines[at].startswith(("s_barrier", "s_endpgm")):
            continue
        seen.add(state)
        line = lines[at]
        if line.startswith("s_waitcnt"):
            count = re.search(r"vmcnt\((\d+)\)", line)
            if count:
                n = int(count.group(1))
                loads = loads[max(0, len(loads) - n):]
                if n < wait_at_least:
                    bad.append("waits for the youngest pair: " + line)
            if "lgkmcnt(0)" in line:
                reads = ()
        elif LDS_LOAD.match(line):
            slot = issued // (2 * row_tiles)
            issued = (issued + 1) % (4 * row_tiles)
            if slot in reads:
                bad.append("loaded while it is read: " + line)
            loads = (loads + (slot,))[-64:]
        elif VMEM.match(line):
            loads = (loads + (None,))[-64:]
        elif line.startswith("ds_read_b128"):
            offset = re.search(r"offset:(\d+)", line)
            slot = (int(offset.group(1)) if offset else 0) // (2048 * row_tiles)
            if slot in loads:
                bad.append("read while it is loaded: " + line)
            reads = tuple(sorted(set(reads + (slot,))))
        if at in target:
            todo.append((target[at], loads, reads, issued))
        if not line.startswith("s_branch"):
            todo.append((at + 1, loads, reads, issued))
    return bad


def test_faults_are_found():
    load, weight, read = "buffer_load_dwordx4 v1, s[0:3], s4 offen lds", "global_load_dwordx4 v[2:5], v[0:1], off nt", "ds_read_b128 v[6:9], v0"
    slots = [weight] * 2 + [load] * 2 + [weight] * 2 + [load] * 2
    done = [read, "s_waitcnt lgkmcnt(0)"]
    assert faults(slots + ["s_waitcnt vmcnt(4)"] + done + [load], 1) == []
    assert faults(slots + ["s_waitcnt vmcnt(5)"] + done, 1)                                  # one of the slot's loads is out
    assert faults([load] * 4 + [weight] * 2 + ["s_waitcnt vmcnt(4)"] + done, 1) == []        # more loads behind it: waits for more
    assert faults([weight] * 4 + [load] * 4 + ["s_waitcnt vmcnt(4)"] + done, 1)              # fewer than the count stands for
    assert faults(slots + ["s_waitcnt vmcnt(4)", read, load], 1)                             # read not over
    assert faults(slots + ["s_waitcnt vmcnt(4)", read + " offset:2048"], 1)                  # the other slot
    assert faults(slots + ["s_waitcnt vmcnt(0)"] + done, 1, wait_at_least=4)
    jump = slots + ["s_cbranch_scc1 1", "s_waitcnt vmcnt(4)"] + done                         # a way past the wait
    assert faults(jump, 1) == [] and faults(jump, 1, [(8, 10)])


@pytest.mark.skipif(not HAVE_TOOLS, reason="no LLVM tools")
def test_rows_are_read_behind_their_loads(tmp_path):
    walked = 0
    for name, (lines, jumps) in disassemble(tmp_path, "linear_rows(?:_grouped)?_kernel").items():
        for last, first in sorted(jumps):
            body = lines[first:last + 1]
            staged = sum(bool(LDS_LOAD.match(l)) for l in body)
            products = sum("v_mfma" in l for l in body)
            inner = not any(a > first and b < last and a < b for b, a in jumps if b != last)
            if first >= last or not staged or not products or not inner or any("s_barrier" in l for l in body):
                continue
            row_tiles, columns = staged // 4, products // staged                  # two slots of two loads to a row tile, two products each
            assert staged == 4 * row_tiles and products == columns * staged, name
            assert sum(l.startswith("ds_read_b128") for l in body) == staged, name
            ahead = [i for i in range(first) if LDS_LOAD.match(lines[i])][-staged]        # both slots' first loads
            bad = faults(body + body, row_tiles, wait_at_least=2 * (row_tiles + columns)) + faults(lines, row_tiles, jumps, ahead)
            assert not bad, (name, bad[:3])
            walked += 1
    assert walked >= 50, walked
