"""No kernel of the built library runs single lanes' work for all 64 lanes.

The flash holds more scalars than there are scalar registers; the compiler
keeps the rest in lanes of vector registers that it saves, restores and
copies for the whole wave (exec = -1).  Its ordinary allocation of those
registers has put single lanes' moves and spills inside such a copy: lanes on
the other side of a branch then lost their values, and a batch of binary cells
read a wild pointer.  Which functions it happens to changes with the code
around them (build.sh builds lanes.hip with another allocation for that
reason), so the built code is looked over: between the instructions that set
exec to all lanes and that put it back there is either one copy and nothing
else, or saves and restores only.

And the masks of finished lanes that a loop adds to keep what they hold.  The
compiler takes a register that holds saved scalars for undefined again at
their first save, which can lie inside the loop: what the loop had saved
there before is then overwritten, or not saved before the register is used for
others.  The results of lanes that left a solver early were lost so (see
Flash::keepInLanes).  Where a block reads a saved scalar, combines it and
saves it again, the value has to be in the register that is read the next
time, on every way around the innermost loop."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from reactive_amd import LIBRARY_PATH

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
SAVES = re.compile(r"s_|v_writelane_b32|v_readlane_b32|scratch_(load|store)_dword")
ALL_LANES = re.compile(r"s_(or|xor)_saveexec_b64 s\S+, -1|s_mov_b64 exec, -1")
ENDS = re.compile(r"s_\w+ exec\b|s_\w+saveexec")


def mixed_regions(lines):
    """(function, instructions) of the regions that hold anything else."""
    found, function, region = [], None, None
    for line in lines:
        if line.endswith(">:\n"):
            function, region = line.split("<", 1)[1][:-3], None
            continue
        text = line.split("//")[0].strip()
        if ALL_LANES.match(text):
            region = []
        elif ENDS.match(text):
            if region:
                work = [i for i in region if not SAVES.match(i)]
                if work and (len(work) > 1 or len(region) > 1 or not work[0].startswith("v_mov_b32")):
                    found.append((function, region))
            region = None
        elif region is not None and text and not text.startswith(("s_nop", "s_waitcnt")):
            region.append(text)
    return found


READ = re.compile(r"v_readlane_b32 s(\d+), v(\d+), (\d+)")
WRITE = re.compile(r"v_writelane_b32 v(\d+), s(\d+), (\d+)")
STORE = re.compile(r"scratch_store_dword off, v(\d+), s33(?: offset:(\d+))?$")
LOAD = re.compile(r"scratch_load_dword v(\d+), off, s33(?: offset:(\d+))?$")
COPY = re.compile(r"v_mov_b32_e32 v(\d+), v(\d+)$")
COMBINE = re.compile(r"s_(andn2|orn2|and|or|xor|add|mov)\w* (\S+), (.*)")
TARGET = re.compile(r"<.*\+0x([0-9a-f]+)>$")


def functions(lines):
    """(name, [(address, instruction, branch target or None)]) per function."""
    name, ops = None, []
    for line in lines:
        if line.endswith(">:\n"):
            if ops:
                yield name, ops
            base, name = int(line.split()[0], 16), line.split("<", 1)[1][:-3]
            ops = []
        elif name and "//" in line:
            text, comment = line.split("//", 1)
            text, comment = text.strip(), comment.strip()
            to = None
            if text.startswith(("s_cbranch", "s_branch")):
                found = TARGET.search(comment)
                to = base + int(found.group(1), 16) if found else base
            ops.append((int(comment.split(":")[0], 16), text, to))
    if ops:
        yield name, ops


def blocks_of(ops):
    """Basic blocks as lists of (instruction, whether all lanes run it), and their successors."""
    leaders = {to for _, _, to in ops if to is not None} | {ops[0][0]}
    blocks, starts, ends, allLanes = [], {}, [], False
    for k, (address, text, to) in enumerate(ops):
        if address in leaders or (k and ops[k - 1][2] is not None):
            starts[address] = len(blocks)
            blocks.append([])
            ends.append(None)
        if ALL_LANES.match(text):
            allLanes = True
        elif allLanes and ENDS.match(text):
            allLanes = False
        else:
            blocks[-1].append((text, allLanes))
        ends[-1] = (text, to)
    successors = []
    for b, (text, to) in enumerate(ends):
        following = [starts[to]] if to in starts else []
        if not text.startswith(("s_branch", "s_setpc", "s_endpgm")) and b + 1 < len(blocks):
            following.append(b + 1)
        successors.append(following)
    return blocks, successors


def innermost_loops(successors):
    """Per block the set of blocks of the smallest natural loop around it (None: no loop)."""
    n = len(successors)
    before = [[] for _ in range(n)]
    for b, to in enumerate(successors):
        for t in to:
            before[t].append(b)
    everything = (1 << n) - 1
    dominators = [everything] * n
    dominators[0] = 1
    changed = True
    while changed:
        changed = False
        for b in range(1, n):
            d = everything
            for p in before[b]:
                d &= dominators[p]
            d |= 1 << b
            if d != dominators[b]:
                dominators[b], changed = d, True
    loops = {}
    for b, to in enumerate(successors):
        for head in to:
            if dominators[b] >> head & 1:
                body, todo = loops.setdefault(head, {head}), [b]
                while todo:
                    x = todo.pop()
                    if x not in body:
                        body.add(x)
                        todo += before[x]
    inner = [None] * n
    for body in loops.values():
        for b in body:
            if inner[b] is None or len(body) < len(inner[b]):
                inner[b] = body
    return inner


def scalars(operand):
    pair = re.match(r"s\[(\d+):(\d+)\]$", operand)
    one = re.match(r"s(\d+)$", operand)
    return set(range(int(pair.group(1)), int(pair.group(2)) + 1)) if pair else {int(one.group(1))} if one else set()


def saved_again(block, start, value, register, lane):
    """Where the scalar read at `start` is saved to its lane again, combined with others (or None)."""
    held = {value}
    for k in range(start + 1, len(block)):
        text = block[k][0]
        write = WRITE.match(text)
        if write:
            if (int(write.group(1)), int(write.group(3))) == (register, lane):
                return k if int(write.group(2)) in held else None
            continue
        read = READ.match(text)
        combine = COMBINE.match(text)
        if read:
            held.discard(int(read.group(1)))
        elif combine:
            to = scalars(combine.group(2).rstrip(","))
            sources = [scalars(o.strip()) for o in combine.group(3).split(",")]
            held = held | to if any(f & held for f in sources) else held - to
        elif text.startswith("s_") and " " in text:
            held = held - scalars(text.split()[1].rstrip(","))
    return None


def places(where, block):
    """The registers and stack slots that hold the lane after the block, of those that held it before."""
    for text, allLanes in block:
        if not allLanes:
            continue
        for kind, pattern in (("store", STORE), ("load", LOAD), ("copy", COPY)):
            m = pattern.match(text)
            if m:
                register, other = ("v", int(m.group(1))), int(m.group(2) or 0)
                to, source = {"store": (("s", other), register), "load": (register, ("s", other)),
                              "copy": (register, ("v", other))}[kind]
                where = where | {to} if source in where else where - {to}
                break
    return where


def lost_masks(ops):
    """How many saved scalars a loop combines, and those it does not find
    again the next time around: (register, lane)."""
    texts = [text for _, text, _ in ops]
    if not any(READ.match(t) for t in texts) or not any(WRITE.match(t) for t in texts):
        return 0, []
    blocks, successors = blocks_of(ops)
    loops = innermost_loops(successors)
    checked, lost = 0, []
    for b, block in enumerate(blocks):
        if loops[b] is None:
            continue
        for start, (text, _) in enumerate(block):
            read = READ.match(text)
            if not read:
                continue
            value, register, lane = map(int, read.groups())
            end = saved_again(block, start, value, register, lane)
            if end is None:
                continue
            checked += 1
            after = places(frozenset({("v", register)}), block[end + 1:])
            seen, todo = {}, [(t, after) for t in successors[b] if t in loops[b]]
            while todo:
                t, where = todo.pop()
                known = seen.get(t)
                where = where if known is None else known & where
                if where == known:
                    continue
                seen[t] = where
                if t == b:
                    if ("v", register) not in places(where, block[:start]):
                        lost.append((register, lane))
                        break
                    continue
                where = places(where, blocks[t])
                todo += [(u, where) for u in successors[t] if u in loops[b]]
    return checked, lost


def test_the_scan_finds_mixed_regions():
    head = "0000000000001900 <kernel>:\n"
    begin, end = "\ts_or_saveexec_b64 s[4:5], -1   // 1\n", "\ts_mov_b64 exec, s[4:5]   // 2\n"
    copy, spill, save = "\tv_mov_b32_e32 v1, v2\n", "\tscratch_store_dword off, v3, s33 offset:4\n", "\tv_writelane_b32 v1, s2, 3\n"
    for inside, bad in (([copy], 0), ([spill, spill], 0), ([save, spill], 0), ([copy, spill], 1), ([copy, copy], 1),
                        (["\tv_add_u32_e32 v1, v2, v3\n"], 1)):
        assert len(mixed_regions([head, begin, *inside, end, copy, copy])) == bad


def test_the_scan_finds_lost_masks():
    def ops(*texts):
        return [(16 * k, t, int(t.split()[1]) if t.startswith("s_cbranch") else None) for k, t in enumerate(texts)]
    # a loop from the third instruction on; v9 holds the mask in lane 7
    head = ["s_mov_b64 s[0:1], 0", "s_nop 0"]
    body = ["v_readlane_b32 s2, v9, 7", "s_or_b64 s[2:3], s[2:3], s[4:5]", "v_writelane_b32 v9, s2, 7"]
    save = ["s_or_saveexec_b64 s[6:7], -1", "scratch_store_dword off, v9, s33 offset:544", "s_mov_b64 exec, s[6:7]"]
    load = ["s_or_saveexec_b64 s[6:7], -1", "scratch_load_dword v9, off, s33 offset:544", "s_mov_b64 exec, s[6:7]"]
    again = ["s_cbranch_execnz 32", "s_setpc_b64 s[30:31]"]
    assert lost_masks(ops(*head, *body, *again)) == (1, [])
    assert lost_masks(ops(*head, *load, *body, *save, *again)) == (1, [])
    assert lost_masks(ops(*head, *load, *body, *again)) == (1, [(9, 7)])


def test_no_lane_works_in_a_whole_wave_copy(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    copy = shutil.copy(LIBRARY_PATH, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", copy], check=True, capture_output=True)
    objects = glob.glob(copy + ".*gfx950")
    assert len(objects) >= 9
    regions = checked = 0
    for code in objects:
        with subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", code], stdout=subprocess.PIPE, text=True) as dump:
            lines = list(dump.stdout)
        assert dump.returncode == 0
        regions += sum(1 for line in lines if ALL_LANES.search(line))
        assert mixed_regions(lines) == []
        for name, ops in functions(lines):
            count, lost = lost_masks(ops)
            checked += count
            assert (name, lost) == (name, [])
    assert checked > 500
    assert regions > 100  # the pattern still matches what the compiler writes
