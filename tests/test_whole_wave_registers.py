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
else, or saves and restores only."""
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


def test_the_scan_finds_mixed_regions():
    head = "0000000000001900 <kernel>:\n"
    begin, end = "\ts_or_saveexec_b64 s[4:5], -1   // 1\n", "\ts_mov_b64 exec, s[4:5]   // 2\n"
    copy, spill, save = "\tv_mov_b32_e32 v1, v2\n", "\tscratch_store_dword off, v3, s33 offset:4\n", "\tv_writelane_b32 v1, s2, 3\n"
    for inside, bad in (([copy], 0), ([spill, spill], 0), ([save, spill], 0), ([copy, spill], 1), ([copy, copy], 1),
                        (["\tv_add_u32_e32 v1, v2, v3\n"], 1)):
        assert len(mixed_regions([head, begin, *inside, end, copy, copy])) == bad


def test_no_lane_works_in_a_whole_wave_copy(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    copy = shutil.copy(LIBRARY_PATH, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", copy], check=True, capture_output=True)
    objects = glob.glob(copy + ".*gfx950")
    assert len(objects) >= 9
    regions = 0
    for code in objects:
        with subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", code], stdout=subprocess.PIPE, text=True) as dump:
            lines = list(dump.stdout)
        assert dump.returncode == 0
        regions += sum(1 for line in lines if ALL_LANES.search(line))
        assert mixed_regions(lines) == []
    assert regions > 100  # the pattern still matches what the compiler writes
