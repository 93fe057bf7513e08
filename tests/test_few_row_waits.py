"""The loops of skinny.hip and the MFMA kernel of rows.hip wait with a counted vmcnt: "this group has landed"
is "at most the next group's loads are outstanding". This compiles both sources to gfx950 assembly (no GPU)
and checks that between one such wait and the next the compiler issues exactly a group's loads, with the
expected number into LDS, that nothing else (a spill, a store) counts there, and that LDS is read only
between the wait and the next loads."""
import os
import re
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def events(source, symbol):
    """Per kernel, its name and its memory events up to the barrier after the loop, in program order: a load
    into registers (r) or LDS (l), another memory access (x), an LDS read (d), a wait (its vmcnt and a blank)."""
    asm = subprocess.run([HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", f"-I{ROOT / 'include'}", "-Xclang",
                          "-target-feature", "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-S",
                          str(ROOT / "splosh_amd/csrc" / source), "-o", "-"], capture_output=True, text=True,
                         check=True).stdout
    for name, body in re.findall(rf"^(_ZN6splosh\d+{symbol}\S*):(.*?)^\.Lfunc_end", asm, re.S | re.M):
        out = ""
        for line in body.split("s_barrier")[0].split("\n"):
            ins = line.split(";")[0].strip()
            if re.match(r"(buffer|global|flat)_load", ins):
                out += "l" if ins.endswith(" lds") else "r"
            elif re.match(r"(buffer|global|flat|scratch)_", ins):
                out += "x"
            elif ins.startswith("ds_read"):
                out += "d"
            elif ins.startswith("s_waitcnt") and (wait := re.search(r"vmcnt\((\d+)\)", ins)):
                out += wait.group(1) + " "
        yield name, out


def groups(loads, into_lds):
    """A run of whole groups' loads, in any order."""
    return lambda run, n: len(run) == n * loads and run.count("l") == n * into_lds and set(run) <= {"r", "l"}


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="needs hipcc")
def test_skinny_waits():
    kernels = list(events("skinny.hip", "q4_skinny_kernel"))
    assert len(kernels) == 4 * 3 * 2  # what the weights are, staged rows, waves
    for name, ev in kernels:
        mode, rm, depth = (int(x) for x in re.search(r"SkinnyModeE(\d)ELi(\d+)ELi\d+ELi(\d+)E", name).groups())
        into_lds = rm // 8
        loads = 3 * (2 if mode >= 2 else 1) + into_lds
        whole = groups(loads, into_lds)
        # Two groups ahead, then each step: wait for the older, read it, load the one after the next.
        assert depth == 2, name
        m = re.fullmatch(rf"([rl]+){loads} (d+)([rl]+){loads} (d+)([rl]+)0 ", ev)
        assert m and whole(m.group(1), 2) and whole(m.group(3), 1) and whole(m.group(5), 1), (name, ev)


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="needs hipcc")
def test_rows_waits():
    (name, ev), = events("rows.hip", "q4_rows_mma_kernel")
    whole = groups(7, 4)
    # One group ahead, then each step: load the next, wait for the older, read it.
    m = re.fullmatch(r"([rl]{7})([rl]+)7 (d+)([rl]+)7 (d+)0 ", ev)
    assert m and all(whole(m.group(i), 1) for i in (1, 2, 4)), ev
