"""The loop of skinny_gguf.hip waits with a counted vmcnt: "tile j has landed" is "at most three tiles
and the next unit's weights are outstanding", so the count of a unit's weight loads (kLoads) must be
what the compiler issues. This compiles the source to gfx950 assembly (no GPU) and checks, for every
kernel, that each run of weight loads (from its marker to the scheduling barrier that ends it) has
exactly the marked number of loads into registers and none into LDS, that each tile's run has only
loads into LDS, and that the waits are the counts these give."""
import os
import re
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="no hipcc")
def test_unit_load_counts():
    asm = subprocess.run([HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", f"-I{ROOT / 'include'}", "-Xclang",
                          "-target-feature", "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-S",
                          str(ROOT / "splosh_amd/csrc/skinny_gguf.hip"), "-o", "-"], capture_output=True, text=True,
                         check=True).stdout
    kernels = re.findall(r"^_ZN6splosh18gguf_skinny_kernelILi(\d+)ELi(\d+)E\S*:(.*?)s_endpgm", asm, re.S | re.M)
    assert len(kernels) == 8 * 3
    for kind, rm, body in kernels:
        label, na = f"type {kind}, {rm} rows", int(rm) // 8
        # (A marker is emitted once for the prologue and once in the loop.)
        runs = re.findall(r"splosh-unit-loads (\d+)(.*?)sched_barrier", body, re.S)
        assert len(runs) == 2, label
        for count, run in runs:
            loads = re.findall(r"^\s+buffer_load\S+.*$", run, re.M)
            assert len(loads) == int(count) and not any(x.rstrip().endswith("lds") for x in loads), label
        count = int(runs[0][0])
        rest = re.sub(r"splosh-unit-loads (\d+)(.*?)sched_barrier", "", body, flags=re.S)
        tiles = [re.findall(r"^\s+buffer_load\S+.*$", g, re.M) for g in rest.split("sched_barrier")]
        tiles = [t for t in tiles if t and any(x.rstrip().endswith("lds") for x in t)]
        assert len(tiles) == 8, label  # four in the prologue, four in the loop
        assert all(len(t) == na and all(x.rstrip().endswith("lds") for x in t) for t in tiles), label
        waits = [int(w) for w in re.findall(r"s_waitcnt vmcnt\((\d+)\)", body)]
        assert waits.count(3 * na + count) >= 4, label
