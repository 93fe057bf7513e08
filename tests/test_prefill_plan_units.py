"""The prefill plan of a format that splits K at units of four 64-groups counts a workgroup's share in those:
no workgroup of a split is left without one, and a tile gets no more slices than shorten its longest share."""
import subprocess
from pathlib import Path

import pytest

import test_mma_waitcounts as wc

LIB = wc.ROOT / "splosh_amd" / "libsplosh_q4.so"
PROGRAM = """
#include "launch.hpp"
#include <cstdio>
int main() {
    for (long rows : {65, 129, 149, 200, 333, 640, 1024, 2048})
        for (long columns : {128, 640, 1024, 4096, 5120, 7936, 17408})
            for (long units = 1; units <= 68; ++units) {
                const splosh::PrefillPlan p = splosh::plan_prefill(rows, columns, 4 * units, (size_t)-1,
                                                                     splosh::kPrefillUnits);
                printf("%ld %ld %ld %d %d %ld\\n", rows, columns, units, p.tiles - p.dp_tiles, p.sk_grid,
                       (long)p.sk_units);
            }
}
"""


@pytest.mark.skipif(not Path(wc.HIPCC).exists() or not LIB.exists(), reason="needs hipcc and the built library")
def test_shares_are_whole_units(tmp_path):
    source, program = tmp_path / "plan.cpp", tmp_path / "plan"
    source.write_text(PROGRAM)
    subprocess.run([wc.HIPCC, "-O1", "-std=c++17", f"-I{wc.ROOT / 'include'}", f"-I{wc.ROOT / 'splosh_amd/csrc'}",
                    str(source), "-o", str(program), f"-L{LIB.parent}", "-lsplosh_q4",
                    f"-Wl,-rpath,{LIB.parent}"], check=True,
                   capture_output=True)
    plans = [[int(x) for x in line.split()] for line in
             subprocess.run([str(program)], check=True, capture_output=True, text=True).stdout.splitlines()]
    assert any(p[5] > 0 for p in plans)
    for rows, columns, units, tiles, workgroups, groups in plans:
        if groups == 0:
            continue
        label = (rows, columns, units, tiles, workgroups)
        assert groups == 4 * units * tiles and workgroups <= units * tiles, label
        slices, rest = divmod(workgroups, tiles)
        if rest == 0 and 2 < slices <= 16:  # (two are the fewest; above 16 the tiles are split over all CUs)
            longest = -(-units // slices)
            assert -(-units // (slices - 1)) > longest, label
