"""Which kernel calls of few rows take where two measured close (the comments at the rules have the times). The
rules are compiled code that asks for the CU count (256 where there is no device)."""
import subprocess
from pathlib import Path

import pytest

import test_mma_waitcounts as wc

LIB = wc.ROOT / "splosh_amd" / "libsplosh_q4.so"

# (rows, columns, inner, pair): does the decode kernel come before the raw-code MFMA kernel?
DECODE = [(f"decode_before_skinny({rows}, {n}, {k}, {pair})", want) for rows, n, k, pair, want in [
    (2, 17408, 5120, 0, 1), (2, 512, 1536, 1, 1), (3, 4096, 1536, 0, 1), (4, 128, 1280, 0, 1), (5, 512, 1536, 0, 0),
    (3, 4096, 1024, 0, 0), (3, 4096, 1792, 0, 0), (3, 4224, 1536, 0, 0), (4, 2048, 1536, 1, 0)]]
# (type, rows, columns, inner): does the barrier-free GGUF kernel take it? (planes: 13 Q5_K, 12 Q4_K)
GGUF = [(f"gguf_skinny_fits({kind}, {rows}, {n}, {k}, {k}, 1 << 20)", want) for kind, rows, n, k, want in [
    (13, 16, 12288, 4096, 0), (12, 12, 14336, 2048, 1), (12, 13, 14336, 2048, 0), (13, 8, 12288, 1536, 0),
    (13, 16, 8192, 1536, 1), (13, 16, 17408, 1536, 1), (13, 16, 9216, 4096, 1), (8, 7, 9216, 8192, 0),
    (13, 8, 9216, 8192, 1), (13, 16, 9216, 8192, 0), (8, 16, 11008, 1536, 0), (8, 16, 12288, 4096, 1),
    (8 | 0x100, 16, 12288, 4096, 0), (23, 16, 12288, 1536, 1), (23, 17, 12288, 1536, 0), (23, 17, 12288, 4096, 1),
    (20, 8, 9216, 1536, 1), (20, 9, 9216, 1536, 0), (14, 16, 12288, 1536, 1), (11, 32, 12288, 4096, 1)]]


@pytest.mark.skipif(not Path(wc.HIPCC).exists() or not LIB.exists(), reason="needs hipcc and the built library")
@pytest.mark.parametrize("checks", [DECODE, GGUF], ids=["decode", "gguf"])
def test_routes(tmp_path, checks):
    source, program = tmp_path / "routes.cpp", tmp_path / "routes"
    lines = "\n".join(f'    printf("%d\\n", (int)({e}));' for e, _ in checks)
    source.write_text(f'#include "launch.hpp"\n#include <cstdio>\nusing namespace splosh;\nint main() {{\n{lines}\n}}\n')
    subprocess.run([wc.HIPCC, "-O1", "-std=c++17", f"-I{wc.ROOT / 'include'}", f"-I{wc.ROOT / 'splosh_amd/csrc'}",
                    str(source), "-o", str(program), f"-L{LIB.parent}", "-lsplosh_q4", f"-Wl,-rpath,{LIB.parent}"],
                   check=True, capture_output=True)
    got = subprocess.run([str(program)], check=True, capture_output=True, text=True).stdout.split()
    assert [e for (e, want), g in zip(checks, got) if int(g) != want] == []
