"""The prefill kernel's lower tiles and grouped form (prefill_tile_kernel) wait for their loads into LDS
as the 256-row one does: the check of test_mma_waitcounts on every instantiation, two or three (or
four) activation loads a wave and group."""
import re
import subprocess
from pathlib import Path

import pytest

import test_mma_waitcounts as wc


@pytest.mark.skipif(not Path(wc.HIPCC).exists(), reason="needs hipcc")
def test_tile_kernels_wait_for_their_loads(tmp_path):
    out = tmp_path / "prefill.s"
    subprocess.run([wc.HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", f"-I{wc.ROOT / 'include'}", "--cuda-device-only", "-S",
                    str(wc.ROOT / "splosh_amd" / "csrc" / "prefill.hip"), "-o", str(out)], check=True,
                   capture_output=True)
    kernels = list(wc._kernels(out.read_text(), r"_ZN6splosh19prefill_tile_kernel\S*"))
    # Two lower tiles of ten stages, three of the grouped one and of Q8_0 and IQ4_NL in whole units.
    assert len(kernels) == 2 * 10 + 3 + 2 * 3
    for name, code in kernels:
        assert any(wc._is_lds(ins) for ins in code), name
        fm = int(re.search(r"Li(\d)EEEvNS_11PrefillArgs", name).group(1))
        assert wc._check_function(name, code, stage=fm)[1] >= 3, name
