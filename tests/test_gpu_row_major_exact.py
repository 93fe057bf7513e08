"""Row-major q4 weights enter the sums exactly in the rows past 64 of a call of 65 or 66 rows, as they do at one
and two: activations with a single nonzero element return the fp32 weights."""
import numpy as np
import pytest
import torch

from qcheck import Q4Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(512, 2048), (1024, 1536)])
@pytest.mark.parametrize("rows", [1, 2, 65, 66])
def test_single_element_rows(rows, n, k):
    from splosh_amd import runtime as rt
    c = Q4Case(n, k, seed=rows + n)
    a = torch.zeros(rows, k, dtype=torch.bfloat16, device="cuda")
    at = [(37 * m + 5) % k for m in range(rows)]
    for m in range(rows):
        a[m, at[m]] = 1.0
    got = rt.gemm(c.w_rm, a, out_dtype=torch.float32).cpu().numpy()
    for m in range(64 if rows > 64 else 0, rows):
        group = c.dense[:, at[m] // 64 * 64: at[m] // 64 * 64 + 64]
        # s (128 + q) + (b - 128 s): a few roundings of values of at most 143 s + |w|, and s at most a third of
        # the group's range (its 64 codes span three or more).
        step = np.ptp(group, axis=1) / 3
        assert np.all(np.abs(got[m] - c.dense[:, at[m]]) <= 2.0 ** -24 * 4 * (143 * step + np.abs(group).max(axis=1)))
