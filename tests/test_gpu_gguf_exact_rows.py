"""Native GGUF weights enter the sums exactly at the streaming kernels' rows (IQ4_NL 1 to 3, Q3_K 1 to 6,
the others 1 to 4), whatever the weight's size: activations with a single nonzero element return the
decoder's weights, where a kernel that rounds them to bf16 is off by up to 2^-9 of each."""
import numpy as np
import pytest
import torch

import oracle
from qcheck import dev_u8

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from splosh_amd import runtime
    return runtime


def check_single_element(rt, kind, n, k, rows32, calls):
    """calls: (rows, the first row that is exact)."""
    native = oracle.gguf_random_native(kind, n, k, seed=kind)
    dense = oracle.gguf_decode(kind, native).reshape(n, k)
    w = rt.GgufWeight(dev_u8(native), kind, n, k)
    w = rt.gguf_repack_rows32(w) if rows32 else w
    for rows, first in calls:
        a = torch.zeros(rows, k, dtype=torch.bfloat16, device="cuda")
        at = [(37 * m + 5) % k for m in range(rows)]
        for m in range(rows):
            a[m, at[m]] = 1.0
        got = rt.gemm(w, a, out_dtype=torch.float32).cpu().numpy()
        # The raw-code forms add s sum x (code + o) and s o sum x: a few fp32 roundings of values of at
        # most 256 s, where a block's largest weight is at least s; 2^-13 of it is above them and under
        # bf16's 2^-9 of a weight of the block's upper sixteenth.
        for m in range(first, rows):
            block = np.abs(dense[:, at[m] // 32 * 32: at[m] // 32 * 32 + 32]).max(axis=1)
            assert np.all(np.abs(got[m] - dense[:, at[m]]) <= 2.0 ** -13 * block), (rows, m)


@pytest.mark.parametrize("rows32", [False, True])
@pytest.mark.parametrize("kind,most", [(8, 4), (11, 6), (14, 4), (20, 3), (21, 4), (23, 4)])
@pytest.mark.parametrize("n,k", [(128, 512), (8192, 2048)])
def test_streaming_rows(rt, kind, most, rows32, n, k):
    calls = [(rows, 0) for rows in range(1, most + 1)]
    # 65 rows and the few after: the rows past 64 are such a call of their own (Q3_K: one tiled call).
    check_single_element(rt, kind, n, k, rows32, calls + ([] if kind == 11 else [(64 + most, 64)]))


def test_rows_past_64_of_a_large_weight(rt):
    check_single_element(rt, 8, 8192, 5120, False, [(65, 64), (68, 64)])
