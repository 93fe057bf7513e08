"""Row-major q4 projections of one or two rows or of few outputs (rows.hip): the dot kernel at the
edges of its outputs a workgroup (1 x 1, 1 x 2, 2 x 4), K above one round of its threads, and the
MFMA kernel at ragged tiles and group counts around its 16 waves; strided activations and outputs,
a residual in place."""
import numpy as np
import pytest
import torch

import oracle
from qcheck import abs_gemm, bf16_tensor, check_close, dev_u16, dev_u32, to_f32

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from splosh_amd import runtime
    return runtime


# (rows, outputs, K): 1 x 1 with one group, with fewer items than a wave, K over 8192; two rows of a
# wide weight; 1 x 2 and 2 x 4 with odd rows and outputs; the last outputs of the dot kernel; the
# MFMA kernel with fewer groups than waves, an uneven share of groups, ragged rows and columns.
SHAPES = [(1, 1, 64), (1, 48, 5120), (1, 1300, 192), (2, 33, 8256), (2, 2500, 128), (5, 481, 320), (33, 48, 5120),
          (64, 47, 1088), (65, 48, 512), (67, 201, 192), (333, 48, 640),
          (342, 48, 192), (129, 129, 1088), (700, 33, 2112), (1000, 255, 64)]


@pytest.mark.parametrize("rows,n,k", SHAPES)
def test_rows_kernels(rt, rows, n, k):
    words, stride, sc, bi = oracle.q4_random_weight(n, k, seed=rows + n)
    w = rt.Q4Weight(dev_u32(words), dev_u16(sc), dev_u16(bi), n, k, rt.ROW_MAJOR, stride)
    dense = oracle.q4_dequant_rowmajor(words, stride, sc, bi, n, k)
    a_bits = oracle.bf16_normal((rows, k), seed=rows + k)
    lda, ldc = k + 8, n + 3
    a = torch.zeros(rows, lda, dtype=torch.bfloat16, device="cuda")
    a[:, :k] = bf16_tensor(a_bits)
    ref = oracle.gemm_a_bf16_w_f32(a_bits, dense)
    scale = abs_gemm(a_bits, dense)
    for dtype in (torch.float32, torch.bfloat16):
        out = torch.full((rows, ldc), 7.0, dtype=dtype, device="cuda")
        rt.gemm(w, a, out=out, residual=out)
        got = to_f32(out)
        assert np.all(got[:, n:] == 7.0)
        check_close(got[:, :n], ref + 7.0, bf16_out=dtype == torch.bfloat16, tight=True, absref=scale,
                    label=f"rows {rows} {n} {k}")
