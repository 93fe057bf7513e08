"""Tiled q4 weights at 3 to 32 rows (skinny.hip) and grouped calls from one row: the staged row
counts' edges (8, 16, 32), K shorter than a round of the waves and ragged against it, K slices with
and without a workspace (few blocks; long K), weights split into their column halves (one pair a
CU; two), the fused pair, strided activations and outputs, a residual in place, rows of zeros and
of large activations."""
import numpy as np
import pytest
import torch

import oracle
from qcheck import Q4Case, abs_gemm, bf16_tensor, check_close, to_f32

pytestmark = pytest.mark.gpu

ROWS = [3, 4, 5, 8, 9, 16, 17, 24, 31, 32]


@pytest.fixture(scope="module")
def rt():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from splosh_amd import runtime
    return runtime


_CASES = {}


def case(n, k, seed=0):
    if (n, k, seed) not in _CASES:
        _CASES[n, k, seed] = Q4Case(n, k, seed=600 + seed + n + k)
    return _CASES[n, k, seed]


def activations(rows, k, pad=0):
    bits = oracle.bf16_normal((rows, k), seed=rows + k)
    if rows > 3:
        bits[1] = 0
        bits[2] = oracle.f32_to_bf16_rne(oracle.bf16_to_f32(bits[2]) * 1e4)
    a = torch.zeros(rows, k + pad, dtype=torch.bfloat16, device="cuda")
    a[:, :k] = bf16_tensor(bits)
    return bits, a


# One 32-column block a wave quarter; one group; ragged K; K slices of few blocks; one pair a CU
# (8448 = 264 blocks, 132 pairs) and the same width that does not halve (8320).
@pytest.mark.parametrize("n,k", [(128, 64), (128, 1088), (384, 2112), (1024, 4096), (8448, 192), (8320, 128)])
@pytest.mark.parametrize("rows", ROWS)
def test_skinny(rt, rows, n, k):
    c = case(n, k)
    bits, a = activations(rows, k, pad=8)
    ref, scale = oracle.gemm_a_bf16_w_f32(bits, c.dense), abs_gemm(bits, c.dense)
    ws = torch.zeros(max(1, rt.workspace_bytes(rows, n, k)), dtype=torch.uint8, device="cuda")
    for dtype in (torch.float32, torch.bfloat16):
        out = torch.full((rows, n + 4), 3.0, dtype=dtype, device="cuda")
        rt.gemm(c.w_tiled, a, out=out, residual=out, workspace=ws)
        again = torch.full_like(out, 3.0)
        rt.gemm(c.w_tiled, a, out=again, residual=again, workspace=ws)
        assert torch.equal(out, again)
        got = to_f32(out)
        assert np.all(got[:, n:] == 3.0)
        check_close(got[:, :n], ref + 3.0, bf16_out=dtype == torch.bfloat16, tight=True, absref=scale,
                    label=f"skinny {rows} {n} {k}")
    whole = to_f32(rt.gemm(c.w_tiled, a, out_dtype=torch.float32, workspace=torch.empty(0, device="cuda")))
    check_close(whole, ref, bf16_out=False, tight=True, absref=scale, label=f"skinny whole {rows} {n} {k}")
    assert not ws[:16384].any()  # the counters are returned to zero


@pytest.mark.parametrize("rows,n,k", [(8, 4352, 12288), (17, 33024, 128), (5, 33024, 128)])
def test_skinny_large(rt, rows, n, k):
    """Long K in slices of a split weight (136 blocks), and two pairs of halves a CU (516)."""
    test_skinny(rt, rows, n, k)
    _CASES.clear()


@pytest.mark.parametrize("n,k", [(128, 64), (640, 1088), (16512, 128)])
@pytest.mark.parametrize("rows", [3, 8, 13, 32])
def test_skinny_pair(rt, rows, n, k):
    """The fused gate+up (516 blocks: the last round of blocks in K slices)."""
    gate, up = case(n, k), case(n, k, 1)
    bits, a = activations(rows, k)
    ws = torch.zeros(max(1, rt.workspace_bytes(rows, n, k)), dtype=torch.uint8, device="cuda")
    ref = oracle.silu_mul(oracle.gemm_a_bf16_w_f32(bits, gate.dense), oracle.gemm_a_bf16_w_f32(bits, up.dense))
    for dtype in (torch.float32, torch.bfloat16):
        got = to_f32(rt.mlp_in(gate.w_tiled, up.w_tiled, a, out_dtype=dtype, workspace=ws))
        check_close(got, ref, bf16_out=dtype == torch.bfloat16, label=f"skinny pair {rows} {n} {k}")


@pytest.mark.parametrize("rows", [1, 2, 3, 9, 32])
def test_skinny_group(rt, rows):
    k, widths = 1088, (384, 128, 256)
    cases = [case(n, k, i) for i, n in enumerate(widths)]
    bits, a = activations(rows, k)
    ws = torch.zeros(max(1, rt.workspace_bytes(rows, sum(widths), k)), dtype=torch.uint8, device="cuda")
    for dtype in (torch.float32, torch.bfloat16):
        outs = rt.gemm_group([c.w_tiled for c in cases], a, out_dtype=dtype, workspace=ws)
        for c, out in zip(cases, outs):
            check_close(to_f32(out), oracle.gemm_a_bf16_w_f32(bits, c.dense), bf16_out=dtype == torch.bfloat16,
                        tight=True, absref=abs_gemm(bits, c.dense), label=f"skinny group {rows} {c.n}")
