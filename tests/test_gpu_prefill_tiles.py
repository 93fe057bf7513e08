"""The prefill kernel's tile heights (128, 192, 256 rows) and cuts of the remaining tiles (whole, S
slices a tile, even over the CUs, after whole rounds), at shapes plan_prefill gives each: one
weight with a residual and ragged rows, the emit, the fused pair, grouped weights whose columns
straddle the tiles, Q5_K planes and a native format; with and without a workspace."""
import numpy as np
import pytest
import torch

import oracle
from qcheck import Q4Case, abs_gemm, bf16_tensor, check_close, dev_u8, to_f32

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from splosh_amd import runtime
    return runtime


def scratch(rt, rows, n, k):
    return torch.zeros(max(1, rt.workspace_bytes(rows, n, k)), dtype=torch.uint8, device="cuda")


# 128-row tiles whole, in slices and over every CU; 192 in slices; 256 in slices, whole.
SHAPES = [(129, 128, 192), (129, 384, 2112), (129, 128, 8320), (200, 640, 2112), (150, 2304, 2112), (330, 1152, 2112),
          (700, 1152, 512), (1100, 2304, 192)]


@pytest.mark.parametrize("rows,n,k", SHAPES)
def test_single(rt, rows, n, k):
    c = Q4Case(n, k, seed=rows + n)
    bits = oracle.bf16_normal((rows, k), seed=rows)
    ref, scale = oracle.gemm_a_bf16_w_f32(bits, c.dense), abs_gemm(bits, c.dense)
    a, ws = bf16_tensor(bits), scratch(rt, rows, n, k)
    for dtype, s in ((torch.float32, ws), (torch.bfloat16, ws), (torch.float32, torch.empty(0, device="cuda"))):
        out = torch.full((rows, n + 4), 2.0, dtype=dtype, device="cuda")
        rt.gemm(c.w_tiled, a, out=out, residual=out, workspace=s, kernel=rt.PREFILL)
        got = to_f32(out)
        assert np.all(got[:, n:] == 2.0)
        check_close(got[:, :n], ref + 2.0, bf16_out=dtype == torch.bfloat16, tight=True, absref=scale,
                    label=f"prefill {rows} {n} {k}")
    wn = (1 + 0.1 * torch.randn(n, device="cuda")).to(torch.bfloat16)
    out, values, sums, squares = rt.gemm_emit(c.w_tiled, a, wn, workspace=ws, kernel=rt.PREFILL)
    want = rt.emit_operand(out, wn)
    assert torch.equal(values.view(torch.int16), want[0].view(torch.int16))
    assert torch.allclose(sums, want[1], rtol=1e-5, atol=1e-3) and torch.allclose(squares, want[2], rtol=1e-5)


@pytest.mark.parametrize("rows,n,k", [(129, 256, 2112), (200, 384, 192), (300, 640, 2112), (700, 1152, 320)])
def test_pair(rt, rows, n, k):
    gate, up = Q4Case(n, k, seed=rows), Q4Case(n, k, seed=rows + 1)
    bits = oracle.bf16_normal((rows, k), seed=rows)
    ref = oracle.silu_mul(oracle.gemm_a_bf16_w_f32(bits, gate.dense), oracle.gemm_a_bf16_w_f32(bits, up.dense))
    for dtype in (torch.float32, torch.bfloat16):
        got = to_f32(rt.mlp_in(gate.w_tiled, up.w_tiled, bf16_tensor(bits), out_dtype=dtype, kernel=rt.PREFILL,
                               workspace=scratch(rt, rows, n, k)))
        check_close(got, ref, bf16_out=dtype == torch.bfloat16, label=f"prefill pair {rows} {n} {k}")


@pytest.mark.parametrize("rows", [65, 100, 128, 129, 200, 330, 700])
@pytest.mark.parametrize("widths,k", [((384, 128, 640), 512), ((128, 256), 2112)])
def test_group(rt, rows, widths, k):
    cases = [Q4Case(n, k, seed=rows + i) for i, n in enumerate(widths)]
    bits = oracle.bf16_normal((rows, k), seed=rows)
    ws = scratch(rt, rows, sum(widths), k)
    for dtype in (torch.float32, torch.bfloat16):
        whole = torch.full((rows, sum(widths) + 8), 5.0, dtype=dtype, device="cuda")
        outs, at = [], 0
        for n in widths:
            outs.append(whole[:, at:at + n])
            at += n
        rt.gemm_group([c.w_tiled for c in cases], bf16_tensor(bits), outs=outs, workspace=ws)
        assert torch.all(whole[:, at:] == 5.0)
        for c, out in zip(cases, outs):
            check_close(to_f32(out), oracle.gemm_a_bf16_w_f32(bits, c.dense), bf16_out=dtype == torch.bfloat16,
                        tight=True, absref=abs_gemm(bits, c.dense), label=f"prefill group {rows} {c.n}")


@pytest.mark.parametrize("rows,n,k", [(200, 384, 2304), (300, 1152, 512)])
def test_gguf(rt, rows, n, k):
    bits = oracle.bf16_normal((rows, k), seed=rows)
    a, ws = bf16_tensor(bits), scratch(rt, rows, n, k)
    native = oracle.q45k_random_native(n, k, seed=n)
    dense = oracle.q45k_decode(native).reshape(n, k)
    got = to_f32(rt.gemm(rt.q5k_repack(dev_u8(native), n, k), a, out_dtype=torch.float32, workspace=ws))
    check_close(got, oracle.gemm_a_bf16_w_f32(bits, dense), bf16_out=False, tight=True, absref=abs_gemm(bits, dense),
                label=f"prefill q5k {rows} {n} {k}")
    for kind in (8, 14):
        native = oracle.gguf_random_native(kind, n, k, seed=n)
        dense = oracle.gguf_decode(kind, native).reshape(n, k)
        got = to_f32(rt.gemm(rt.GgufWeight(dev_u8(native), kind, n, k), a, out_dtype=torch.float32, workspace=ws))
        check_close(got, oracle.gemm_a_bf16_w_f32(bits, dense), bf16_out=False, tight=True,
                    absref=abs_gemm(bits, dense), label=f"prefill native {kind} {rows} {n} {k}")
