"""GGUF weights at a few activation rows (skinny_gguf.hip): every type, the file's order and ROWS32, at
the staged row counts' edges, one unit of K, ragged unit counts and columns, K slices with and
without a workspace, strided activations and outputs and a residual in place."""
import numpy as np
import pytest
import torch

import oracle
from qcheck import abs_gemm, bf16_tensor, check_close, dev_u8, to_f32

pytestmark = pytest.mark.gpu

NATIVE = [8, 11, 14, 20, 21, 23]


@pytest.fixture(scope="module")
def rt():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from splosh_amd import runtime
    return runtime


def weight(rt, kind, n, k, rows32):
    """(device weight, dense fp32): 12 / 13 are Q4_K / Q5_K planes."""
    if kind in (12, 13):
        native = oracle.q45k_random_native(n, k, seed=n + k, fifth_bit=kind == 13)
        w = (rt.q5k_repack if kind == 13 else rt.q4k_repack)(dev_u8(native), n, k)
        return w, oracle.q45k_decode(native, fifth_bit=kind == 13).reshape(n, k)
    native = oracle.gguf_random_native(kind, n, k, seed=n + k)
    w = rt.GgufWeight(dev_u8(native), kind, n, k)
    return (rt.gguf_repack_rows32(w) if rows32 else w), oracle.gguf_decode(kind, native).reshape(n, k)


def run(rt, w, dense, rows, n, k, label):
    bits = oracle.bf16_normal((rows, k), seed=rows + k)
    if rows > 1:
        bits[rows // 2] = 0
    a = torch.zeros(rows, k + 8, dtype=torch.bfloat16, device="cuda")
    a[:, :k] = bf16_tensor(bits)
    ref, scale = oracle.gemm_a_bf16_w_f32(bits, dense), abs_gemm(bits, dense)
    shift = np.float32(np.abs(ref).max())
    ws = torch.zeros(max(4, rt.workspace_bytes(rows, n, k)), dtype=torch.uint8, device="cuda")
    none = torch.empty(0, device="cuda")
    for dtype, scratch in ((torch.float32, ws), (torch.bfloat16, ws), (torch.float32, none)):
        out = torch.full((rows, n + 3), float(shift), dtype=dtype, device="cuda")
        rt.gemm(w, a, out=out, residual=out, workspace=scratch)
        got = to_f32(out)
        base = to_f32(torch.full((1,), float(shift), dtype=dtype))[0]
        assert np.all(got[:, n:] == base), label
        check_close(got[:, :n], ref + base, bf16_out=dtype == torch.bfloat16, tight=True, absref=scale, label=label)
    assert not ws[:16384].any(), label  # the counters are returned to zero


@pytest.mark.parametrize("rows32", [False, True])
@pytest.mark.parametrize("kind", NATIVE)
@pytest.mark.parametrize("n,k", [(72, 256), (161, 1280), (96, 16384)])
def test_native(rt, kind, rows32, n, k):
    w, dense = weight(rt, kind, n, k, rows32)
    for rows in (5, 8, 9, 16) + ((17, 31, 32) if kind in (11, 14, 21, 23) else ()):
        if kind == 11 and rows == 5 and not rows32:
            rows = 7
        run(rt, w, dense, rows, n, k, f"native {kind} rows32={rows32} {rows} {n} {k}")


@pytest.mark.parametrize("kind", [12, 13])
@pytest.mark.parametrize("n,k", [(128, 256), (256, 1280), (128, 16384)])
def test_planes(rt, kind, n, k):
    w, dense = weight(rt, kind, n, k, False)
    for rows in (5, 8, 9, 16):
        run(rt, w, dense, rows, n, k, f"planes {kind} {rows} {n} {k}")


@pytest.mark.parametrize("kind", [8, 11, 12, 13, 14, 20, 21, 23])
def test_two_to_four_rows(rt, kind):
    """From 2048 blocks x units (the one-row route of Q3_K among them)."""
    n, k = 8192, 2048
    w, dense = weight(rt, kind, n, k, False)
    for rows in (1, 2, 3, 4):
        run(rt, w, dense, rows, n, k, f"wide {kind} {rows}")
