"""The prefill kernel over native GGUF blocks in whole units of 256 elements: every format, the file's
order and ROWS32, one unit of K and unit counts that no split divides, ragged rows around the tile
heights, few columns (cut over K) and many (whole tiles), strided activations and outputs with a
residual in place; with the call's scratch, with none and, head-ordered, with the least that the
call accepts."""
import numpy as np
import pytest
import torch

import oracle
from qcheck import abs_gemm, bf16_tensor, check_close, dev_u8, to_f32

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from splosh_amd import runtime
    return runtime


def weight(rt, kind, n, k, rows32):
    native = oracle.gguf_random_native(kind, n, k, seed=n + k)
    w = rt.GgufWeight(dev_u8(native), kind, n, k)
    return (rt.gguf_repack_rows32(w) if rows32 else w), oracle.gguf_decode(kind, native).reshape(n, k)


def scratch(rt, nbytes):
    return torch.zeros(max(4, nbytes), dtype=torch.uint8, device="cuda")


@pytest.mark.parametrize("rows32", [False, True])
@pytest.mark.parametrize("kind", [8, 11, 14, 20, 21, 23])
@pytest.mark.parametrize("n,k", [(128, 256), (384, 1792), (128, 8448)])
def test_units(rt, kind, rows32, n, k):
    w, dense = weight(rt, kind, n, k, rows32)
    for rows in (65, 129, 192, 257):
        bits = oracle.bf16_normal((rows, k), seed=rows + k)
        a = torch.zeros(rows, k + 8, dtype=torch.bfloat16, device="cuda")
        a[:, :k] = bf16_tensor(bits)
        ref, scale = oracle.gemm_a_bf16_w_f32(bits, dense), abs_gemm(bits, dense)
        shift = np.float32(np.abs(ref).max())
        ws, label = scratch(rt, rt.workspace_bytes(rows, n, k)), f"units {kind} {rows} {n} {k}"
        for dtype, s in ((torch.float32, ws), (torch.bfloat16, ws), (torch.float32, torch.empty(0, device="cuda"))):
            out = torch.full((rows, n + 4), float(shift), dtype=dtype, device="cuda")
            rt.gemm(w, a, out=out, residual=out, workspace=s)
            got = to_f32(out)
            base = to_f32(torch.full((1,), float(shift), dtype=dtype))[0]
            assert np.all(got[:, n:] == base), label
            check_close(got[:, :n], ref + base, bf16_out=dtype == torch.bfloat16, tight=True, absref=scale, label=label)
        assert not ws[:16384].any(), label  # other kernels' counters


@pytest.mark.parametrize("kind", [8, 14, 21])
def test_whole_tiles_after_rounds(rt, kind):
    """More tiles than CUs: whole rounds, then the rest (4096 outputs: 16 columns of tiles)."""
    rows, n, k = 2309, 4096, 512
    w, dense = weight(rt, kind, n, k, True)
    bits = oracle.bf16_normal((rows, k), seed=1)
    got = to_f32(rt.gemm(w, bf16_tensor(bits), out_dtype=torch.float32))
    check_close(got, oracle.gemm_a_bf16_w_f32(bits, dense), bf16_out=False, tight=True, absref=abs_gemm(bits, dense),
                label="rounds")


@pytest.mark.parametrize("kind", [8, 11, 14, 20, 21, 23])
@pytest.mark.parametrize("rows", [65, 128, 129, 255])
def test_heads_with_less_scratch(rt, kind, rows):
    """A head-ordered call gives the same result with its documented workspace (the prefill kernel) and
    with only room for the permuted activations (the kernels without scratch, 16 KiB of counters)."""
    n, k, key_heads = 128, 6144, 16
    w, dense = weight(rt, kind, n, k, True)
    bits = oracle.bf16_normal((rows, k), seed=rows)
    a = bf16_tensor(bits)
    full = rt.heads_workspace_bytes(rows, n, k)
    least = full - rt.workspace_bytes(rows, n, k) + 16384
    scale = abs_gemm(bits, dense)
    got = [to_f32(rt.gemm(w, a, out_dtype=torch.float32, workspace=scratch(rt, b), key_heads=key_heads))
           for b in (full, least)]
    # Each weight's bf16 rounding may fall to either side (a step is at most 2^-8 of it; scale is
    # sum |a||w| in the weight's own column order, so its largest element stands for all), and the two fp32 sums of 6144 products differ by less than 6144 roundings of 2^-24.
    assert np.all(np.abs(got[0] - got[1]) <= (2.0 ** -8 + 6144 * 2.0 ** -24) * scale.max())
