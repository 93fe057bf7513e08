"""The scratch a q4 call allocates by itself under AUTO: sized by splosh_q4_workspace_bytes, with only
its counters zeroed. Each call cuts its work as it does with a zeroed workspace of
splosh_workspace_bytes, so the results are the same bits, also where the allocator hands out a
block that holds other values."""
import numpy as np
import pytest
import torch

from qcheck import Q4Case, bf16_tensor
import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    from splosh_amd import runtime
    return runtime


@pytest.mark.parametrize("other_stream", [False, True])
@pytest.mark.parametrize("tiled", [True, False])
@pytest.mark.parametrize("rows", [1, 2, 3, 16, 17, 33, 65, 200])
def test_own_scratch_gives_the_same_bits(rt, rows, tiled, other_stream):
    n, k = 8448, 1088  # 264 blocks of 32 columns: a last round to split
    case = Q4Case(n, k, seed=rows)
    w = case.w_tiled if tiled else case.w_rm
    a = bf16_tensor(oracle.bf16_normal((rows, k), seed=rows + 1))
    full = torch.zeros(rt.workspace_bytes(rows, n, k), dtype=torch.uint8, device="cuda")
    want = rt.gemm(w, a, out_dtype=torch.float32, workspace=full)
    want_pair = rt.mlp_in(w, w, a, out_dtype=torch.float32, workspace=full)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream() if other_stream else None
    for _ in range(2):
        with torch.cuda.stream(stream) if stream else torch.cuda.stream(torch.cuda.current_stream()):
            dirt = torch.full((max(full.numel(), 1 << 20),), 0xA5, dtype=torch.uint8, device="cuda")
        del dirt
        got = rt.gemm(w, a, out_dtype=torch.float32, stream=stream)
        got_pair = rt.mlp_in(w, w, a, out_dtype=torch.float32, stream=stream)
        torch.cuda.synchronize()
        assert np.array_equal(got.cpu().numpy().view(np.uint32), want.cpu().numpy().view(np.uint32))
        assert np.array_equal(got_pair.cpu().numpy().view(np.uint32), want_pair.cpu().numpy().view(np.uint32))
