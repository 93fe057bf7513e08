"""The fused pair at 9 to 32 rows on the launch shapes of skinny.hip that depend on the rows: between one and two
blocks of 32 columns a CU (four waves a workgroup), K slices of few blocks with long K (one workgroup a CU from
17 rows, two below), and long K without slices; with scratch of exactly splosh_workspace_bytes and without."""
import pytest
import torch

import oracle
from qcheck import Q4Case, bf16_tensor, check_close, to_f32

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def weights():
    made = {}

    def get(n, k):
        if (n, k) not in made:
            made.clear()
            made[n, k] = Q4Case(n, k, seed=n), Q4Case(n, k, seed=n + 1)
        return made[n, k]
    return get


@pytest.mark.parametrize("n,k", [(8448, 192), (16256, 64), (512, 12352), (4224, 12288)])
@pytest.mark.parametrize("rows", [9, 16, 17, 32])
def test_pair(weights, rows, n, k):
    from splosh_amd import runtime as rt
    gate, up = weights(n, k)
    bits = oracle.bf16_normal((rows, k), seed=rows + k)
    bits[0] = 0
    ref = oracle.silu_mul(oracle.gemm_a_bf16_w_f32(bits, gate.dense), oracle.gemm_a_bf16_w_f32(bits, up.dense))
    ws = torch.zeros(max(1, rt.workspace_bytes(rows, n, k)), dtype=torch.uint8, device="cuda")
    for scratch in (ws, torch.empty(0, device="cuda")):
        got = rt.mlp_in(gate.w_tiled, up.w_tiled, bf16_tensor(bits), out_dtype=torch.float32, workspace=scratch)
        check_close(to_f32(got), ref, bf16_out=False, tight=True, label=f"pair {rows} {n} {k}")
    assert not ws[:16384].any()  # the counters are returned to zero
