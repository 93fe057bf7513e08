"""At three and four rows of tiled q4 the kernel AUTO takes is no further from 64 bits than the decode kernel
(STREAM by name), whose weights are exact and whose sums are fp32 too: weights centred on zero as a quantiser
leaves them, activations of both signs, and of one sign, where the code sums and the row sums of the group
identity cancel the most."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("one_sign", [False, True])
@pytest.mark.parametrize("n,k", [(1024, 64), (640, 1088), (2048, 5120)])
@pytest.mark.parametrize("rows", [3, 4])
def test_no_further_from_64_bits(rows, n, k, one_sign):
    from splosh_amd import runtime as rt
    gen = torch.Generator(device="cuda").manual_seed(rows + n + k)
    q = torch.randint(0, 16, (n, k), device="cuda", generator=gen)
    s = (0.004 * (0.75 + 0.5 * torch.rand(n, k // 64, device="cuda", generator=gen))).bfloat16()
    b = (-7.5 * s.float()).bfloat16()
    packed = (q.view(n, k // 8, 8) << (4 * torch.arange(8, device="cuda"))).sum(-1)
    packed = torch.where(packed >= 2 ** 31, packed - 2 ** 32, packed).to(torch.int32)
    w = rt.q4_to_tiled(rt.Q4Weight(packed, s.view(torch.int16), b.view(torch.int16), n, k, rt.ROW_MAJOR, k // 8))
    a = torch.randn(rows, k, device="cuda", generator=gen).bfloat16()
    a = a.abs() if one_sign else a
    ref = a.double() @ (q.double() * s.double().repeat_interleave(64, 1) + b.double().repeat_interleave(64, 1)).T
    off = [float((rt.gemm(w, a, out_dtype=torch.float32, kernel=kernel).double() - ref).norm() / ref.norm())
           for kernel in (rt.AUTO, rt.STREAM)]
    # (A tenth: the norm of 2000 or more roundings varies by a few percent.)
    assert off[0] <= 1.1 * off[1], off
