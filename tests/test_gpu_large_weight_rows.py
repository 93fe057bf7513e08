"""80 to 128 rows of a large q4 weight under AUTO: one call of the prefill kernel where its scratch is
given, else the two calls of at most 64 rows; the fused pair likewise."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from splosh_amd import runtime
    return runtime


def random_weight(rt, n, k):
    return rt.Q4Weight(torch.randint(-2**31, 2**31 - 1, (n * k // 8,), dtype=torch.int32, device="cuda"),
                       (torch.rand(n * k // 64, device="cuda") * 0.01).bfloat16(),
                       (torch.rand(n * k // 64, device="cuda") * 0.01 - 0.07).bfloat16(), n, k)


@pytest.mark.parametrize("rows", [79, 80, 127, 128])
@pytest.mark.parametrize("n,k", [(16384, 5120), (5120, 16384 + 64)])  # 80 Mi elements, and a ragged K above it
def test_large(rt, rows, n, k):
    torch.manual_seed(rows)
    w, up = random_weight(rt, n, k), random_weight(rt, n, k)
    a = torch.randn(rows, k, device="cuda").bfloat16()
    ws = torch.zeros(rt.workspace_bytes(rows, n, k), dtype=torch.uint8, device="cuda")
    none = torch.empty(0, device="cuda")
    def both(kernel, s):
        return (rt.gemm(w, a, out_dtype=torch.float32, kernel=kernel, workspace=s),
                rt.mlp_in(w, up, a, out_dtype=torch.float32, kernel=kernel, workspace=s))
    auto, named, parts = both(rt.AUTO, ws), both(rt.PREFILL, ws), both(rt.AUTO, none)
    dense = rt.dequant(w)
    ref = (a.float().cpu() @ dense.cpu().T).cuda()
    scale = (a.float().abs().cpu() @ dense.abs().cpu().T).cuda()
    # The weights rounded to bf16 (2^-9 of each), and fp32 sums of k products.
    bound = (2.0 ** -9 + k * 2.0 ** -24) * scale
    for got in (auto[0], parts[0]):
        assert torch.all((got - ref).abs() <= bound)
    if rows >= 80:
        assert all(torch.equal(x, y) for x, y in zip(auto, named))
    # silu(g) u moves by at most 1.1 |u| dg + |silu(g)| du; |silu(g)| <= |g|.
    g, u = ref, (a.float().cpu() @ rt.dequant(up).cpu().T).cuda()
    du = bound.max()
    assert torch.all((auto[1] - parts[1]).abs() <= 2.2 * (u.abs() + du) * du + 2 * (g.abs() + du) * du)
