"""Infinite activations and scales, and activations whose products are finite though sums on raw codes
(128 + q) overflow, give what the dequantized weights give: infinities of the product's sign, not NaN."""
import numpy as np
import pytest
import torch

import oracle
from qcheck import Q4Case, bf16_tensor, to_f32

pytestmark = pytest.mark.gpu

INF = [("inf", 0), ("-inf", 0.5), ("inf", 1), ("huge", 0), ("huge", 1)]  # value, place along K


@pytest.fixture(scope="module")
def rt():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from splosh_amd import runtime
    return runtime


_CASES = {}


def case(n, k, seed=0):
    if (n, k, seed) not in _CASES:
        _CASES[n, k, seed] = Q4Case(n, k, seed=900 + seed + n + k)
    return _CASES[n, k, seed]


def activations(rows, k, value, place):
    """bf16 normals whose last row has `value` at one place."""
    bits = oracle.bf16_normal((rows, k), seed=rows + k)
    at = min(k - 1, int(place * (k - 1)))
    bits[rows - 1, at] = {"inf": 0x7F80, "-inf": 0xFF80, "huge": 0x7D70}[value]  # 2^123.9
    return bits


def reference(bits, dense):
    a = oracle.bf16_to_f32(bits).astype(np.float64)
    out = a[:-1] @ dense.T.astype(np.float64)
    with np.errstate(invalid="ignore"):
        return np.vstack([out, (a[-1] * dense.astype(np.float64)).sum(axis=1)])


def check(got, ref, label):
    got, finite = to_f32(got).astype(np.float64), np.isfinite(ref)
    assert np.array_equal(np.isnan(got), np.isnan(ref)), label
    assert np.array_equal(got[~finite], ref[~finite], equal_nan=True), label
    # Weights rounded to bf16 (2^-9 of each) in a row's sums, whose size is the row's largest output.
    size = np.where(finite, np.abs(ref), 0).max(axis=1, keepdims=True)
    bound = np.broadcast_to(2.0 ** -6 * size, ref.shape)
    assert np.all(np.abs(got[finite] - ref[finite]) <= bound[finite]), label


def workspaces(rt, rows, n, k):
    return (torch.zeros(max(4, rt.workspace_bytes(rows, n, k)), dtype=torch.uint8, device="cuda"),
            torch.empty(0, device="cuda"))


def infinite_scale(rt, c, tiled):
    """The weight with row 0's first group 2 inf + b; activations of that group have to be positive."""
    import dataclasses
    w = c.w_tiled if tiled else c.w_rm
    packed, scales = w.packed.clone(), w.scales.clone()
    packed.view(torch.int32).view(-1)[:8] = 0x22222222
    scales.view(torch.int16).view(-1)[0] = 0x7F80
    dense = c.dense.copy()
    dense[0, :64] = np.inf
    return dataclasses.replace(w, packed=packed, scales=scales), dense


def check_weight(rt, n, k, rows, tiled=True):
    c = case(n, k)
    for value, place in INF:
        bits = activations(rows, k, value, place)
        ref = reference(bits, c.dense)
        for ws in workspaces(rt, rows, n, k):
            check(rt.gemm(c.w_tiled if tiled else c.w_rm, bf16_tensor(bits), out_dtype=torch.float32, workspace=ws), ref,
                  f"{rows} {n} {k} {value} {place}")
    w, dense = infinite_scale(rt, c, tiled)
    bits = activations(rows, k, "inf", 1) & 0x7FFF
    bits[-1, -1] = 0x3F80
    got = to_f32(rt.gemm(w, bf16_tensor(bits), out_dtype=torch.float32, workspace=workspaces(rt, rows, n, k)[0]))
    assert np.all(got[:, 0] == np.inf), f"{rows} {n} {k} scale"
    check(torch.from_numpy(got[:, 1:].copy()), reference(bits, dense[1:]), f"{rows} {n} {k} scale")


# One block and wave quarter; K slices; a weight in its column halves (up to 16 rows).
@pytest.mark.parametrize("n,k,many", [(128, 64, True), (384, 2112, True), (1024, 4096, True), (8448, 192, False)])
@pytest.mark.parametrize("rows", [5, 8, 16, 17, 32])
def test_few_rows(rt, rows, n, k, many):
    if rows <= 16 or many:
        check_weight(rt, n, k, rows)


@pytest.mark.parametrize("rows", [1, 2, 9, 32])
def test_group(rt, rows):
    k, widths = 1088, (384, 128, 256)
    cases = [case(n, k, i) for i, n in enumerate(widths)]
    for value, place in INF:
        bits = activations(rows, k, value, place)
        for ws in workspaces(rt, rows, sum(widths), k):
            outs = rt.gemm_group([c.w_tiled for c in cases], bf16_tensor(bits), out_dtype=torch.float32, workspace=ws)
            for c, out in zip(cases, outs):
                check(out, reference(bits, c.dense), f"group {rows} {c.n} {value} {place}")


@pytest.mark.parametrize("rows,n,k", [(5, 640, 1088), (16, 640, 1088), (32, 128, 64)])
def test_pair(rt, rows, n, k):
    gate, up = case(n, k), case(n, k, 1)
    for value, place in INF[:3]:
        bits = activations(rows, k, value, place)
        got = rt.mlp_in(gate.w_tiled, up.w_tiled, bf16_tensor(bits), out_dtype=torch.float32,
                        workspace=workspaces(rt, rows, n, k)[0])
        with np.errstate(invalid="ignore", over="ignore"):
            g, u = reference(bits, gate.dense), reference(bits, up.dense)
            check(got, g * (1 / (1 + np.exp(-g))) * u, f"pair {rows} {n} {k} {value} {place}")


# Row-major weights: the dot kernel with 1 x 1, 1 x 2 and 2 x 4 outputs a workgroup, K over one round.
@pytest.mark.parametrize("rows,n,k", [(3, 48, 1088), (2, 1024, 5120), (33, 48, 192), (5, 481, 320), (64, 96, 8256)])
def test_row_major_few_outputs(rt, rows, n, k):
    check_weight(rt, n, k, rows, tiled=False)


# The MFMA kernel for more rows: fewer groups than its 16 waves, even and odd numbers of groups a wave.
@pytest.mark.parametrize("rows,n,k", [(70, 512, 192), (333, 96, 1024), (129, 129, 1088), (600, 48, 2112)])
def test_row_major_more_rows(rt, rows, n, k):
    check_weight(rt, n, k, rows, tiled=False)


# Prefill: whole tiles and cut ones whose jobs have odd numbers of groups, one and several weights.
@pytest.mark.parametrize("rows,n,k", [(129, 384, 2112), (200, 640, 192), (333, 1152, 1088), (700, 1152, 320)])
def test_prefill(rt, rows, n, k):
    c, d = case(n, k), case(128, k)
    for value, place in INF:
        bits = activations(rows, k, value, place)
        a, ref = bf16_tensor(bits), reference(bits, c.dense)
        for ws in workspaces(rt, rows, n + 128, k):
            check(rt.gemm(c.w_tiled, a, out_dtype=torch.float32, workspace=ws, kernel=rt.PREFILL), ref,
                  f"prefill {rows} {n} {k} {value} {place}")
            outs = rt.gemm_group([c.w_tiled, d.w_tiled], a, out_dtype=torch.float32, workspace=ws)
            check(outs[0], ref, f"grouped prefill {rows} {n} {k} {value} {place}")
            check(outs[1], reference(bits, d.dense), f"grouped prefill {rows} 128 {k} {value} {place}")


@pytest.mark.parametrize("rows,k", [(129, 1280), (333, 2304)])
def test_prefill_planes(rt, rows, k):
    n = 384
    native = oracle.q45k_random_native(n, k, seed=n)
    dense = oracle.q45k_decode(native).reshape(n, k)
    from qcheck import dev_u8
    w = rt.q5k_repack(dev_u8(native), n, k)
    for value, place in INF:
        bits = activations(rows, k, value, place)
        for ws in workspaces(rt, rows, n, k):
            check(rt.gemm(w, bf16_tensor(bits), out_dtype=torch.float32, workspace=ws, kernel=rt.PREFILL),
                  reference(bits, dense), f"prefill planes {rows} {k} {value} {place}")
