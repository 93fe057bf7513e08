"""An infinite block scale (fp16) reaches the output as the decoder gives it, in the native
formats' one-row, few-row, 64-row and prefill kernels: codes of one sign times a positive infinity are
infinities, not NaN."""
import numpy as np
import pytest
import torch

import oracle
from qcheck import dev_u8

pytestmark = pytest.mark.gpu
SCALE = {8: (34, 0), 14: (210, 208), 11: (110, 108), 20: (18, 0), 21: (110, 0), 23: (136, 0)}  # block bytes, offset of d


@pytest.fixture(scope="module")
def rt():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from splosh_amd import runtime
    return runtime


@pytest.mark.parametrize("rows", [1, 8, 24, 40, 64, 100, 130, 256])
@pytest.mark.parametrize("kind", [8, 14, 11, 20, 21, 23])
def test_infinite_scale(rt, kind, rows):
    n, k = 128, 512
    native = np.array(oracle.gguf_random_native(kind, n, k, seed=3)).view(np.uint8).reshape(-1).copy()
    size, at = SCALE[kind]
    blocks = native.reshape(-1, size)
    blocks[0] = 0 if kind in (11, 21) else 0x11  # row 0's first block: codes of one sign
    blocks[0, at:at + 2] = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)
    dense = oracle.gguf_decode(kind, native).reshape(n, k)
    first = dense[0][np.isinf(dense[0])]
    assert first.size and np.all(first == first[0]) and not np.any(np.isnan(dense[0]))
    a = torch.ones(rows, k, device="cuda").bfloat16()
    got = rt.gemm(rt.GgufWeight(dev_u8(native), kind, n, k), a, out_dtype=torch.float32).cpu().numpy()
    assert np.all(got[:, 0] == first[0])
    assert np.all(np.isfinite(got[:, 1:]))
