"""The f16-path GEMM of Q6_K weights (dequantized in registers) at the edges of its tiles and K
splits, against 64-bit products of the f16-rounded operands."""
import numpy as np
import pytest

import oracle
from tl_amd import GGML_Q6_K, QTensor
from tl_amd.quant import random_q6_k_blocks

pytestmark = pytest.mark.gpu


def test_q6_k_f16_two_to_the_30_weights(dev):
    """A weight whose f16 copy would pass 2 GiB: the GEMM makes none, and its own bytes fit."""
    m, n, k = 5, 131072, 8192
    rng = np.random.default_rng(0x715b0800)
    raw = np.tile(random_q6_k_blocks(rng, 1024, k).reshape(1024, -1), (n // 1024, 1))
    raw[-3:] = random_q6_k_blocks(rng, 3, k).reshape(3, -1)
    x = rng.standard_normal((m, k)).astype(np.float32)
    y = dev.tl_qtensor_matmul_f16(dev.tensor_new(x), QTensor(GGML_Q6_K, raw.reshape(-1), (n, k))).to_numpy()
    x16 = x.astype(np.float16).astype(np.float64)
    for a, b in ((0, 1024), (n - 1024, n)):
        w = oracle.dequantize(GGML_Q6_K, raw[a:b].reshape(-1), (b - a) * k).reshape(b - a, k)
        w = w.astype(np.float16).astype(np.float64)
        assert np.all(np.abs(y[:, a:b] - x16 @ w.T) <= (k / 8 + 20) * 2.0 ** -24 * (np.abs(x16) @ np.abs(w).T) + 1e-37)
    assert np.array_equal(y[:, :1024], y[:, 65536:66560])


@pytest.mark.parametrize("m,n,k", [(5, 3, 256), (16, 127, 5632), (17, 65, 512), (32, 1000, 2048), (33, 256, 2048),
                                   (64, 63, 11008), (65, 129, 768), (128, 2048, 1024), (129, 3001, 256),
                                   (301, 514, 5632), (512, 4096, 512), (200, 32000, 256)])
def test_q6_k_f16_edges(dev, m, n, k):
    rng = np.random.default_rng(0x715b0000 + m + n + k)
    raw = random_q6_k_blocks(rng, n, k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    y = dev.tl_qtensor_matmul_f16(dev.tensor_new(x), QTensor(GGML_Q6_K, raw, (n, k))).to_numpy()
    # both operands rounded once to f16 (subnormal halves included), then f32 sums: at most k / 8
    # roundings of at most the sum of magnitudes each
    w = oracle.dequantize(GGML_Q6_K, raw, n * k).reshape(n, k).astype(np.float16).astype(np.float64)
    x16 = x.astype(np.float16).astype(np.float64)
    assert np.all(np.abs(y - x16 @ w.T) <= (k / 8 + 20) * 2.0 ** -24 * (np.abs(x16) @ np.abs(w).T) + 1e-37)
