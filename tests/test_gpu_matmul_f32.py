"""The f32 batched matmul (tl_tensor_matmul) at the edges of its 64 x 64 x 32 tiles, with rows that
are whole float4s and rows that are not, batched and shared right operands, against 64-bit sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,m,n,k", [(1, 1, 1, 1), (3, 64, 64, 32), (2, 65, 63, 33), (5, 63, 68, 4), (1, 128, 130, 31),
                                         (4, 7, 129, 96), (2, 100, 4, 1000), (32, 128, 128, 64), (1, 17, 1025, 5)])
@pytest.mark.parametrize("shared", [False, True])
def test_matmul_f32_edges(dev, batch, m, n, k, shared):
    rng = np.random.default_rng(0x3A770000 + batch + m + n + k)
    a = rng.standard_normal((batch, m, k)).astype(np.float32)
    b = rng.standard_normal((k, n) if shared else (batch, k, n)).astype(np.float32)
    got = dev.tensor_matmul(dev.tensor_new(a), dev.tensor_new(b)).to_numpy()
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    # one f32 rounding per product and per addition, each at most 2^-24 of the running magnitude
    assert got.shape == (batch, m, n)
    assert np.all(np.abs(got - a64 @ b64) <= (k + 2) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64)))


def test_matmul_f32_specials(dev):
    """Infinities and NaN reach the outputs of their own row or column only, and subnormal
    operands count."""
    rng = np.random.default_rng(0x3A77F000)
    a = rng.standard_normal((70, 40)).astype(np.float32)
    b = rng.standard_normal((40, 66)).astype(np.float32)
    a[3, 7], a[65, 39], b[39, 65] = np.inf, np.nan, -np.inf
    a[10], b[:, 10] = 0, 1
    a[10, 5] = 1e-40
    got = dev.tensor_matmul(dev.tensor_new(a), dev.tensor_new(b)).to_numpy()
    want = a.astype(np.float64) @ b.astype(np.float64)
    fin = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    assert np.allclose(got[fin], want[fin], rtol=1e-4, atol=1e-4)
    assert got[10, 10] == np.float32(1e-40)
