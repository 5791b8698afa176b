"""Row softmax over lengths of every form: a wavefront per row, a workgroup per row, sums in index order."""
import numpy as np
import pytest

from tl_amd import HipDevice

pytestmark = pytest.mark.gpu

LENGTHS = [1, 4, 12, 15, 16, 17, 63, 64, 65, 128, 255, 256, 257, 301, 511, 512, 513, 1023, 1024, 1025, 2047,
           2049, 2050, 4097, 27586, 32767, 32768, 32769, 40000]


@pytest.mark.parametrize("n", LENGTHS)
def test_softmax_row_lengths(n):
    dev = HipDevice(0)
    rng = np.random.default_rng(n)
    x = (rng.standard_normal((7, n)) * 3).astype(np.float32)
    if n > 2:
        x[1, n // 2:] = -np.inf  # masked entries
        x[2] = -1e9
        x[3] = -np.inf
        x[4, n // 3] = np.nan
        x[5, n - 1] = np.inf
    got = dev.tensor_softmax(dev.tensor_new(x), -1).to_numpy()
    with np.errstate(invalid="ignore"):
        e = np.exp(x.astype(np.float64) - np.where(np.isnan(x), -np.inf, x).max(-1, keepdims=True))
        want = e / e.sum(-1, keepdims=True)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    # a sum of n f32 terms in index order: at most n roundings of 2^-24; the exponent of a difference
    # below 30 and its exp, the divide: below 1e-5
    np.testing.assert_allclose(got, want, rtol=1e-5 + n * 2.0**-24, atol=1e-37)
