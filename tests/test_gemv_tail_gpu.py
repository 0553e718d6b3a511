"""GEMV with double rows of odd length, where the last column is read ahead of the vectors: every group width,
chunked rows, a last group with one row; NaN beside the matrix shows any column read too much."""
import numpy as np
import pytest

from gpu_util import ctx, dev, empty, host, p

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 7, 8, 9, 15, 63, 64, 65, 101, 255, 256, 257, 4095, 4097, 20001])
@pytest.mark.parametrize("m", [1, 2, 3, 131])
@pytest.mark.parametrize("pad", [0, 1])
def test_rows(n, m, pad):
    rng = np.random.default_rng(n * 1000 + m)
    A = rng.integers(-8, 9, (m, n)).astype(np.float64)
    x = rng.integers(-8, 9, n).astype(np.float64)
    z = rng.integers(-8, 9, m).astype(np.float64)
    lda = n + pad
    buf = np.full(m * lda + 8, np.nan)
    np.lib.stride_tricks.as_strided(buf, (m, n), (lda * 8, 8))[:] = A
    xg = np.full(n + 8, np.nan)
    xg[:n] = x
    dA, dx, dz, y, yt = dev(buf), dev(xg), dev(z), empty(m, np.float64), empty(n, np.float64)
    ctx().call("bzg_dgemv", m, n, 1.0, p(dA), lda, p(dx), 0.0, p(y))
    ctx().call("bzg_dgemv_t", m, n, 1.0, p(dA), lda, p(dz), 0.0, p(yt))
    assert np.array_equal(host(y), A @ x)  # sums of small integers: exact
    assert np.array_equal(host(yt), z @ A)
