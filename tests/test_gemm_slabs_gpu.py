"""GEMM at the inner lengths where the last slab is dropped to its first half (32 x 32 and 64 x 64
tiles, slabs of 16 to 64): small integers, so every sum is exact."""
import numpy as np
import pytest

from gpu_util import ctx, dev, host, p

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,name", [(np.float64, "bzg_dgemm_ex"), (np.float32, "bzg_sgemm_ex")])
@pytest.mark.parametrize("m,n", [(33, 47), (1000, 1100)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 1)])
def test_half_slabs(dtype, name, m, n, ta, tb):
    rng = np.random.default_rng(m + n)
    for k in (1, 7, 8, 9, 15, 16, 17, 24, 25, 31, 32, 33, 40, 48, 49, 63, 64, 65, 80, 96, 97, 127, 129, 160, 161, 225):
        A = rng.integers(-4, 5, (m, k)).astype(dtype)
        B = rng.integers(-4, 5, (k, n)).astype(dtype)
        a, b = np.ascontiguousarray(A.T if ta else A), np.ascontiguousarray(B.T if tb else B)
        dA, dB, dC = dev(a), dev(b), dev(np.full((m, n), np.nan, dtype))
        ctx().call(name, ta, tb, m, n, k, 1.0, p(dA), a.shape[1], p(dB), b.shape[1], 0.0, p(dC), n)
        assert np.array_equal(host(dC), A @ B), k
