"""GEMM where the last tile overlaps its neighbour: sizes just above one and several tiles, in all four
storage-order forms, with beta (an element stored twice would take it twice), short and long inner lengths;
NaN around the operands, guard values around the target.  Small integers: every sum is exact."""
import numpy as np
import pytest

from gpu_util import ctx, dev, host, p

pytestmark = pytest.mark.gpu

SIZES = [(31, 31), (33, 65), (63, 33), (65, 97), (127, 129), (321, 40), (40, 321),     # 32 x 32 tiles
         (897, 965), (1025, 833),                                                      # 64 x 64
         (3969, 4001)]                                                                 # 128 x 128, 128 x 256


@pytest.mark.parametrize("dtype,name", [(np.float64, "bzg_dgemm_ex"), (np.float32, "bzg_sgemm_ex")])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n", SIZES)
def test_last_tiles(dtype, name, ta, tb, m, n):
    rng = np.random.default_rng(m * 10000 + n)
    for k in (3, 16, 45, 150) if m < 3000 else (19,):
        def operand(X):
            ld = X.shape[1] + 1
            buf = np.full(1 + X.shape[0] * ld + 64, np.nan, dtype)
            np.lib.stride_tricks.as_strided(buf[1:], X.shape, (ld * buf.itemsize, buf.itemsize))[:] = X
            return dev(buf), ld

        A = rng.integers(-4, 5, (m, k)).astype(dtype)
        B = rng.integers(-4, 5, (k, n)).astype(dtype)
        C0 = rng.integers(-4, 5, (m + 2, n + 3)).astype(dtype)
        dA, lda = operand(A.T if ta else A)
        dB, ldb = operand(B.T if tb else B)
        d = dev(C0)
        ctx().call(name, ta, tb, m, n, k, 1.0, p(dA[1:]), lda, p(dB[1:]), ldb, 3.0, p(d), n + 3)
        want = C0.copy()
        want[:m, :n] = A @ B + 3 * C0[:m, :n]
        assert np.array_equal(host(d), want), k
