"""FP64 / FP32 GEMM at the edges of tiles and K slabs, in all four storage-order forms, with operands
that are only element-aligned and surrounded by NaN; sizes that reach every tile shape, each compared
with float64 and, bit for bit, with the small product of its last rows and columns."""
import numpy as np
import pytest

from gpu_util import ctx, dev, host, p

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (3, 5, 2), (31, 33, 15), (32, 32, 32), (33, 31, 65), (64, 64, 64), (65, 63, 127), (127, 129, 33),
          (70, 40, 130), (40, 70, 257), (1, 300, 64), (300, 1, 63), (128, 96, 192),  # 32 x 32 tiles
          (897, 901, 31), (960, 900, 97),       # 64 x 64
          (3970, 4091, 17), (4096, 3969, 48)]   # 128 x 128, FP32 128 x 256


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_edges(dtype, ta, tb, m, n, k):
    rng = np.random.default_rng(m * 10000 + n * 100 + k)
    name = "bzg_dgemm_ex" if dtype is np.float64 else "bzg_sgemm_ex"

    def operand(rows, cols, t):
        X = rng.uniform(-1, 1, (rows, cols)).astype(dtype)
        S = X.T if t else X
        ld = S.shape[1] + 1
        buf = np.full(1 + S.shape[0] * ld + 64, np.nan, dtype)
        np.lib.stride_tricks.as_strided(buf[1:], S.shape, (ld * buf.itemsize, buf.itemsize))[:] = S
        return X, dev(buf), ld

    A, dA, lda = operand(m, k, ta)
    B, dB, ldb = operand(k, n, tb)
    C0 = rng.uniform(-1, 1, (m, n)).astype(dtype)

    def run(r0, c0):
        """Rows r0.. and columns c0.. of 2 op(A) op(B) - C0, in a target with guard columns."""
        rows, cols = m - r0, n - c0
        out = np.full((rows, cols + 3), 9.5, dtype)
        out[:, :cols] = C0[r0:, c0:]
        d = dev(out)
        ctx().call(name, ta, tb, rows, cols, k, 2.0, p(dA[1 + (r0 if ta else r0 * lda):]), lda,
                   p(dB[1 + (c0 * ldb if tb else c0):]), ldb, -1.0, p(d), cols + 3)
        got = host(d)
        assert np.all(got[:, cols:] == 9.5)
        return got[:, :cols]

    got = run(0, 0)
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    bound = 2 * (k + 3) * (np.finfo(dtype).eps / 2) * (np.abs(A64) @ np.abs(B64) + np.abs(C0))
    assert np.all(np.abs(got - (2.0 * (A64 @ B64) - C0)) <= bound)
    r0, c0 = max(0, m - 37), max(0, n - 45)
    assert np.array_equal(run(r0, c0), got[r0:, c0:])
