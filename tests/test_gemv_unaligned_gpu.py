"""GEMV with operands that are only element-aligned: base pointers one element past a 16-byte
boundary, odd leading dimensions, tails shorter than a 16-byte vector, rows chunked unevenly."""
import numpy as np
import pytest

import oracle
from gpu_util import ctx, dev, empty, host, p

pytestmark = pytest.mark.gpu

FORMS = {np.float64: ("bzg_dgemv", "bzg_dgemv_t"), np.float32: ("bzg_sgemv", "bzg_sgemv_t"),
         np.int32: ("bzg_igemv", "bzg_igemv_t")}


@pytest.mark.parametrize("dtype", list(FORMS))
@pytest.mark.parametrize("m,n,lda,off", [(1, 1, 1, 1), (5, 3, 3, 1), (17, 7, 9, 1), (64, 129, 129, 0), (1000, 31, 33, 3),
                                         (333, 515, 517, 1), (3, 9001, 9001, 1), (4099, 1027, 1029, 1)])
def test_element_aligned_operands(dtype, m, n, lda, off):
    rng = np.random.default_rng(m * 1000 + n)
    if dtype is np.int32:
        A = rng.integers(-2 ** 31, 2 ** 31, (m, n)).astype(np.int32)
        xs = [rng.integers(-2 ** 31, 2 ** 31, s).astype(np.int32) for s in (n, m)]
    else:
        A = rng.uniform(-1, 1, (m, n)).astype(dtype)
        xs = [rng.uniform(-1, 1, s).astype(dtype) for s in (n, m)]
    buf = np.zeros(off + m * lda, dtype)
    np.lib.stride_tricks.as_strided(buf[off:], (m, n), (lda * buf.itemsize, buf.itemsize))[:] = A
    dA = dev(buf)
    for trans, x in ((0, xs[0]), (1, xs[1])):
        dx = dev(np.concatenate([np.zeros(off, dtype), x]))
        y = empty(n if trans else m, dtype)
        ctx().call(FORMS[dtype][trans], m, n, 1, p(dA[off:]), lda, p(dx[off:]), 0, p(y))
        got, op = host(y), A.T if trans else A
        if dtype is np.int32:
            assert np.array_equal(got, oracle.gemv(np.ascontiguousarray(op), x))
        else:
            # gamma_k bound of a k-term sum in any order
            u = np.finfo(dtype).eps / 2
            ref = op.astype(np.float64) @ x.astype(np.float64)
            assert np.all(np.abs(got - ref) <= (len(x) + 2) * u * (np.abs(op).astype(np.float64) @ np.abs(x)))
