"""Transposed GEMV where the number of row partitions changes its rule (8 rows per lane up to 256
partitions, then 16, then one full round of workgroups) and where a row's last vector overlaps its
neighbour's columns."""
import numpy as np
import pytest

import oracle
from gpu_util import ctx, dev, empty, host, p

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 7, 8, 9, 2047, 2048, 2049, 4095, 4096, 4097, 33000])
@pytest.mark.parametrize("n", [2, 3, 4, 5, 257, 1023])
def test_partitions(m, n):
    rng = np.random.default_rng(m * 2000 + n)
    A = rng.integers(-2 ** 31, 2 ** 31, (m, n)).astype(np.int32)
    x = rng.integers(-2 ** 31, 2 ** 31, m).astype(np.int32)
    dA, dx, guard = dev(A), dev(x), dev(np.full(n + 8, 7, np.int32))
    ctx().call("bzg_igemv_t", m, n, 1, p(dA), n, p(dx), 0, p(guard))
    out = host(guard)
    assert np.array_equal(out[:n], oracle.gemv(np.ascontiguousarray(A.T), x))
    assert np.all(out[n:] == 7)
    D, z = rng.uniform(-1, 1, (m, n)), rng.uniform(-1, 1, m)
    dD, dz, y = dev(D), dev(z), empty(n, np.float64)
    ctx().call("bzg_dgemv_t", m, n, 1.0, p(dD), n, p(dz), 0.0, p(y))
    # gamma_m bound of an m-term sum in any order
    assert np.all(np.abs(host(y) - z @ D) <= 2 * (m + 2) * 2.0 ** -53 * (np.abs(z) @ np.abs(D)))
