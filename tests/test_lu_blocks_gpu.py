"""Batched FP64 LU at the edges of its blocks: orders around multiples of the panel (16) and of the block
(32), around the 64 rows that a register holds, and where the second instance (order > 256: panel 8, block
16) begins and ends.  The systems lie back to back, so a write outside one of them shows in another."""
import numpy as np
import pytest
import scipy.linalg as sl

from gpu_util import ctx
from blaze_amd import solve as bsolve

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 95, 96, 97, 127, 128, 129, 191, 193, 255, 256,
         257, 263, 264, 265, 271, 272, 273, 511, 512]


def check(A, LU, ip):
    n = len(A)
    _, pl = sl.lu_factor(A, check_finite=False)
    assert np.array_equal(ip - 1, pl)
    perm = np.arange(n)
    for i, q in enumerate(pl):
        perm[[i, q]] = perm[[q, i]]
    L, U = np.tril(LU, -1) + np.eye(n), np.triu(LU)
    # |P A - L U| <= gamma_n |L| |U| elementwise
    assert np.all(np.abs(A[perm] - L @ U) <= 2 * n * 2.0 ** -53 * (np.abs(L) @ np.abs(U)))


@pytest.mark.parametrize("lpt", [True, False])
def test_edges(lpt):
    rng = np.random.default_rng(41)
    As = [rng.uniform(-1, 1, (n, n)) for n in EDGES]
    LUs, ips, infos = bsolve.getrf_batched(ctx(), As, lpt=lpt)
    assert np.all(infos == 0)
    for A, LU, ip in zip(As, LUs, ips):
        check(A, LU, ip)


@pytest.mark.filterwarnings("ignore:Diagonal number")
@pytest.mark.filterwarnings("ignore::RuntimeWarning")
def test_zero_columns():
    """A column of zeros stays exactly zero through every update: info names the first one, its row is not
    interchanged and the columns after it are factored as ever."""
    rng = np.random.default_rng(42)
    As, want = [], []
    for n in (17, 33, 64, 100, 256, 257, 300):
        for z in sorted({0, 15, 16, 31, 32, n - 1}):
            if z < n:
                A = rng.uniform(-1, 1, (n, n))
                A[:, z] = 0.0
                As.append(A)
                want.append(z + 1)
    LUs, ips, infos = bsolve.getrf_batched(ctx(), As)
    assert np.array_equal(infos, want)
    for A, LU, ip, z in zip(As, LUs, ips, want):
        assert ip[z - 1] == z
        check(A, LU, ip)
